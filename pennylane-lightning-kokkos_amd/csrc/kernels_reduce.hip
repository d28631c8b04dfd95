// The Jacobian entries of a sweep from the partial sums its launches left:
// one wave per (entry, observable) adds the blocks of up to three rows in a
// fixed order and combines them.
#include "device_common.hpp"

namespace plk {

namespace {

__global__ void __launch_bounds__(64)
    entries_kernel(const double *__restrict__ partials, const RtEntry *__restrict__ entries, int width,
                   double *__restrict__ jac, int ld) {
    const RtEntry e = entries[blockIdx.x / static_cast<unsigned>(width)];
    const int j = static_cast<int>(blockIdx.x % static_cast<unsigned>(width)) - e.j0;
    if (j < 0 || j >= e.width) {
        return;
    }
    const double *p = partials + e.base;
    double v = 0.0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        if (e.row[k] < 0) {
            continue;
        }
        const double *row = p + static_cast<uint64_t>(e.row[k] + j) * static_cast<uint64_t>(e.blocks);
        double s = 0.0;
        for (int b = static_cast<int>(threadIdx.x); b < e.blocks; b += 64) {
            s += row[b];
        }
        v = fma(e.m[k], s, v);
    }
    v = wave_sum(v);
    if (threadIdx.x == 0) {
        jac[static_cast<uint64_t>(e.j0 + j) * ld + e.col] = v;
    }
}

} // namespace

void launch_rtile_entries(Device &dev, const double *partials, const RtEntry *entries, int count, int width,
                          double *d_jac, int ld) {
    if (count <= 0 || width <= 0) {
        return;
    }
    hipLaunchKernelGGL(entries_kernel, dim3(static_cast<unsigned>(count) * static_cast<unsigned>(width)), dim3(64),
                       0, dev.stream, partials, entries, width, d_jac, ld);
    PLK_HIP(hipGetLastError());
}

} // namespace plk
