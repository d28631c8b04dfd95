// Whole circuits in one launch: a workgroup runs every register-tile pass of
// a circuit, forward and backward, with a barrier between passes.
//
// A small state has so few tiles that a launch per pass is all latency (12
// qubits: 8 tiles; a pass and its launch gap cost more than its arithmetic).
// Here one workgroup owns the state: it copies the input state (or |0...0>)
// to its scratch, runs the forward passes, forms h = H phi and <phi|H|phi>
// for its observable, and runs the reverse passes over phi and h, writing the
// Jacobian entries of each pass as it ends. Every observable of a circuit is a
// workgroup of its own with its own phi: repeating the forward passes on
// another CU costs no time, and nothing is shared between workgroups. The
// states (a few thousand amplitudes each) stay in the CU's L1 and the
// XCD's L2; waves of a workgroup exchange tiles through them, ordered by the
// barrier. States smaller than a tile fill part of it (the bits above the
// state's are idle, their amplitudes zero and never stored).
//
// Bound: the serial chain of one wave per tile (instruction decode, branches and
// FP64 latency, about 0.6 us an operation; two waves per SIMD at 12 qubits).
// 12 qubits complex128, 12 observables, 96 one-wire runs and CNOTs each way: 0.20
// ms in the kernel and 0.36 ms a call, against 0.53 ms a call with one launch per
// pass replayed from a HIP graph. Observables of many words take the general path
// (the observable step has one workgroup here).
//
// Jacobian sums are FP64 and in a fixed order: row halves by DPP, LDS per half and
// wave, then halves and waves in order.
#include "rtile_device.hpp"

namespace plk {

namespace {

// Per-wave LDS: the pass's sums and a dummy slot per lane.
constexpr int kWaveSums = RT_SLOTS_MAX * RT_CELLS + 64;

template <typename T, int NS, int R>
__device__ __forceinline__ void run_pass(const SweepArgs &A, const SweepPass &P, int n, Cx<T> *phi, Cx<T> *h,
                                         double *jac, double *sums, double *totals) {
    constexpr int NA = 1 << R;
    const int lane = static_cast<int>(__lane_id());
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int nwaves = static_cast<int>(blockDim.x) >> 6;
    double *lacc = sums + wave * kWaveSums;
    const int dummy = P.nslots * RT_CELLS;
    if constexpr (NS > 1) {
        for (int i = lane; i < dummy; i += 64) {
            lacc[i] = 0.0;
        }
    }
    CT<unsigned char> *prog = (CT<unsigned char> *)(A.blob + P.prog);
    uint32_t vin = 0, vout = 0;
#pragma unroll
    for (int p = 0; p < RT_LANE_BITS; p++) {
        vin |= static_cast<uint32_t>(lbit(lane, p)) << P.lane_in[p];
        vout |= static_cast<uint32_t>(lbit(lane, p)) << P.lane_out[p];
    }
    const Ins<T> first = fetch<T>(prog, 0);
    const uint32_t len = uint32_t{1} << n;
    const int ntiles = n > R + RT_LANE_BITS ? 1 << (n - R - RT_LANE_BITS) : 1;
    Cx<T> *const sp[2] = {phi, h};
    for (int t = wave; t < ntiles; t += nwaves) {
        uint64_t base = static_cast<uint64_t>(t);
#pragma unroll
        for (int q = 0; q < R + RT_LANE_BITS; q++) {
            base = insert_zero(base, P.tb[q]);
        }
        Cx<T> v[NS][NA];
#pragma unroll
        for (int s = 0; s < NS; s++) {
#pragma unroll
            for (int k = 0; k < NA; k++) {
                const uint32_t i = static_cast<uint32_t>(base) + vin +
                                   static_cast<uint32_t>(slot_off<T, R>(P.reg_in, k) / sizeof(Cx<T>));
                v[s][k] = i < len ? ldg(sp[s], i) : Cx<T>{T(0), T(0)};
            }
        }
        run_program<T, NS, R>(v, first, prog, P.ninstr, lacc, dummy, lane, base);
#pragma unroll
        for (int s = 0; s < NS; s++) {
#pragma unroll
            for (int k = 0; k < NA; k++) {
                const uint32_t i = static_cast<uint32_t>(base) + vout +
                                   static_cast<uint32_t>(slot_off<T, R>(P.reg_out, k) / sizeof(Cx<T>));
                if (i < len) {
                    stg(sp[s], i, v[s][k]);
                }
            }
        }
    }
    __syncthreads();
    if constexpr (NS > 1) {
        if (P.nslots > 0) {
            for (int i = static_cast<int>(threadIdx.x); i < P.nslots; i += static_cast<int>(blockDim.x)) {
                double s = 0.0;
                for (int w = 0; w < nwaves; w++) {
                    for (int q = 0; q < RT_CELLS; q++) {
                        s += sums[w * kWaveSums + i * RT_CELLS + q];
                    }
                }
                totals[i] = s;
            }
            __syncthreads();
            for (int e = static_cast<int>(threadIdx.x); e < P.entry_count; e += static_cast<int>(blockDim.x)) {
                const SweepEntry t = A.entries[P.entry_first + e];
                double x = 0.0;
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    if (t.slot[k] >= 0) {
                        x = fma(t.m[k], totals[t.slot[k]], x);
                    }
                }
                jac[t.col] = x;
            }
        }
    }
}

// h = H phi (a sum of Pauli words) and, into *out, <phi|H|phi>.
template <typename T>
__device__ __forceinline__ void observable(const SweepArgs &A, const SweepJob &J, const Cx<T> *phi, Cx<T> *h,
                                           double *red) {
    const uint32_t len = uint32_t{1} << J.n;
    double e = pauli_share<T>(A.terms + J.term_first, J.term_count, phi, h, threadIdx.x, blockDim.x, len);
    e = wave_sum(e);
    if ((threadIdx.x & 63) == 0) {
        red[threadIdx.x >> 6] = e;
    }
    __syncthreads();
    if (threadIdx.x == 0 && J.expval != nullptr) {
        double tot = 0.0;
        for (int w = 0; w < static_cast<int>(blockDim.x) >> 6; w++) {
            tot += red[w];
        }
        *J.expval = tot;
    }
    __syncthreads();
}

template <typename T, int R>
__global__ void __launch_bounds__(64 * kSweepWaves, 4) sweep_kernel(SweepArgs A) {
    extern __shared__ double sums[]; // kWaveSums per wave
    __shared__ double totals[RT_SLOTS_MAX];
    __shared__ double red[kSweepWaves];
    const SweepJob J = load_uniform(A.jobs + blockIdx.x);
    Cx<T> *phi = static_cast<Cx<T> *>(J.phi);
    Cx<T> *h = static_cast<Cx<T> *>(J.h);
    const uint32_t len = uint32_t{1} << J.n;
    for (int i = static_cast<int>(threadIdx.x); i < J.jac_len; i += static_cast<int>(blockDim.x)) {
        J.jac[i] = 0.0;
    }
    if (J.ref != J.phi) {
        const Cx<T> *ref = static_cast<const Cx<T> *>(J.ref);
        for (uint32_t i = threadIdx.x; i < len; i += blockDim.x) {
            stg(phi, i, ref != nullptr ? ldg(ref, i) : Cx<T>{static_cast<T>(i == 0 ? 1 : 0), T(0)});
        }
        __syncthreads();
    }
    for (int p = 0; p < J.fwd_count; p++) {
        run_pass<T, 1, R>(A, load_uniform(A.passes + J.fwd_first + p), J.n, phi, h, J.jac, sums, totals);
    }
    if (h == nullptr) {
        return;
    }
    observable<T>(A, J, phi, h, red);
    for (int p = 0; p < J.rev_count; p++) {
        run_pass<T, 2, R>(A, load_uniform(A.passes + J.rev_first + p), J.n, phi, h, J.jac, sums, totals);
    }
}

} // namespace

void launch_sweep(Device &dev, int dtype, const SweepArgs &A, int jobs, int waves) {
    if (jobs <= 0) {
        return;
    }
    if (waves < 1 || waves > kSweepWaves) {
        raise(PLK_ERR_INVALID, "whole-circuit launch: 1 to 8 waves a workgroup");
    }
    const size_t lds = static_cast<size_t>(waves) * kWaveSums * sizeof(double);
    ProfScope prof("circuit_sweep", 0.0, dev.stream);
    if (dtype == PLK_C64) {
        hipLaunchKernelGGL((sweep_kernel<float, sweep_reg_bits<float>()>), dim3(static_cast<unsigned>(jobs)),
                           dim3(64 * static_cast<unsigned>(waves)), lds, dev.stream, A);
    } else {
        hipLaunchKernelGGL((sweep_kernel<double, sweep_reg_bits<double>()>), dim3(static_cast<unsigned>(jobs)),
                           dim3(64 * static_cast<unsigned>(waves)), lds, dev.stream, A);
    }
    PLK_HIP(hipGetLastError());
}

} // namespace plk
