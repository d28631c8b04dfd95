// Batched adjoint Jacobians: many independent circuits, each from |0...0>
// with one observable, as register-tile programs.
//
// A circuit whose state is a few tiles runs whole in one workgroup
// (kernels_sweep.hip). The others run pass by pass, all together: launch k
// runs pass k of every circuit that has one, a wave per one or more tiles, then
// h = H phi with <phi|H|phi>, then the reverse passes likewise, with each pass's
// sums left per block. One workgroup per circuit left the chip waiting for the
// widest one (1024 circuits of 6-16 qubits complex64: 32 ms, the time of one
// 16-qubit, 8-layer circuit); now 2.5 ms: 0.8 for the whole circuits, 0.6, 0.1
// and 1.2 for the staged ones' forward passes, observables and reverse passes,
// each launch bound by the vector issue and latency of two waves of tiles per
// SIMD (states stay in the 256 MB last-level cache).
//
// Jacobian sums are FP64 and in a fixed order: row halves by DPP, LDS per half, the
// blocks of a pass in order.
#include "rtile_device.hpp"

namespace plk {

namespace {

template <typename T, int NS, int R>
__global__ void __launch_bounds__(64, 4) stage_kernel(BatchArgs A, const BatchBlock *__restrict__ blocks) {
    constexpr int NA = 1 << R;
    constexpr int TB = R + RT_LANE_BITS;
    __shared__ double lacc[NS > 1 ? RT_SLOTS_MAX * RT_CELLS + 64 : 1];
    const BatchBlock b = load_uniform(blocks + blockIdx.x);
    const BatchCircuit c = load_uniform(A.circuits + b.circuit);
    const SweepPass P = load_uniform(A.passes + b.pass);
    const int lane = static_cast<int>(__lane_id());
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
    Cx<T> *const scratch = static_cast<Cx<T> *>(A.scratch);
    Cx<T> *const sp[2] = {scratch + c.phi, scratch + c.h};
    const bool init = b.first != 0;
    const Ins<T> first = fetch<T>(prog, 0);
    for (int t = b.block; t < 1 << (c.n - TB); t += c.blocks) {
        uint64_t base = static_cast<uint64_t>(t);
#pragma unroll
        for (int q = 0; q < TB; q++) {
            base = insert_zero(base, P.tb[q]);
        }
        Cx<T> v[NS][NA];
#pragma unroll
        for (int s = 0; s < NS; s++) {
#pragma unroll
            for (int k = 0; k < NA; k++) {
                const uint32_t i = static_cast<uint32_t>(base) + vin +
                                   static_cast<uint32_t>(slot_off<T, R>(P.reg_in, k) / sizeof(Cx<T>));
                v[s][k] = NS == 1 && init ? Cx<T>{static_cast<T>(i == 0 ? 1 : 0), T(0)} : ldg(sp[s], i);
            }
        }
        run_program<T, NS, R>(v, first, prog, P.ninstr, lacc, dummy, lane, base);
#pragma unroll
        for (int s = 0; s < NS; s++) {
#pragma unroll
            for (int k = 0; k < NA; k++) {
                const uint32_t i = static_cast<uint32_t>(base) + vout +
                                   static_cast<uint32_t>(slot_off<T, R>(P.reg_out, k) / sizeof(Cx<T>));
                stg(sp[s], i, v[s][k]);
            }
        }
    }
    if constexpr (NS > 1) {
        __syncthreads();
        for (int i = lane; i < P.nslots; i += 64) {
            double s = 0.0;
#pragma unroll
            for (int q = 0; q < RT_CELLS; q++) {
                s += lacc[i * RT_CELLS + q];
            }
            A.parts[P.parts + static_cast<int64_t>(i) * c.blocks + b.block] = s;
        }
    }
}

// h = H phi over a block's share of the state, and its part of <phi|H|phi>.
template <typename T>
__global__ void __launch_bounds__(256) stage_observable_kernel(BatchArgs A, const BatchBlock *__restrict__ blocks) {
    __shared__ double red[4];
    const BatchBlock b = load_uniform(blocks + blockIdx.x);
    const BatchCircuit c = load_uniform(A.circuits + b.circuit);
    const Cx<T> *phi = static_cast<const Cx<T> *>(A.scratch) + c.phi;
    Cx<T> *h = static_cast<Cx<T> *>(A.scratch) + c.h;
    const uint32_t len = uint32_t{1} << c.n;
    double e = pauli_share<T>(A.terms + c.term_first, c.term_count, phi, h,
                              static_cast<uint32_t>(b.block) * 256 + threadIdx.x,
                              static_cast<uint32_t>(c.blocks) * 256, len);
    e = wave_sum(e);
    if ((threadIdx.x & 63) == 0) {
        red[threadIdx.x >> 6] = e;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        A.parts[c.eparts + b.block] = red[0] + red[1] + red[2] + red[3];
    }
}

// One thread per Jacobian entry or expectation value (entry < 0) of the
// staged circuits.
__global__ void __launch_bounds__(256)
    tail_kernel(BatchArgs A, const BatchTail *__restrict__ tails, int count) {
    const int t = static_cast<int>(blockIdx.x * 256 + threadIdx.x);
    if (t >= count) {
        return;
    }
    const BatchTail b = tails[t];
    double x = 0.0;
    if (b.entry < 0) {
        for (int k = 0; k < b.blocks; k++) {
            x += A.parts[b.parts + k];
        }
        A.expvals[b.out] = x;
        return;
    }
    const SweepEntry e = A.entries[b.entry];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        if (e.slot[k] >= 0) {
            const double *row = A.parts + b.parts + static_cast<int64_t>(e.slot[k]) * b.blocks;
            double s = 0.0;
            for (int q = 0; q < b.blocks; q++) {
                s += row[q];
            }
            x = fma(e.m[k], s, x);
        }
    }
    A.jac[b.out + e.col] = x;
}

// 2x2 complex FP64 matrices, row-major.
struct M2 {
    double r[4], i[4];
};
__device__ __forceinline__ M2 mul(const M2 &a, const M2 &b) {
    M2 c;
#pragma unroll
    for (int p = 0; p < 2; p++) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
            c.r[2 * p + q] = a.r[2 * p] * b.r[q] - a.i[2 * p] * b.i[q] + a.r[2 * p + 1] * b.r[2 + q] -
                             a.i[2 * p + 1] * b.i[2 + q];
            c.i[2 * p + q] = a.r[2 * p] * b.i[q] + a.i[2 * p] * b.r[q] + a.r[2 * p + 1] * b.i[2 + q] +
                             a.i[2 * p + 1] * b.r[2 + q];
        }
    }
    return c;
}

__device__ __forceinline__ M2 gate_matrix(const BatchGate &g, const double *params, const double *consts) {
    if (g.gate == BPG_CONST) {
        const double *m = consts + 8 * static_cast<int64_t>(g.param);
        return {{m[0], m[2], m[4], m[6]}, {m[1], m[3], m[5], m[7]}};
    }
    const double t = g.adj ? -params[g.param] : params[g.param];
    double s, c;
    if (g.gate == BPG_PHASE) {
        sincos(t, &s, &c);
        return {{1, 0, 0, c}, {0, 0, 0, s}};
    }
    sincos(0.5 * t, &s, &c);
    if (g.gate == BPG_RX) {
        return {{c, 0, 0, c}, {0, -s, -s, 0}};
    }
    if (g.gate == BPG_RY) {
        return {{c, -s, s, c}, {0, 0, 0, 0}};
    }
    return {{c, 0, 0, c}, {-s, 0, 0, s}}; // RZ
}

// One thread per run: its matrix from this call's angles, and the Pauli
// parts V^dag G V of its trainable gates (V the gates before one).
template <typename T>
__global__ void __launch_bounds__(256)
    batch_patch_kernel(unsigned char *__restrict__ blob, SweepEntry *__restrict__ entries,
                       const BatchRun *__restrict__ runs, int64_t count, const BatchGate *__restrict__ gates,
                       const double *__restrict__ params, const double *__restrict__ consts) {
    const int64_t i = int64_t{blockIdx.x} * blockDim.x + threadIdx.x;
    if (i >= count) {
        return;
    }
    const BatchRun run = runs[i];
    M2 V{{1, 0, 0, 1}, {0, 0, 0, 0}};
    int e = run.entry;
    for (int k = 0; k < run.count; k++) {
        const BatchGate g = gates[run.first + k];
        if (g.coef != 0.0 && run.entry >= 0) {
            M2 G{{0, 0, 0, 0}, {0, 0, 0, 0}};
            if (g.gate == BPG_RX) {
                G.r[1] = G.r[2] = 1.0;
            } else if (g.gate == BPG_RY) {
                G.i[1] = -1.0;
                G.i[2] = 1.0;
            } else {
                G.r[0] = 1.0;
                G.r[3] = -1.0;
            }
            const M2 Vd{{V.r[0], V.r[2], V.r[1], V.r[3]}, {-V.i[0], -V.i[2], -V.i[1], -V.i[3]}};
            const M2 W = mul(Vd, mul(G, V));
            const double m[3] = {g.coef * 0.5 * (W.r[1] + W.r[2]), g.coef * 0.5 * (W.i[2] - W.i[1]),
                                 g.coef * 0.5 * (W.r[0] - W.r[3])};
            if (run.parts == 7) {
                entries[e].m[0] = m[0];
                entries[e].m[1] = m[1];
                entries[e].m[2] = m[2];
            } else {
                entries[e].m[0] = run.parts == 1 ? m[0] : run.parts == 2 ? m[1] : m[2];
            }
            e++;
        }
        V = mul(gate_matrix(g, params, consts), V);
    }
    T *u = reinterpret_cast<T *>(blob + run.ins);
    if (run.ukind == U_DIAG) {
        u[0] = static_cast<T>(V.r[0]);
        u[1] = static_cast<T>(V.i[0]);
        u[2] = static_cast<T>(V.r[3]);
        u[3] = static_cast<T>(V.i[3]);
    } else if (run.ukind == U_REAL) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            u[k] = static_cast<T>(V.r[k]);
        }
    } else {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            u[2 * k] = static_cast<T>(V.r[k]);
            u[2 * k + 1] = static_cast<T>(V.i[k]);
        }
    }
}

} // namespace

void launch_batch_patch(Device &dev, int dtype, unsigned char *blob, SweepEntry *entries, const BatchRun *runs,
                        int64_t count, const BatchGate *gates, const double *params, const double *consts) {
    if (count <= 0) {
        return;
    }
    const unsigned grid = static_cast<unsigned>((count + 255) / 256);
    ProfScope prof("batch_patch", 0.0, dev.stream);
    if (dtype == PLK_C64) {
        hipLaunchKernelGGL(batch_patch_kernel<float>, dim3(grid), dim3(256), 0, dev.stream, blob, entries, runs,
                           count, gates, params, consts);
    } else {
        hipLaunchKernelGGL(batch_patch_kernel<double>, dim3(grid), dim3(256), 0, dev.stream, blob, entries, runs,
                           count, gates, params, consts);
    }
    PLK_HIP(hipGetLastError());
}

void launch_batch_stage(Device &dev, int dtype, const BatchArgs &A, const BatchBlock *blocks, int count,
                        BatchStage stage) {
    if (count <= 0) {
        return;
    }
    constexpr int RF = sweep_reg_bits<float>(), RD = sweep_reg_bits<double>();
    const dim3 grid(static_cast<unsigned>(count));
    if (stage == BATCH_OBSERVABLE) {
        if (dtype == PLK_C64) {
            hipLaunchKernelGGL(stage_observable_kernel<float>, grid, dim3(256), 0, dev.stream, A, blocks);
        } else {
            hipLaunchKernelGGL(stage_observable_kernel<double>, grid, dim3(256), 0, dev.stream, A, blocks);
        }
    } else if (stage == BATCH_FORWARD) {
        if (dtype == PLK_C64) {
            hipLaunchKernelGGL((stage_kernel<float, 1, RF>), grid, dim3(64), 0, dev.stream, A, blocks);
        } else {
            hipLaunchKernelGGL((stage_kernel<double, 1, RD>), grid, dim3(64), 0, dev.stream, A, blocks);
        }
    } else {
        if (dtype == PLK_C64) {
            hipLaunchKernelGGL((stage_kernel<float, 2, RF>), grid, dim3(64), 0, dev.stream, A, blocks);
        } else {
            hipLaunchKernelGGL((stage_kernel<double, 2, RD>), grid, dim3(64), 0, dev.stream, A, blocks);
        }
    }
    PLK_HIP(hipGetLastError());
}

void launch_batch_tails(Device &dev, const BatchArgs &A, const BatchTail *tails, int count) {
    if (count <= 0) {
        return;
    }
    hipLaunchKernelGGL(tail_kernel, dim3(static_cast<unsigned>((count + 255) / 256)), dim3(256), 0, dev.stream, A,
                       tails, count);
    PLK_HIP(hipGetLastError());
}

} // namespace plk
