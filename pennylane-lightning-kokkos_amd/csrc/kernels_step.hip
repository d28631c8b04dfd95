// Single-operation adjoint steps for the operations the fused passes do not
// hold: dense matrices on 3 or 4 wires (Toffoli, CSWAP, DoubleExcitation±,
// 3-4-wire matrices, MultiRZ on 3-4 wires) and parity phases on any number of
// wires (MultiRZ).
//
// The reference takes one such step as a copy mu = lambda, U^dagger on
// lambda, G on mu, one blocking inner product per observable and U^dagger on
// every H_j lambda (AdjointDiffKokkos.hpp:454-476): 3 + 2 n_obs launches.
// Here one launch per chunk of observable states does the whole step. An op
// on m wires acts on groups of 2^m amplitudes (the op's wires, all other
// bits fixed), but most such ops move only a few of a group's states
// (DoubleExcitation: 2 of 16, Toffoli and CSWAP: 2 of 8). The host passes
// the D-state subspace outside which U is the identity and G is zero
// (D = 2, 4, 8 or 16) with U and G restricted to it. Each thread owns one
// group: it loads phi's D amplitudes, forms G phi in registers (phi before
// U, as the reference's mu), stores U phi (with the last chunk), and for each
// observable state h_j loads the group's D amplitudes, adds Im<h_j|G phi> in
// FP64 and writes U h_j back: (1 + w + 2 nj) (D / 2^m) S per launch, in
// whole cache lines when the op's wires include the lowest index bits. U and
// G are FP64 matrices read through the scalar cache; amplitudes of complex64
// states are widened to FP64 for the products and rounded once on the
// store.
//
// Jacobian sums: per thread in LDS (one slot per observable state), then a
// fixed-order block sum into the partials as [j][block], which the sweep's
// reduction adds in order.
#include "device_common.hpp"

namespace plk {

namespace {

constexpr int kStepBlock = 256;
constexpr int kSlabThreads = 512;

__device__ __forceinline__ double block_total(double v, double *red) {
    v = wave_sum(v);
    __syncthreads(); // red is reused across calls
    if ((threadIdx.x & 63) == 0) {
        red[threadIdx.x >> 6] = v;
    }
    __syncthreads();
    return red[0] + red[1] + red[2] + red[3];
}

// Writes the block's FP64 totals of the nj per-thread slots.
__device__ __forceinline__ void step_partials(const double *sacc, int nj, double *partials) {
    __shared__ double red[kStepBlock / 64];
    for (int j = 0; j < nj; j++) {
        const double t = block_total(sacc[j * kStepBlock + threadIdx.x], red);
        if (threadIdx.x == 0) {
            partials[static_cast<uint64_t>(j) * gridDim.x + blockIdx.x] = t;
        }
    }
}

// w = M x for a D x D FP64 matrix (row-major, double2 entries); stored
// through the group's offsets.
template <typename T, int D>
__device__ __forceinline__ void mat_store(Cx<T> *p, uint64_t base, const uint64_t *off,
                                          const double2 *__restrict__ M, const double *xr,
                                          const double *xi) {
#pragma unroll
    for (int r = 0; r < D; r++) {
        // One row of matrix loads at a time (scalar registers hold a row).
        __asm__ volatile("" ::: "memory");
        double wr = 0.0, wi = 0.0;
#pragma unroll
        for (int c = 0; c < D; c++) {
            const double2 m = M[r * D + c];
            wr = fma(m.x, xr[c], fma(-m.y, xi[c], wr));
            wi = fma(m.x, xi[c], fma(m.y, xr[c], wi));
        }
        st(p, base + off[r], Cx<T>{static_cast<T>(wr), static_cast<T>(wi)});
    }
}

template <typename T, int D>
__global__ void __launch_bounds__(kStepBlock)
    step_dense_kernel(Cx<T> *__restrict__ phi, SegPtrs<T> hp, const double2 *__restrict__ mats,
                      StepLaunch a, double *__restrict__ partials) {
    const double2 *U = mats;
    const double2 *G = mats + D * D;
    __shared__ double sacc[SEG_NJMAX * kStepBlock];
    for (int j = 0; j < a.nj; j++) {
        sacc[j * kStepBlock + threadIdx.x] = 0.0;
    }
    uint64_t off[D];
#pragma unroll
    for (int k = 0; k < D; k++) {
        off[k] = a.off[k];
    }
    for (uint64_t g = uint64_t{blockIdx.x} * kStepBlock + threadIdx.x; g < a.groups;
         g += uint64_t{gridDim.x} * kStepBlock) {
        uint64_t base = g;
#pragma unroll
        for (int q = 0; q < STEP_MMAX; q++) {
            if (q < a.m) {
                base = insert_zero(base, a.bits[q]);
            }
        }
        double vr[D], vi[D];
#pragma unroll
        for (int k = 0; k < D; k++) {
            const Cx<T> c = ld(phi, base + off[k]);
            vr[k] = c.r;
            vi[k] = c.i;
        }
        double gr[D], gi[D];
        if (a.trainable) {
#pragma unroll
            for (int r = 0; r < D; r++) {
                __asm__ volatile("" ::: "memory");
                double wr = 0.0, wi = 0.0;
#pragma unroll
                for (int c = 0; c < D; c++) {
                    const double2 m = G[r * D + c];
                    wr = fma(m.x, vr[c], fma(-m.y, vi[c], wr));
                    wi = fma(m.x, vi[c], fma(m.y, vr[c], wi));
                }
                gr[r] = wr;
                gi[r] = wi;
            }
        }
        // phi is read only here, so its update can be stored first and its
        // registers reused for the observable states.
        if (a.write_phi) {
            mat_store<T, D>(phi, base, off, U, vr, vi);
        }
        for (int j = 0; j < a.nj; j++) {
            Cx<T> *h = hp.p[j];
            double xr[D], xi[D];
#pragma unroll
            for (int k = 0; k < D; k++) {
                const Cx<T> c = ld(h, base + off[k]);
                xr[k] = c.r;
                xi[k] = c.i;
            }
            if (a.trainable) {
                double s = 0.0;
#pragma unroll
                for (int k = 0; k < D; k++) {
                    s = fma(xr[k], gi[k], fma(-xi[k], gr[k], s));
                }
                sacc[j * kStepBlock + threadIdx.x] += s;
            }
            mat_store<T, D>(h, base, off, U, xr, xi);
        }
    }
    if (a.trainable) {
        step_partials(sacc, a.nj, partials);
    }
}

// One group of a two-state step: the amplitudes of phi and of every observable
// state are loaded before any is used. M: U, then G, row-major.
template <typename T>
__device__ __forceinline__ void pair_update(Cx<T> *__restrict__ phi, const SegPtrs<T> &hp, uint64_t i0, uint64_t i1,
                                            const double2 *__restrict__ M, int nj, bool trainable, bool write_phi,
                                            double (&acc)[SEG_NJMAX]) {
    const double2 u0 = M[0], u1 = M[1], u2 = M[2], u3 = M[3];
    auto store = [&](Cx<T> *p, const Cx<T> &xa, const Cx<T> &xb) {
        const double ar = xa.r, ai = xa.i, br = xb.r, bi = xb.i;
        st(p, i0,
           Cx<T>{static_cast<T>(fma(u1.x, br, fma(-u1.y, bi, fma(u0.x, ar, -u0.y * ai)))),
                 static_cast<T>(fma(u1.x, bi, fma(u1.y, br, fma(u0.x, ai, u0.y * ar))))});
        st(p, i1,
           Cx<T>{static_cast<T>(fma(u3.x, br, fma(-u3.y, bi, fma(u2.x, ar, -u2.y * ai)))),
                 static_cast<T>(fma(u3.x, bi, fma(u3.y, br, fma(u2.x, ai, u2.y * ar))))});
    };
    const Cx<T> fa = ld(phi, i0), fb = ld(phi, i1);
    Cx<T> ha[SEG_NJMAX], hb[SEG_NJMAX];
#pragma unroll
    for (int j = 0; j < SEG_NJMAX; j++) {
        if (j < nj) {
            ha[j] = ld(hp.p[j], i0);
            hb[j] = ld(hp.p[j], i1);
        }
    }
    if (trainable) {
        const double2 g0 = M[4], g1 = M[5], g2 = M[6], g3 = M[7];
        const double ar = fa.r, ai = fa.i, br = fb.r, bi = fb.i;
        const double xr = fma(g1.x, br, fma(-g1.y, bi, fma(g0.x, ar, -g0.y * ai)));
        const double xi = fma(g1.x, bi, fma(g1.y, br, fma(g0.x, ai, g0.y * ar)));
        const double yr = fma(g3.x, br, fma(-g3.y, bi, fma(g2.x, ar, -g2.y * ai)));
        const double yi = fma(g3.x, bi, fma(g3.y, br, fma(g2.x, ai, g2.y * ar)));
#pragma unroll
        for (int j = 0; j < SEG_NJMAX; j++) {
            if (j < nj) {
                const double cr = ha[j].r, ci = ha[j].i, dr = hb[j].r, di = hb[j].i;
                acc[j] = fma(cr, xi, fma(-ci, xr, fma(dr, yi, fma(-di, yr, acc[j]))));
            }
        }
    }
    if (write_phi) {
        store(phi, fa, fb);
    }
#pragma unroll
    for (int j = 0; j < SEG_NJMAX; j++) {
        if (j < nj) {
            store(hp.p[j], ha[j], hb[j]);
        }
    }
}

// step_dense_kernel for a two-state subspace (DoubleExcitation moves 2 of its 16
// local states, SingleExcitation 2 of 4, CNOT-like gates 2). Such a step moves
// so little that latency counts: the amplitudes of phi and of every observable
// state are loaded before any is used, and the block sums take one barrier
// (block_total takes two per observable). 20 qubits complex128, five
// observables: 10.1 us a DoubleExcitation step (25 MB at 16 bytes of every 128-byte
// line its low wires split, and the launch), 17.4 us a SingleExcitation step (100
// MB, 5.8 TB/s), 4.2 and 6.1 us forward.
template <typename T>
__global__ void __launch_bounds__(kStepBlock)
    step_pair_kernel(Cx<T> *__restrict__ phi, SegPtrs<T> hp, const double2 *__restrict__ mats, StepLaunch a,
                     double *__restrict__ partials) {
    double acc[SEG_NJMAX];
#pragma unroll
    for (int j = 0; j < SEG_NJMAX; j++) {
        acc[j] = 0.0;
    }
    for (uint64_t g = uint64_t{blockIdx.x} * kStepBlock + threadIdx.x; g < a.groups;
         g += uint64_t{gridDim.x} * kStepBlock) {
        uint64_t base = g;
#pragma unroll
        for (int q = 0; q < STEP_MMAX; q++) {
            if (q < a.m) {
                base = insert_zero(base, a.bits[q]);
            }
        }
        pair_update(phi, hp, base + a.off[0], base + a.off[1], mats, a.nj, a.trainable != 0, a.write_phi != 0, acc);
    }
    if (!a.trainable) {
        return;
    }
    __shared__ double red[SEG_NJMAX][kStepBlock / 64];
#pragma unroll
    for (int j = 0; j < SEG_NJMAX; j++) {
        if (j < a.nj) {
            const double v = wave_sum(acc[j]);
            if ((threadIdx.x & 63) == 0) {
                red[j][threadIdx.x >> 6] = v;
            }
        }
    }
    __syncthreads();
    const int j = static_cast<int>(threadIdx.x);
    if (j < a.nj) {
        partials[static_cast<uint64_t>(j) * gridDim.x + blockIdx.x] = red[j][0] + red[j][1] + red[j][2] + red[j][3];
    }
}

// Consecutive two-state steps whose wires all lie in one set of at most
// kSlabBits state bits: a workgroup owns the slab of amplitudes that differ in
// those bits only and takes every step on it, with a barrier between steps, so
// that one launch replaces many.
// Bound: launch and ramp of a step (2 us between launches of a graph, and 2 to 4
// us until its loads return) where it moves little, HBM where it moves half the
// state. 20 qubits complex128, 5 observables, 180 excitations forward and back: 360
// launches, 3.4 ms busy and 0.8 ms between them, now 96 launches and 2.8 ms;
// 12 qubits, 90 excitations: 1.46 -> 1.06 ms a Jacobian. Without the lowest bits
// in the slab more steps share a launch, but each reads whole lines for a part
// of them: 3.8 ms a Jacobian with three of them, 4.0 with two, 6.2 with none.
template <typename T>
__global__ void __launch_bounds__(kSlabThreads)
    slab_steps_kernel(Cx<T> *__restrict__ phi, SegPtrs<T> hp, const unsigned char *__restrict__ mats,
                      const SlabStep *__restrict__ steps, SlabLaunch a, double *__restrict__ partials) {
    __shared__ uint64_t lo[64], hi[64]; // state offset of a slab index, six bits each
    __shared__ double red[2][SEG_NJMAX][kSlabThreads / 64];
    const int tid = static_cast<int>(threadIdx.x);
    if (tid < 128) {
        const int first = tid < 64 ? 0 : 6;
        uint64_t v = 0;
        for (int q = 0; q < 6; q++) {
            if (first + q < a.S && ((tid >> q) & 1)) {
                v |= uint64_t{1} << a.sb[first + q];
            }
        }
        (tid < 64 ? lo : hi)[tid & 63] = v;
    }
    uint64_t base = blockIdx.x;
    for (int q = 0; q < a.S; q++) {
        base = insert_zero(base, a.sb[q]);
    }
    __syncthreads();
    for (int s = 0; s < a.nsteps; s++) {
        const SlabStep &p = steps[s];
        const bool sums = a.nj > 0 && p.trainable != 0;
        const auto *M = reinterpret_cast<const double2 *>(mats + p.mats);
        double acc[SEG_NJMAX];
#pragma unroll
        for (int j = 0; j < SEG_NJMAX; j++) {
            acc[j] = 0.0;
        }
        for (int g = tid; g < (1 << (a.S - p.m)); g += kSlabThreads) {
            uint64_t l = static_cast<uint64_t>(g);
#pragma unroll
            for (int q = 0; q < STEP_MMAX; q++) {
                if (q < p.m) {
                    l = insert_zero(l, p.lb[q]);
                }
            }
            const uint64_t at = base | lo[l & 63] | hi[l >> 6];
            pair_update(phi, hp, at + p.off0, at + p.off1, M, a.nj, sums, true, acc);
        }
        if (sums) {
#pragma unroll
            for (int j = 0; j < SEG_NJMAX; j++) {
                if (j < a.nj) {
                    const double v = wave_sum(acc[j]);
                    if ((tid & 63) == 0) {
                        red[s & 1][j][tid >> 6] = v;
                    }
                }
            }
        }
        __syncthreads(); // the step's stores before the next one's loads; the sums
        if (sums && tid < a.nj) {
            double t = 0.0;
#pragma unroll
            for (int w = 0; w < kSlabThreads / 64; w++) {
                t += red[s & 1][tid][w];
            }
            partials[p.part + static_cast<uint64_t>(tid) * gridDim.x + blockIdx.x] = t;
        }
    }
}

// Parity phases: U multiplies amplitude i by ue or uo by the parity of
// i & umask; G multiplies it by +1 / -1 by the parity of i & gmask.
template <typename T>
__global__ void __launch_bounds__(kStepBlock)
    step_parity_kernel(Cx<T> *__restrict__ phi, SegPtrs<T> hp, StepLaunch a,
                       double *__restrict__ partials) {
    __shared__ double sacc[SEG_NJMAX * kStepBlock];
    for (int j = 0; j < a.nj; j++) {
        sacc[j * kStepBlock + threadIdx.x] = 0.0;
    }
    for (uint64_t i = uint64_t{blockIdx.x} * kStepBlock + threadIdx.x; i < a.groups;
         i += uint64_t{gridDim.x} * kStepBlock) {
        const bool uodd = __popcll(i & a.umask) & 1;
        const double pr = uodd ? a.uo[0] : a.ue[0];
        const double pi = uodd ? a.uo[1] : a.ue[1];
        const double sg = (__popcll(i & a.gmask) & 1) ? -1.0 : 1.0;
        const Cx<T> v = ld(phi, i);
        const double gr = sg * static_cast<double>(v.r), gi = sg * static_cast<double>(v.i);
        for (int j = 0; j < a.nj; j++) {
            Cx<T> *h = hp.p[j];
            const Cx<T> x = ld(h, i);
            const double xr = x.r, xi = x.i;
            if (a.trainable) {
                sacc[j * kStepBlock + threadIdx.x] += fma(xr, gi, -xi * gr);
            }
            st(h, i, Cx<T>{static_cast<T>(pr * xr - pi * xi), static_cast<T>(pr * xi + pi * xr)});
        }
        if (a.write_phi) {
            const double xr = v.r, xi = v.i;
            st(phi, i, Cx<T>{static_cast<T>(pr * xr - pi * xi), static_cast<T>(pr * xi + pi * xr)});
        }
    }
    if (a.trainable) {
        step_partials(sacc, a.nj, partials);
    }
}

template <typename T>
void launch_step_t(Device &dev, const State &phi, void *const *h_ptrs, const void *d_mats,
                   const StepLaunch &L, double *partials) {
    SegPtrs<T> hp{};
    for (int j = 0; j < L.nj; j++) {
        hp.p[j] = static_cast<Cx<T> *>(h_ptrs[j]);
    }
    const unsigned grid = static_cast<unsigned>(step_blocks(dev, L));
    const double bytes = (1.0 + L.write_phi + 2.0 * L.nj) * static_cast<double>(phi.bytes());
    ProfScope prof(L.nj > 0 ? "adjoint_step" : "apply_step", bytes, dev.stream);
    auto *p = static_cast<Cx<T> *>(phi.d);
    const auto *m = static_cast<const double2 *>(d_mats);
    switch (L.m == 0 ? 0 : L.dim) {
    case 0:
        hipLaunchKernelGGL((step_parity_kernel<T>), dim3(grid), dim3(kStepBlock), 0, dev.stream, p,
                           hp, L, partials);
        break;
    case 2:
        hipLaunchKernelGGL(step_pair_kernel<T>, dim3(grid), dim3(kStepBlock), 0, dev.stream, p, hp, m, L,
                           partials);
        break;
    case 4:
        hipLaunchKernelGGL((step_dense_kernel<T, 4>), dim3(grid), dim3(kStepBlock), 0, dev.stream,
                           p, hp, m, L, partials);
        break;
    case 8:
        hipLaunchKernelGGL((step_dense_kernel<T, 8>), dim3(grid), dim3(kStepBlock), 0, dev.stream,
                           p, hp, m, L, partials);
        break;
    case 16:
        hipLaunchKernelGGL((step_dense_kernel<T, 16>), dim3(grid), dim3(kStepBlock), 0, dev.stream,
                           p, hp, m, L, partials);
        break;
    default:
        raise(PLK_ERR_INVALID, "single-op step kernels take subspaces of 2, 4, 8 or 16 states");
    }
    PLK_HIP(hipGetLastError());
}

} // namespace

void launch_slab_steps(Device &dev, const State &phi, void *const *h_ptrs, const unsigned char *d_mats,
                       const unsigned char *d_steps, const SlabLaunch &L, double *partials) {
    bool ok = L.n == phi.n && L.S >= 1 && L.S <= std::min(L.n, kSlabBits) && L.nj >= 0 && L.nj <= SEG_NJMAX &&
              L.nsteps >= 1 && (L.nj == 0 || partials != nullptr);
    for (int q = 0; ok && q < L.S; q++) {
        ok = L.sb[q] >= 0 && L.sb[q] < L.n && (q == 0 || L.sb[q] > L.sb[q - 1]);
    }
    if (!ok) {
        raise(PLK_ERR_INVALID, "single-op steps do not match the state");
    }
    const uint64_t slabs = uint64_t{1} << (L.n - L.S);
    if (slabs > (uint64_t{1} << 31) - 1) {
        raise(PLK_ERR_UNSUPPORTED, "single-op steps: too many slabs");
    }
    ProfScope prof(L.nj > 0 ? "adjoint_step" : "apply_step",
                   L.nsteps * (2.0 + 2.0 * L.nj) * static_cast<double>(phi.bytes()), dev.stream);
    auto go = [&](auto tag) {
        using T = decltype(tag);
        SegPtrs<T> hp{};
        for (int j = 0; j < L.nj; j++) {
            hp.p[j] = static_cast<Cx<T> *>(h_ptrs[j]);
        }
        hipLaunchKernelGGL(slab_steps_kernel<T>, dim3(static_cast<unsigned>(slabs)), dim3(kSlabThreads), 0,
                           dev.stream, static_cast<Cx<T> *>(phi.d), hp, d_mats,
                           reinterpret_cast<const SlabStep *>(d_steps), L, partials);
    };
    if (phi.dtype == PLK_C64) {
        go(float{});
    } else {
        go(double{});
    }
    PLK_HIP(hipGetLastError());
}

int step_blocks(const Device &dev, const StepLaunch &L) {
    const uint64_t blocks = (L.groups + kStepBlock - 1) / kStepBlock;
    return static_cast<int>(
        std::max<uint64_t>(1, std::min<uint64_t>(blocks, static_cast<uint64_t>(dev.num_cus) * 8)));
}

void launch_step(Device &dev, const State &phi, void *const *h_ptrs, const void *d_mats,
                 const StepLaunch &L, double *partials) {
    if (L.nj < 0 || L.nj > SEG_NJMAX) {
        raise(PLK_ERR_INVALID, "single-op step: observable chunk out of range");
    }
    if (L.m != 0 && (L.m < 1 || L.m > STEP_MMAX || d_mats == nullptr || L.dim < 2 ||
                     L.dim > (1 << L.m))) {
        raise(PLK_ERR_INVALID, "single-op step: bad matrix width");
    }
    if (L.m > 0 && (uint64_t{1} << L.m) * L.groups != phi.len) {
        raise(PLK_ERR_INVALID, "single-op step: groups do not cover the state");
    }
    if (L.m == 0 && L.groups != phi.len) {
        raise(PLK_ERR_INVALID, "single-op step: parity step must cover the state");
    }
    if (L.trainable && L.nj > 0 && partials == nullptr) {
        raise(PLK_ERR_INVALID, "single-op step: no buffer for the partial sums");
    }
    if (phi.dtype == PLK_C64) {
        launch_step_t<float>(dev, phi, h_ptrs, d_mats, L, partials);
    } else {
        launch_step_t<double>(dev, phi, h_ptrs, d_mats, L, partials);
    }
}

} // namespace plk
