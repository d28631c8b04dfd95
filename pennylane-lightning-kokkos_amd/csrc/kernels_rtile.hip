// Register-tile passes: many fused operations per HBM pass, with the tile in
// VGPRs instead of LDS.
//
// Each wavefront owns one tile at a time: the 2^(R+6) amplitudes whose index
// bits outside the pass's tile bits are fixed. Every lane holds 2^R of them
// per state (R register bits); the 6 lane bits select the lane. Which tile
// bit sits on which register bit or lane position is the pass's layout,
// chosen on the host and changed by remaps.
//
// A pass program is a list of fixed-size instructions read through the scalar
// cache: a 32-byte header and the eight reals most operations need. The next
// instruction is fetched while the current one runs, so its latency is off
// the critical path; only wider payloads are read where they are used. An
// instruction first applies up to two remaps -- exchanges of a register bit
// with a lane position, in place -- then one operation:
//   RT_REG1   one wire on register bit a;
//   RT_REG2   two wires on register bits a > b;
//   RT_SEL    mixing register bit a, with the op's other wire on lane position
//             s0: each lane applies the 2x2 block its lane bit selects
//             (controlled gates with the control on a lane, diagonal gates
//             across a register and a lane bit);
//   RT_LANE   diagonal on lane positions only: one factor per lane.
// A selector s0 / s1 of 64 + b names a global index bit b outside the tile
// instead of a lane: its value is fixed for the whole tile, so an operation
// whose non-mixing wires (a control, a diagonal factor) lie outside the tile
// needs no tile bit for them, and RT_SEL becomes RT_REG1 with one block.
//
// Operations work in place on the register tile. A second copy of one state
// (out-of-place application through a rotating spare buffer) costs a quarter
// of the registers at four states and unrolls the whole instruction switch
// once per buffer position: 398 KB of code against a 64 KB instruction cache.
// In place the four-state kernel has 164 KB, of which a pass runs a part, and
// 168 VGPRs (three waves per SIMD instead of two).
//
// Bound (24 qubits complex128, 9 observables, 29 passes of 33 gates, 1.61 ms a
// pass = 3.3 TB/s of the in-place ceiling of 5.2): FP64 issue, busy 65 to 73 % at
// the 2.0 GHz the card holds under this load, and memory, for which the waves
// wait 30 % of their time; out of place with five mixed bits a pass it was 50
// passes of 1.74 ms. One state (26-qubit stream of 600 gates, 32 amplitudes a
// lane): 25 passes of 0.53 ms, 4.1 TB/s; with 16 amplitudes 29 passes of 0.53,
// with 8 and no exchange below position 4, 66 of 0.47.
//
// The host fuses the one-wire gates that follow each other on a wire into one
// 2x2 matrix. For trainable gates V_1, V_2, ... of such a run the derivative
// of the k-th is Im<h| (V_{k-1}...V_1)^dag G_k (V_{k-1}...V_1) |phi> with phi
// and h as they enter the run, and that operator is a real combination of X,
// Y and Z of the wire. So the run adds the FP64 sums Im<h_j|X phi>,
// Im<h_j|Y phi>, Im<h_j|Z phi> once (only those it needs) and the reduction
// forms every gate's derivative from them.
//
// The lanes of two quads are summed by DPP and one lane adds the total into
// LDS (ds_add_f64, one address per two quads, so the order is fixed). After
// its last tile the wavefront writes per-block partials; a second kernel sums
// them in a fixed order. No LDS staging of states and no barriers: each
// wavefront streams its tiles independently.
#include "rtile_device.hpp"

namespace plk {

namespace {

// Observable-state pointers of one launch: nc chunks of NJ states.
template <typename T> struct RtPtrs {
    Cx<T> *p[RT_OBS_MAX];
};

// C: precision of the program and of the registers.
template <typename T, int NJ, int R, typename C>
__global__ void __launch_bounds__(64, (rt_waves<C, NJ, R>()))
    rtile_kernel(Cx<T> *phi, Cx<T> *phi_out, RtPtrs<T> hp, const unsigned char *__restrict__ prog_g,
                 RtLaunch L, double *__restrict__ partials) {
    constexpr int A = 1 << R;
    constexpr int NS = NJ + 1;
    // Block -> (chunk c, block b of that chunk). Ids are taken in groups of
    // xgroup (consecutive ids land on different XCDs), so the nc blocks that
    // stream the same tiles for different chunks share an XCD and its L2.
    const int nc = L.nc;
    const unsigned xg = static_cast<unsigned>(L.xgroup);
    const unsigned kq = blockIdx.x / xg;
    const int c = static_cast<int>(kq % static_cast<unsigned>(nc));
    const unsigned b = (kq / static_cast<unsigned>(nc)) * xg + blockIdx.x % xg;
    const unsigned bpc = gridDim.x / static_cast<unsigned>(nc);
    const bool writes_phi = L.write_phi && c == nc - 1;
    // This chunk's states and its first state in the launch: nbig chunks of
    // NJ, then chunks of NJ - 1 (their last register state stays unused).
    const int njc = c < L.nbig ? NJ : NJ - 1;
    const int jc0 = c < L.nbig ? c * NJ : L.nbig * NJ + (c - L.nbig) * (NJ - 1);
    const int width = L.nbig * NJ + (nc - L.nbig) * (NJ - 1);
    // FP64 sums [slot * NJ + j][cell], then one dummy slot per lane.
    extern __shared__ double lacc[];
    const int lane = static_cast<int>(__lane_id());
    const int dummy = L.nslots * NJ * RT_CELLS;
    if constexpr (NJ > 0) {
        for (int i = lane; i < dummy; i += 64) {
            lacc[i] = 0.0;
        }
    }
    CT<unsigned char> *prog = (CT<unsigned char> *)(prog_g);
    Cx<T> *sp[NS];
    sp[0] = phi;
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        sp[j + 1] = j < njc ? hp.p[jc0 + j] : phi;
    }
    // Per-lane byte offsets of the load and store layouts; the tile base and
    // the register slot's offset are uniform.
    uint64_t vin = 0, vout = 0;
#pragma unroll
    for (int p = 0; p < RT_LANE_BITS; p++) {
        vin |= static_cast<uint64_t>(lbit(lane, p)) << L.lane_in[p];
        vout |= static_cast<uint64_t>(lbit(lane, p)) << L.lane_out[p];
    }
    vin *= sizeof(Cx<T>);
    vout *= sizeof(Cx<T>);
    const uint64_t ntiles = uint64_t{1} << (L.n - L.T);
    const Ins<C> first = fetch<C>(prog, 0);
    for (uint64_t g = b; g < ntiles; g += bpc) {
        uint64_t base = g;
        for (int q = 0; q < L.T; q++) {
            base = insert_zero(base, L.tb[q]);
        }
        Cx<C> v[NS][A];
#pragma unroll
        for (int s = 0; s < NS; s++) {
            if (s > njc) {
#pragma unroll
                for (int k = 0; k < A; k++) {
                    v[s][k] = Cx<C>{C(0), C(0)};
                }
                continue;
            }
#pragma unroll
            for (int k = 0; k < A; k++) {
                const Cx<T> x = ldo(sp[s], base * sizeof(Cx<T>) + slot_off<T, R>(L.reg_in, k) + vin);
                v[s][k] = Cx<C>{static_cast<C>(x.r), static_cast<C>(x.i)};
            }
        }
        run_program<C, NS, R>(v, first, prog, L.ninstr, lacc, dummy, lane, base);
#pragma unroll
        for (int s = 0; s < NS; s++) {
            if ((s == 0 && !writes_phi) || s > njc) {
                continue;
            }
            Cx<T> *dst = s == 0 ? phi_out : sp[s];
#pragma unroll
            for (int k = 0; k < A; k++) {
                sto(dst, base * sizeof(Cx<T>) + slot_off<T, R>(L.reg_out, k) + vout,
                    Cx<T>{static_cast<T>(v[s][k].r), static_cast<T>(v[s][k].i)});
            }
        }
    }
    if constexpr (NJ > 0) {
        __syncthreads();
        const int per = L.nslots * NJ;
        for (int i = lane; i < per; i += 64) {
            double s = 0.0;
#pragma unroll
            for (int q = 0; q < RT_CELLS; q++) {
                s += lacc[i * RT_CELLS + q];
            }
            // Local (slot, j) -> launch-wide (slot, jc0 + j).
            const int slot = i / NJ, j = i % NJ;
            if (j < njc) {
                const uint64_t row = static_cast<uint64_t>(slot) * width + jc0 + j;
                partials[row * bpc + b] = s;
            }
        }
    }
}

} // namespace

// f(R, C) for the launch's register bits and its program's precision.
template <typename T, int NJ, int R = rt_reg_min<T>(NJ), typename F> void with_reg(const RtLaunch &L, F &&f) {
    if constexpr (R < rt_reg_max<T>(NJ)) {
        if (L.R != R) {
            with_reg<T, NJ, R + 1>(L, f);
            return;
        }
    }
    if constexpr (NJ == 0) {
        if (L.wide) {
            f(IC<R>{}, double{});
            return;
        }
    }
    f(IC<R>{}, T{});
}

template <typename T, int NJ, int R, typename C> int blocks_per_chunk(const Device &dev, const RtLaunch &L, int nc) {
    const void *kfn = reinterpret_cast<const void *>(&rtile_kernel<T, NJ, R, C>);
    const size_t lds = rt_lds_bytes(NJ, L.nslots);
    static int per_cu[RT_SLOTS_MAX + 1] = {}; // by slots: the kernel's LDS follows from them
    int &nb = per_cu[NJ > 0 ? L.nslots : 0];
    if (nb == 0) {
        PLK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kfn, 64, lds));
        nb = std::max(1, std::min(nb, 32));
    }
    const uint64_t ntiles = uint64_t{1} << (L.n - L.T);
    const uint64_t cap = static_cast<uint64_t>(dev.num_cus) * nb;
    uint64_t bpc = std::max<uint64_t>(1, std::min(ntiles, cap / static_cast<uint64_t>(nc)));
    // Without sums a block costs nothing to start: a block a tile lets the
    // hardware even out the wavefronts' speeds (resident blocks end between 70 %
    // and 100 % of a pass). 26-qubit stream of 400 gates: complex128 10.4 -> 9.7 ms,
    // complex64 (an FP64 program) 7.7 -> 7.2. From four rounds on: with 2 to 2.7 (24
    // qubits) the last round is too empty, 2.49 -> 2.60 and 1.97 -> 2.06 ms.
    if (NJ == 0 && ntiles >= 4 * cap) {
        bpc = ntiles;
    }
    if (bpc >= 8) {
        bpc = bpc / 8 * 8;
    }
    return static_cast<int>(bpc);
}

// Blocks per chunk of a launch: the chunks share the resident blocks; in
// groups of 8 (one per XCD) when there are enough.
template <typename T, int NJ> int rtile_blocks_t(const Device &dev, const RtLaunch &L, int nc) {
    int blocks = 0;
    with_reg<T, NJ>(L, [&](auto R, auto C) {
        blocks = blocks_per_chunk<T, NJ, decltype(R)::value, decltype(C)>(dev, L, nc);
    });
    return blocks;
}

// Launcher of one (precision, observable chunk) variant. The build compiles
// this file once per variant with PLK_RT_T and PLK_RT_NJ defined, so the
// variants compile in parallel.
template <typename T, int NJ>
void rtile_launch_t(Device &dev, const State &phi, void *phi_out, void *const *h_ptrs,
                    const void *d_prog, const RtLaunch &Lin, int bpc, double *partials) {
    RtLaunch L = Lin;
    L.xgroup = bpc >= 8 ? 8 : 1;
    const int width = rt_width(L);
    RtPtrs<T> hp{};
    for (int j = 0; j < width; j++) {
        hp.p[j] = static_cast<Cx<T> *>(h_ptrs[j]);
    }
    const unsigned grid = static_cast<unsigned>(bpc) * static_cast<unsigned>(L.nc);
    // Algorithmic bytes: phi read once and written once, every observable
    // state read and written once.
    const double bytes = (1.0 + L.write_phi + 2.0 * width) * static_cast<double>(phi.bytes());
    ProfScope prof(NJ > 0 ? "adjoint_rtile" : "apply_rtile", bytes, dev.stream);
    with_reg<T, NJ>(L, [&](auto R, auto C) {
        hipLaunchKernelGGL((rtile_kernel<T, NJ, decltype(R)::value, decltype(C)>), dim3(grid), dim3(64),
                           rt_lds_bytes(NJ, L.nslots), dev.stream, static_cast<Cx<T> *>(phi.d),
                           static_cast<Cx<T> *>(phi_out), hp, static_cast<const unsigned char *>(d_prog), L,
                           partials);
    });
    PLK_HIP(hipGetLastError());
}

#if defined(PLK_RT_T) && defined(PLK_RT_NJ)
template int rtile_blocks_t<PLK_RT_T, PLK_RT_NJ>(const Device &, const RtLaunch &, int);
template void rtile_launch_t<PLK_RT_T, PLK_RT_NJ>(Device &, const State &, void *, void *const *, const void *,
                                                  const RtLaunch &, int, double *);
#endif

} // namespace plk
