// Device side of register-tile programs (see kernels_rtile.hip for the tile,
// the instructions and what bounds them): instruction fetch, remaps, in-place
// operations and the FP64 sums of trainable instructions, shared by the pass
// kernel and the whole-circuit kernel.
#pragma once

#include "device_common.hpp"

namespace plk {

template <typename T> using CT = const __attribute__((address_space(4))) T;

__device__ __forceinline__ bool lbit(int lane, int p) { return (lane >> p) & 1; }

// Block selector of RT_SEL / RT_LANE: a lane position (0-5), or 64 + a
// global index bit outside the tile, whose value is the same for the whole
// tile (tbase: the tile's first amplitude index).
__device__ __forceinline__ bool selbit(int lane, uint64_t tbase, int s) {
    return s < 64 ? lbit(lane, s) : ((tbase >> (s - 64)) & 1);
}

// ---------------------------------------------------------------------------
// Remap: exchange register bit Q with lane position P, in place. Afterwards
// lanes whose lane bit P is 1 hold the partner's b in a, and lanes whose bit
// is 0 hold the partner's a in b. Positions 5 and 4 are one
// v_permlane32/16_swap per 32-bit word pair; the others take three
// instructions (DPP within the 16-lane row: rotate by 8 or shift by 4 with
// the bank mask selecting the lanes written, quad permutations with selects).
// So any of a tile's bits can be mixed in a pass, 9 to 11 instead of the 5 or
// 6 that registers and positions 5 and 4 hold.
// ---------------------------------------------------------------------------
template <int P> __device__ __forceinline__ void xchg_word(uint32_t &a, uint32_t &b, int lane) {
    const int ia = static_cast<int>(a), ib = static_cast<int>(b);
    if constexpr (P == 5) {
        const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
        a = r[0];
        b = r[1];
    } else if constexpr (P == 4) {
        const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
        a = r[0];
        b = r[1];
    } else if constexpr (P == 3) {
        a = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(ia, ib, 0x128, 0xF, 0xC, false));
        b = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(ib, ia, 0x128, 0xF, 0x3, false));
    } else if constexpr (P == 2) {
        a = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(ia, ib, 0x114, 0xF, 0xA, false));
        b = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(ib, ia, 0x104, 0xF, 0x5, false));
    } else {
        constexpr int ctrl = P == 1 ? 0x4E : 0xB1;
        const bool hi = lbit(lane, P);
        const int s = hi ? ia : ib;
        const int r = __builtin_amdgcn_mov_dpp(s, ctrl, 0xF, 0xF, false);
        a = static_cast<uint32_t>(hi ? r : ia);
        b = static_cast<uint32_t>(hi ? ib : r);
    }
}

template <int P> __device__ __forceinline__ void xchg(double &a, double &b, int lane) {
    uint64_t ua = __double_as_longlong(a), ub = __double_as_longlong(b);
    uint32_t a0 = static_cast<uint32_t>(ua), a1 = static_cast<uint32_t>(ua >> 32);
    uint32_t b0 = static_cast<uint32_t>(ub), b1 = static_cast<uint32_t>(ub >> 32);
    xchg_word<P>(a0, b0, lane);
    xchg_word<P>(a1, b1, lane);
    a = __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(a1) << 32) | a0));
    b = __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(b1) << 32) | b0));
}

template <int P> __device__ __forceinline__ void xchg(float &a, float &b, int lane) {
    uint32_t ua = __float_as_uint(a), ub = __float_as_uint(b);
    xchg_word<P>(ua, ub, lane);
    a = __uint_as_float(ua);
    b = __uint_as_float(ub);
}

template <int R, int Q = 0, typename F> __device__ __forceinline__ void dispatch_q(int q, F &&f) {
    if constexpr (Q + 1 >= R) {
        f(IC<Q>{});
    } else if (q == Q) {
        f(IC<Q>{});
    } else {
        dispatch_q<R, Q + 1>(q, f);
    }
}

// Register bits a > b.
template <int R, int QA = 1, int QB = 0, typename F>
__device__ __forceinline__ void dispatch_q2(int a, int b, F &&f) {
    if constexpr (QA + 1 >= R && QB + 1 >= QA) {
        f(IC<QA>{}, IC<QB>{});
    } else if (a == QA && b == QB) {
        f(IC<QA>{}, IC<QB>{});
    } else {
        dispatch_q2<R, QB + 1 < QA ? QA : QA + 1, QB + 1 < QA ? QB + 1 : 0>(a, b, f);
    }
}

template <typename T, int NS, int A, int Q, int P>
__device__ __forceinline__ void remap_qp(Cx<T> (&v)[NS][A], int lane) {
#pragma unroll
    for (int s = 0; s < NS; s++) {
#pragma unroll
        for (int k = 0; k < A; k++) {
            if (k & (1 << Q)) {
                continue;
            }
            xchg<P>(v[s][k].r, v[s][k | (1 << Q)].r, lane);
            xchg<P>(v[s][k].i, v[s][k | (1 << Q)].i, lane);
        }
    }
}

template <typename T, int NS, int R>
__device__ __forceinline__ void remap(Cx<T> (&v)[NS][1 << R], int q, int p, int lane) {
    constexpr int A = 1 << R;
    dispatch_q<R>(q, [&](auto Qc) {
        constexpr int Q = decltype(Qc)::value;
        if (p >= 4) {
            if (p == 5) {
                remap_qp<T, NS, A, Q, 5>(v, lane);
            } else {
                remap_qp<T, NS, A, Q, 4>(v, lane);
            }
        } else if (p >= 2) {
            if (p == 3) {
                remap_qp<T, NS, A, Q, 3>(v, lane);
            } else {
                remap_qp<T, NS, A, Q, 2>(v, lane);
            }
        } else if (p == 1) {
            remap_qp<T, NS, A, Q, 1>(v, lane);
        } else {
            remap_qp<T, NS, A, Q, 0>(v, lane);
        }
    });
}

// One instruction in scalar registers.
template <typename T> struct Ins {
    int32_t w[8];
    T u[8];
};

template <typename T>
__device__ __forceinline__ Ins<T> fetch(CT<unsigned char> *prog, int pc) {
    CT<unsigned char> *p = prog + static_cast<int64_t>(pc) * rt_stride<T>();
    Ins<T> in;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        in.w[k] = reinterpret_cast<CT<int32_t> *>(p)[k];
    }
#pragma unroll
    for (int k = 0; k < 8; k++) {
        in.u[k] = reinterpret_cast<CT<T> *>(p + 32)[k];
    }
    return in;
}

// ---------------------------------------------------------------------------
// FP64 sums of a trainable instruction: NV values per lane, summed by DPP over
// the quad, then over two quads of the 16-lane row (lane r of a quad for values
// r, r + 4, ...: every lane holds every total of its quad), and added into one
// of the value's RT_CELLS cells in LDS; lanes without a value or cell add to a
// dummy slot of their own. No branch on the lane, so the instruction switch
// around this stays free of divergent control flow. A cell per quad instead
// took twice the LDS: passes of more than 30 sums of three states then fitted
// fewer than the three wavefronts per SIMD that their registers allow, and ran
// in two rounds (24 qubits complex128, 33 sums: 2.5 to 2.9 ms, now 1.9 to 2.2).
// ---------------------------------------------------------------------------
template <int CTRL> __device__ __forceinline__ double dpp_f64(double v) {
    const uint64_t b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp(static_cast<int>(b & 0xffffffffu), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp(static_cast<int>(b >> 32), CTRL, 0xF, 0xF, false);
    return __longlong_as_double(static_cast<long long>(
        (static_cast<uint64_t>(static_cast<uint32_t>(hi)) << 32) | static_cast<uint32_t>(lo)));
}

template <int NV>
__device__ __forceinline__ void add_slots(double (&d)[NV], double *lacc, int base, int dummy, int lane) {
#pragma unroll
    for (int v = 0; v < NV; v++) {
        d[v] += dpp_f64<0xB1>(d[v]); // quad_perm [1,0,3,2]
        d[v] += dpp_f64<0x4E>(d[v]); // quad_perm [2,3,0,1]
    }
    const int r = lane & 3;
    const int cell = ((lane >> 4) << 1) | ((lane >> 2) & 1);
#pragma unroll
    for (int v0 = 0; v0 < NV; v0 += 4) {
        double x = d[v0];
#pragma unroll
        for (int v = v0 + 1; v < v0 + 4 && v < NV; v++) {
            x = (r == v - v0) ? d[v] : x;
        }
        const bool full = v0 + 4 <= NV;
        x += dpp_f64<0x128>(x); // row_ror:8
        const bool mine = (lane & 8) == 0 && (full || v0 + r < NV);
        const int idx = mine ? (base + v0 + r) * RT_CELLS + cell : dummy + lane;
        atomicAdd(&lacc[idx], x);
    }
}

template <typename T> struct Dx {
    double r, i;
};
template <typename T> __device__ __forceinline__ Dx<T> wide(const Cx<T> &c) {
    return {static_cast<double>(c.r), static_cast<double>(c.i)};
}
// s + Im(conj(h) g), s + Re(conj(h) g) and their negatives.
template <typename T> __device__ __forceinline__ double im_add(double s, const Dx<T> &h, const Dx<T> &g) {
    return fma(h.r, g.i, fma(-h.i, g.r, s));
}
template <typename T> __device__ __forceinline__ double im_sub(double s, const Dx<T> &h, const Dx<T> &g) {
    return fma(-h.r, g.i, fma(h.i, g.r, s));
}
template <typename T> __device__ __forceinline__ double re_add(double s, const Dx<T> &h, const Dx<T> &g) {
    return fma(h.r, g.r, fma(h.i, g.i, s));
}
template <typename T> __device__ __forceinline__ double re_sub(double s, const Dx<T> &h, const Dx<T> &g) {
    return fma(-h.r, g.r, fma(-h.i, g.i, s));
}

// Sums over the pairs of register bit Q: Im<h_j|P phi> for P = X (bit 0 of
// C), Y (bit 1), Z (bit 2), in that order.
template <typename T, int NS, int A, int Q, int C>
__device__ __forceinline__ void acc_pauli(const Cx<T> (&v)[NS][A], double *lacc, int slot, int dummy, int lane) {
    constexpr int NJ = NS - 1;
    constexpr int NC = (C & 1) + ((C >> 1) & 1) + (C >> 2);
    constexpr int OY = C & 1, OZ = (C & 1) + ((C >> 1) & 1);
    double d[NC * NJ];
#pragma unroll
    for (int e = 0; e < NC * NJ; e++) {
        d[e] = 0.0;
    }
#pragma unroll
    for (int k = 0; k < A; k++) {
        if (k & (1 << Q)) {
            continue;
        }
        const Dx<T> f0 = wide(v[0][k]), f1 = wide(v[0][k | (1 << Q)]);
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const Dx<T> h0 = wide(v[j + 1][k]), h1 = wide(v[j + 1][k | (1 << Q)]);
            if constexpr (C & 1) {
                d[j] = im_add(im_add(d[j], h0, f1), h1, f0);
            }
            if constexpr (C & 2) {
                // (Y f)_0 = -i f_1, (Y f)_1 = i f_0.
                d[OY * NJ + j] = re_add(re_sub(d[OY * NJ + j], h0, f1), h1, f0);
            }
            if constexpr (C & 4) {
                d[OZ * NJ + j] = im_sub(im_add(d[OZ * NJ + j], h0, f0), h1, f1);
            }
        }
    }
    add_slots<NC * NJ>(d, lacc, slot * NJ, dummy, lane);
}

// Sums Im<h_j|G phi> for a 2x2 generator on register bit Q: real diagonal
// (g[0], g[1]) or dense (row-major complex).
template <typename T, int NS, int A, int Q, bool DIAG>
__device__ __forceinline__ void acc_gen1(const Cx<T> (&v)[NS][A], const T *g, double *lacc, int slot, int dummy,
                                         int lane) {
    constexpr int NJ = NS - 1;
    double d[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        d[j] = 0.0;
    }
#pragma unroll
    for (int k = 0; k < A; k++) {
        if (k & (1 << Q)) {
            continue;
        }
        const Cx<T> f0 = v[0][k], f1 = v[0][k | (1 << Q)];
        Cx<T> g0, g1;
        if constexpr (DIAG) {
            g0 = {g[0] * f0.r, g[0] * f0.i};
            g1 = {g[1] * f1.r, g[1] * f1.i};
        } else {
            g0 = cmad(Cx<T>{g[2], g[3]}, f1, cmul(Cx<T>{g[0], g[1]}, f0));
            g1 = cmad(Cx<T>{g[6], g[7]}, f1, cmul(Cx<T>{g[4], g[5]}, f0));
        }
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            d[j] = im_add(im_add(d[j], wide(v[j + 1][k]), wide(g0)), wide(v[j + 1][k | (1 << Q)]), wide(g1));
        }
    }
    add_slots<NJ>(d, lacc, slot * NJ, dummy, lane);
}

template <int QA, int QB> __device__ __forceinline__ constexpr int lidx(int k) {
    return (((k >> QA) & 1) << 1) | ((k >> QB) & 1);
}

// Sums Im<h_j|G phi> for a 4x4 generator on register bits QA > QB: KIND
// G_Z (parity sign), G_DIAG (four reals) or G_DENSE (row-major complex).
template <typename T, int NS, int A, int QA, int QB, int KIND>
__device__ __forceinline__ void acc_gen2(const Cx<T> (&v)[NS][A], CT<T> *G, double *lacc, int slot, int dummy,
                                         int lane) {
    constexpr int NJ = NS - 1;
    constexpr int MQ = (1 << QA) | (1 << QB);
    double d[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        d[j] = 0.0;
    }
#pragma unroll
    for (int k = 0; k < A; k++) {
        if (k & MQ) {
            continue;
        }
        const int idx[4] = {k, k | (1 << QB), k | (1 << QA), k | MQ};
#pragma unroll
        for (int r = 0; r < 4; r++) {
            Cx<T> t;
            if constexpr (KIND == G_Z) {
                const Cx<T> f = v[0][idx[r]];
                t = (r == 1 || r == 2) ? Cx<T>{-f.r, -f.i} : f;
            } else if constexpr (KIND == G_DIAG) {
                const Cx<T> f = v[0][idx[r]];
                t = {G[r] * f.r, G[r] * f.i};
            } else {
                t = cmul(Cx<T>{G[8 * r], G[8 * r + 1]}, v[0][idx[0]]);
#pragma unroll
                for (int c = 1; c < 4; c++) {
                    t = cmad(Cx<T>{G[8 * r + 2 * c], G[8 * r + 2 * c + 1]}, v[0][idx[c]], t);
                }
            }
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                d[j] = im_add(d[j], wide(v[j + 1][idx[r]]), wide(t));
            }
        }
    }
    add_slots<NJ>(d, lacc, slot * NJ, dummy, lane);
}

// ---------------------------------------------------------------------------
// In-place operations on every state.
//
// Each result is formed as (sum of the other terms) + u x with x the register
// it replaces, and the last step is written as an instruction whose
// destination is that register: the compiler's own choice, v_fmac, puts the
// result into the other terms' register and copies it back (one v_mov_b64 per
// result, a fifth of the kernel's vector instructions).
// ---------------------------------------------------------------------------
// x = u x + t; u uniform (scalar register) or per lane.
template <bool UNI> __device__ __forceinline__ void fma_ip(double &x, double u, double t) {
    if constexpr (UNI) {
        asm("v_fma_f64 %0, %1, %0, %2" : "+v"(x) : "s"(u), "v"(t));
    } else {
        asm("v_fma_f64 %0, %1, %0, %2" : "+v"(x) : "v"(u), "v"(t));
    }
}
template <bool UNI> __device__ __forceinline__ void fma_ip(float &x, float u, float t) {
    if constexpr (UNI) {
        asm("v_fma_f32 %0, %1, %0, %2" : "+v"(x) : "s"(u), "v"(t));
    } else {
        asm("v_fma_f32 %0, %1, %0, %2" : "+v"(x) : "v"(u), "v"(t));
    }
}

// x = u x for complex u.
template <bool UNI, typename T> __device__ __forceinline__ void scale_ip(Cx<T> &x, T ur, T ui) {
    const T tr = -ui * x.i, ti = ui * x.r;
    fma_ip<UNI>(x.r, ur, tr);
    fma_ip<UNI>(x.i, ur, ti);
}

// Exchange of x and y, on every lane or on the lanes of `mask` (all lanes
// are active here).
template <bool ALL> __device__ __forceinline__ void swap_words(uint32_t &x0, uint32_t &y0, uint32_t &x1, uint32_t &y1,
                                                               uint64_t mask) {
    if constexpr (ALL) {
        asm("v_swap_b32 %0, %1\n\tv_swap_b32 %2, %3" : "+v"(x0), "+v"(y0), "+v"(x1), "+v"(y1));
    } else {
        uint64_t saved;
        asm("s_mov_b64 %4, exec\n\ts_and_b64 exec, exec, %5\n\tv_swap_b32 %0, %1\n\tv_swap_b32 %2, %3\n\t"
            "s_mov_b64 exec, %4"
            : "+v"(x0), "+v"(y0), "+v"(x1), "+v"(y1), "=&s"(saved)
            : "s"(mask)
            : "scc");
    }
}
template <bool ALL> __device__ __forceinline__ void swap_ip(double &x, double &y, uint64_t mask) {
    const uint64_t ux = __double_as_longlong(x), uy = __double_as_longlong(y);
    uint32_t x0 = static_cast<uint32_t>(ux), x1 = static_cast<uint32_t>(ux >> 32);
    uint32_t y0 = static_cast<uint32_t>(uy), y1 = static_cast<uint32_t>(uy >> 32);
    swap_words<ALL>(x0, y0, x1, y1, mask);
    x = __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(x1) << 32) | x0));
    y = __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(y1) << 32) | y0));
}
template <bool ALL, typename T> __device__ __forceinline__ void swapc(Cx<T> &x, Cx<T> &y, uint64_t mask) {
    if constexpr (sizeof(T) == 8) {
        swap_ip<ALL>(x.r, y.r, mask);
        swap_ip<ALL>(x.i, y.i, mask);
    } else {
        uint32_t x0 = __float_as_uint(x.r), x1 = __float_as_uint(x.i);
        uint32_t y0 = __float_as_uint(y.r), y1 = __float_as_uint(y.i);
        swap_words<ALL>(x0, y0, x1, y1, mask);
        x = {__uint_as_float(x0), __uint_as_float(x1)};
        y = {__uint_as_float(y0), __uint_as_float(y1)};
    }
}

template <typename T, int NS, int A, int Q, typename M>
__device__ __forceinline__ void each_pair(Cx<T> (&v)[NS][A], M &&m) {
#pragma unroll
    for (int s = 0; s < NS; s++) {
#pragma unroll
        for (int k = 0; k < A; k++) {
            if (!(k & (1 << Q))) {
                m(v[s][k], v[s][k | (1 << Q)]);
            }
        }
    }
}

// U on register bit Q; u in scalar registers (UNI) or one block per lane.
// U_SWAP exchanges on the lanes of `mask`.
template <typename T, int NS, int A, int Q, bool UNI>
__device__ __forceinline__ void apply1(Cx<T> (&v)[NS][A], int ukind, const T (&u)[8], uint64_t mask) {
    if (ukind == U_DENSE) {
        each_pair<T, NS, A, Q>(v, [&](Cx<T> &a, Cx<T> &b) {
            T tr = u[2] * b.r, ti = u[2] * b.i, qr = u[4] * a.r, qi = u[4] * a.i;
            tr = fma(-u[3], b.i, tr);
            ti = fma(u[3], b.r, ti);
            qr = fma(-u[5], a.i, qr);
            qi = fma(u[5], a.r, qi);
            tr = fma(-u[1], a.i, tr);
            ti = fma(u[1], a.r, ti);
            qr = fma(-u[7], b.i, qr);
            qi = fma(u[7], b.r, qi);
            fma_ip<UNI>(a.r, u[0], tr);
            fma_ip<UNI>(a.i, u[0], ti);
            fma_ip<UNI>(b.r, u[6], qr);
            fma_ip<UNI>(b.i, u[6], qi);
        });
    } else if (ukind == U_REAL) {
        each_pair<T, NS, A, Q>(v, [&](Cx<T> &a, Cx<T> &b) {
            const T tr = u[1] * b.r, ti = u[1] * b.i, qr = u[2] * a.r, qi = u[2] * a.i;
            fma_ip<UNI>(a.r, u[0], tr);
            fma_ip<UNI>(a.i, u[0], ti);
            fma_ip<UNI>(b.r, u[3], qr);
            fma_ip<UNI>(b.i, u[3], qi);
        });
    } else if (ukind == U_DIAG) {
        each_pair<T, NS, A, Q>(v, [&](Cx<T> &a, Cx<T> &b) {
            scale_ip<UNI>(a, u[0], u[1]);
            scale_ip<UNI>(b, u[2], u[3]);
        });
    } else if (ukind == U_SWAP) {
        each_pair<T, NS, A, Q>(v, [&](Cx<T> &a, Cx<T> &b) { swapc<UNI>(a, b, mask); });
    }
}

template <typename T, int NS, int A, int QA, int QB, typename M>
__device__ __forceinline__ void each_quad(Cx<T> (&v)[NS][A], M &&m) {
    constexpr int MQ = (1 << QA) | (1 << QB);
#pragma unroll
    for (int s = 0; s < NS; s++) {
#pragma unroll
        for (int k = 0; k < A; k++) {
            if (!(k & MQ)) {
                m(v[s][k], v[s][k | (1 << QB)], v[s][k | (1 << QA)], v[s][k | MQ]);
            }
        }
    }
}

template <typename T, int NS, int A, int QA, int QB>
__device__ __forceinline__ void apply2(Cx<T> (&v)[NS][A], int ukind, int swp, const T (&u)[8], CT<T> *U) {
    using C = Cx<T>;
    if (ukind == U_DIAG) {
        each_quad<T, NS, A, QA, QB>(v, [&](C &a, C &b, C &c, C &d) {
            scale_ip<true>(a, u[0], u[1]);
            scale_ip<true>(b, u[2], u[3]);
            scale_ip<true>(c, u[4], u[5]);
            scale_ip<true>(d, u[6], u[7]);
        });
    } else if (ukind == U_SWAP) {
        if (swp == 11) { // 2 <-> 3: CNOT controlled by a
            each_quad<T, NS, A, QA, QB>(v, [&](C &, C &, C &c, C &d) { swapc<true>(c, d, 0); });
        } else if (swp == 7) { // 1 <-> 3: CNOT controlled by b
            each_quad<T, NS, A, QA, QB>(v, [&](C &, C &b, C &, C &d) { swapc<true>(b, d, 0); });
        } else if (swp == 6) { // 1 <-> 2: SWAP
            each_quad<T, NS, A, QA, QB>(v, [&](C &, C &b, C &c, C &) { swapc<true>(b, c, 0); });
        } else if (swp == 1) {
            each_quad<T, NS, A, QA, QB>(v, [&](C &a, C &b, C &, C &) { swapc<true>(a, b, 0); });
        } else if (swp == 2) {
            each_quad<T, NS, A, QA, QB>(v, [&](C &a, C &, C &c, C &) { swapc<true>(a, c, 0); });
        } else {
            each_quad<T, NS, A, QA, QB>(v, [&](C &a, C &, C &, C &d) { swapc<true>(a, d, 0); });
        }
    } else if (ukind == U_REAL) {
        each_quad<T, NS, A, QA, QB>(v, [&](C &a, C &b, C &c, C &d) {
            C *x[4] = {&a, &b, &c, &d};
            C t[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int e0 = (r + 1) & 3;
                t[r] = {U[4 * r + e0] * x[e0]->r, U[4 * r + e0] * x[e0]->i};
#pragma unroll
                for (int q = 2; q < 4; q++) {
                    const int e = (r + q) & 3;
                    t[r].r = fma(U[4 * r + e], x[e]->r, t[r].r);
                    t[r].i = fma(U[4 * r + e], x[e]->i, t[r].i);
                }
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                fma_ip<true>(x[r]->r, U[5 * r], t[r].r);
                fma_ip<true>(x[r]->i, U[5 * r], t[r].i);
            }
        });
    } else {
        each_quad<T, NS, A, QA, QB>(v, [&](C &a, C &b, C &c, C &d) {
            C *x[4] = {&a, &b, &c, &d};
            C t[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int e0 = (r + 1) & 3;
                t[r] = cmul(C{U[2 * (4 * r + e0)], U[2 * (4 * r + e0) + 1]}, *x[e0]);
#pragma unroll
                for (int q = 2; q < 4; q++) {
                    const int e = (r + q) & 3;
                    t[r] = cmad(C{U[2 * (4 * r + e)], U[2 * (4 * r + e) + 1]}, *x[e], t[r]);
                }
                t[r].r = fma(-U[10 * r + 1], x[r]->i, t[r].r);
                t[r].i = fma(U[10 * r + 1], x[r]->r, t[r].i);
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                fma_ip<true>(x[r]->r, U[10 * r], t[r].r);
                fma_ip<true>(x[r]->i, U[10 * r], t[r].i);
            }
        });
    }
}

// out = the block of NV reals at base that the lane's (or tile's) bit picks.
template <typename T, int NV>
__device__ __forceinline__ void pick(T (&out)[NV], CT<T> *base, bool c) {
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const T x0 = base[i], x1 = base[NV + i];
        out[i] = c ? x1 : x0;
    }
}

// ---------------------------------------------------------------------------
// One instruction.
// ---------------------------------------------------------------------------
template <typename T, int NS, int R>
__device__ __forceinline__ void step(Cx<T> (&v)[NS][1 << R], Ins<T> &in, CT<unsigned char> *prog,
                                     double *lacc, int dummy, int lane, uint64_t tbase) {
    constexpr int A = 1 << R;
    const int nremap = static_cast<int8_t>(in.w[5]);
    if (nremap > 0) {
        remap<T, NS, R>(v, static_cast<int8_t>(in.w[5] >> 8), static_cast<int8_t>(in.w[5] >> 16), lane);
        if (nremap > 1) {
            remap<T, NS, R>(v, static_cast<int8_t>(in.w[5] >> 24), static_cast<int8_t>(in.w[6]), lane);
        }
    }
    int code = static_cast<int8_t>(in.w[0]);
    const int a = static_cast<int8_t>(in.w[0] >> 8);
    const int b = static_cast<int8_t>(in.w[0] >> 16);
    const int s0 = static_cast<int8_t>(in.w[0] >> 24);
    const int s1 = static_cast<int8_t>(in.w[1]);
    int ukind = static_cast<int8_t>(in.w[1] >> 8);
    const int gkind = static_cast<int8_t>(in.w[1] >> 16);
    const int swp = static_cast<int8_t>(in.w[1] >> 24);
    const int slot = in.w[2];
    CT<T> *U = reinterpret_cast<CT<T> *>(prog + in.w[3]);
    CT<T> *G = reinterpret_cast<CT<T> *>(prog + in.w[4]);
    if (code == RT_SEL && s0 >= 64) {
        // The selecting bit is fixed for the tile: one block for all lanes.
        const bool c = (tbase >> (s0 - 64)) & 1;
        if (ukind == U_SWAP) {
            ukind = (c ? in.u[1] : in.u[0]) != T(0) ? U_SWAP : U_NONE;
        } else if (ukind == U_DENSE) {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                in.u[e] = U[(c ? 8 : 0) + e];
            }
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                in.u[e] = c ? in.u[4 + e] : in.u[e];
            }
        }
        if (c) {
            G += gkind == G_DIAG ? 2 : 8;
        }
        code = RT_REG1;
    }
    if (code == RT_REG1) {
        dispatch_q<R>(a, [&](auto Qc) {
            constexpr int Q = decltype(Qc)::value;
            if constexpr (NS > 1) {
                if (slot >= 0) {
                    if (gkind == G_XYZ) {
                        acc_pauli<T, NS, A, Q, 7>(v, lacc, slot, dummy, lane);
                    } else if (gkind == G_X) {
                        acc_pauli<T, NS, A, Q, 1>(v, lacc, slot, dummy, lane);
                    } else if (gkind == G_Y) {
                        acc_pauli<T, NS, A, Q, 2>(v, lacc, slot, dummy, lane);
                    } else if (gkind == G_Z) {
                        acc_pauli<T, NS, A, Q, 4>(v, lacc, slot, dummy, lane);
                    } else if (gkind == G_DIAG) {
                        const T g[2] = {G[0], G[1]};
                        acc_gen1<T, NS, A, Q, true>(v, g, lacc, slot, dummy, lane);
                    } else {
                        const T g[8] = {G[0], G[1], G[2], G[3], G[4], G[5], G[6], G[7]};
                        acc_gen1<T, NS, A, Q, false>(v, g, lacc, slot, dummy, lane);
                    }
                }
            }
            apply1<T, NS, A, Q, true>(v, ukind, in.u, 0);
        });
    } else if (code == RT_REG2) {
        dispatch_q2<R>(a, b, [&](auto QAc, auto QBc) {
            constexpr int QA = decltype(QAc)::value, QB = decltype(QBc)::value;
            if constexpr (NS > 1) {
                if (slot >= 0) {
                    if (gkind == G_Z) {
                        acc_gen2<T, NS, A, QA, QB, G_Z>(v, G, lacc, slot, dummy, lane);
                    } else if (gkind == G_DIAG) {
                        acc_gen2<T, NS, A, QA, QB, G_DIAG>(v, G, lacc, slot, dummy, lane);
                    } else {
                        acc_gen2<T, NS, A, QA, QB, G_DENSE>(v, G, lacc, slot, dummy, lane);
                    }
                }
            }
            apply2<T, NS, A, QA, QB>(v, ukind, swp, in.u, U);
        });
    } else if (code == RT_SEL) {
        const bool c0 = lbit(lane, s0);
        dispatch_q<R>(a, [&](auto Qc) {
            constexpr int Q = decltype(Qc)::value;
            if constexpr (NS > 1) {
                if (slot >= 0) {
                    if (gkind == G_DIAG) {
                        T g[2];
                        pick<T, 2>(g, G, c0);
                        acc_gen1<T, NS, A, Q, true>(v, g, lacc, slot, dummy, lane);
                    } else {
                        T g[8];
                        pick<T, 8>(g, G, c0);
                        acc_gen1<T, NS, A, Q, false>(v, g, lacc, slot, dummy, lane);
                    }
                }
            }
            T u[8] = {};
            uint64_t mask = 0;
            if (ukind == U_SWAP) {
                mask = __ballot((c0 ? in.u[1] : in.u[0]) != T(0));
            } else if (ukind == U_DENSE) {
                pick<T, 8>(u, U, c0);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    u[e] = c0 ? in.u[4 + e] : in.u[e];
                }
            }
            apply1<T, NS, A, Q, false>(v, ukind, u, mask);
        });
    } else if (code == RT_LANE) {
        // G phi = g phi on this lane, so the products scale by g.
        const bool c0 = selbit(lane, tbase, s0);
        const bool c1 = s1 >= 0 ? selbit(lane, tbase, s1) : false;
        if constexpr (NS > 1) {
            if (slot >= 0) {
                T g = c0 ? G[1] : G[0];
                if (s1 >= 0) {
                    const T g1 = c0 ? G[3] : G[2];
                    g = c1 ? g1 : g;
                }
                constexpr int NJ = NS - 1;
                double d[NJ];
#pragma unroll
                for (int j = 0; j < NJ; j++) {
                    double x = 0.0;
#pragma unroll
                    for (int k = 0; k < A; k++) {
                        x = im_add(x, wide(v[j + 1][k]), wide(v[0][k]));
                    }
                    d[j] = x * static_cast<double>(g);
                }
                add_slots<NJ>(d, lacc, slot * NJ, dummy, lane);
            }
        }
        Cx<T> f{c0 ? in.u[2] : in.u[0], c0 ? in.u[3] : in.u[1]};
        if (s1 >= 0) {
            const Cx<T> f1{c0 ? in.u[6] : in.u[4], c0 ? in.u[7] : in.u[5]};
            f = {c1 ? f1.r : f.r, c1 ? f1.i : f.i};
        }
#pragma unroll
        for (int s = 0; s < NS; s++) {
#pragma unroll
            for (int k = 0; k < A; k++) {
                scale_ip<false>(v[s][k], f.r, f.i);
            }
        }
    }
}

// Byte offset of register slot k: the sum over its set bits q of 2^reg[q].
template <typename T, int R> __device__ __forceinline__ uint64_t slot_off(const int *reg, int k) {
    uint64_t o = 0;
#pragma unroll
    for (int q = 0; q < R; q++) {
        if ((k >> q) & 1) {
            o += uint64_t{sizeof(Cx<T>)} << reg[q];
        }
    }
    return o;
}

// A table entry through the scalar cache (tables are written before the launch).
template <typename S> __device__ __forceinline__ S load_uniform(const S *p) {
    static_assert(sizeof(S) % 4 == 0, "whole words");
    CT<uint32_t> *w = (CT<uint32_t> *)(p);
    uint32_t buf[sizeof(S) / 4];
#pragma unroll
    for (size_t k = 0; k < sizeof(S) / 4; k++) {
        buf[k] = w[k];
    }
    S out;
    __builtin_memcpy(&out, buf, sizeof(S));
    return out;
}

// Loads and stores of a state whose pointer comes from a table: a generic
// pointer would make them flat instructions, which also count as LDS
// operations, so that every operation on the tile would wait for the fetch of
// the next instruction.
template <typename T> __device__ __forceinline__ Cx<T> ldg(const Cx<T> *p, uint32_t i) {
    typedef T V __attribute__((ext_vector_type(2)));
    const V v = ((const __attribute__((address_space(1))) V *)(p))[i];
    return {v.x, v.y};
}
template <typename T> __device__ __forceinline__ void stg(Cx<T> *p, uint32_t i, const Cx<T> &c) {
    typedef T V __attribute__((ext_vector_type(2)));
    ((__attribute__((address_space(1))) V *)(p))[i] = V{c.r, c.i};
}

// (H phi)_i of a sum of Pauli words at U indices i0 + u * step: U gathers in
// flight a word, the next word read ahead. One index at a time took 166 ns a word
// and index (12 qubits complex128).
template <typename T, int U>
__device__ __forceinline__ void pauli_sum(const SweepTerm *terms, int count, const Cx<T> *phi, uint32_t i0,
                                          uint32_t step, double (&sr)[U], double (&si)[U]) {
#pragma unroll
    for (int u = 0; u < U; u++) {
        sr[u] = 0.0;
        si[u] = 0.0;
    }
    if (count <= 0) {
        return;
    }
    SweepTerm next = load_uniform(terms);
#pragma unroll 1
    for (int k = 0; k < count; k++) {
        const SweepTerm t = next;
        next = load_uniform(terms + (k + 1 < count ? k + 1 : k));
        Cx<T> p[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            p[u] = ldg(phi, (i0 + static_cast<uint32_t>(u) * step) ^ t.x);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const double sg = (__popc((i0 + static_cast<uint32_t>(u) * step) & t.zy) & 1) ? -1.0 : 1.0;
            const double cr = sg * t.cr, ci = sg * t.ci;
            const double pr = static_cast<double>(p[u].r), pi = static_cast<double>(p[u].i);
            sr[u] += cr * pr - ci * pi;
            si[u] += cr * pi + ci * pr;
        }
    }
}

// h = H phi at the indices i0 + u * step (u < U); returns their part of
// <phi|H|phi>.
template <typename T, int U>
__device__ __forceinline__ double pauli_apply(const SweepTerm *terms, int count, const Cx<T> *phi, Cx<T> *h,
                                              uint32_t i0, uint32_t step) {
    double sr[U], si[U], e = 0.0;
    pauli_sum<T, U>(terms, count, phi, i0, step, sr, si);
#pragma unroll
    for (int u = 0; u < U; u++) {
        const uint32_t i = i0 + static_cast<uint32_t>(u) * step;
        const Cx<T> a = ldg(phi, i);
        e += static_cast<double>(a.r) * sr[u] + static_cast<double>(a.i) * si[u];
        stg(h, i, Cx<T>{static_cast<T>(sr[u]), static_cast<T>(si[u])});
    }
    return e;
}

// h = H phi at every step-th index from i0 < len (both powers of two), up to
// eight at a time; returns their part of <phi|H|phi>.
template <typename T>
__device__ __forceinline__ double pauli_share(const SweepTerm *terms, int count, const Cx<T> *phi, Cx<T> *h,
                                              uint32_t i0, uint32_t step, uint32_t len) {
    double e = 0.0;
    if (len >= 8 * step) {
        for (uint32_t i = i0; i < len; i += 8 * step) {
            e += pauli_apply<T, 8>(terms, count, phi, h, i, step);
        }
    } else if (len >= 4 * step) {
        e = pauli_apply<T, 4>(terms, count, phi, h, i0, step);
    } else if (len >= 2 * step) {
        e = pauli_apply<T, 2>(terms, count, phi, h, i0, step);
    } else if (i0 < len) {
        e = pauli_apply<T, 1>(terms, count, phi, h, i0, step);
    }
    return e;
}

// Runs a program on the tile: the next instruction is fetched while the
// current one runs.
template <typename T, int NS, int R>
__device__ __forceinline__ void run_program(Cx<T> (&v)[NS][1 << R], const Ins<T> &first, CT<unsigned char> *prog,
                                            int ninstr, double *lacc, int dummy, int lane, uint64_t tbase) {
    Ins<T> cur = first;
#pragma unroll 1
    for (int pc = 0; pc < ninstr; pc++) {
        const Ins<T> nxt = fetch<T>(prog, pc + 1);
        step<T, NS, R>(v, cur, prog, lacc, dummy, lane, tbase);
        cur = nxt;
    }
}

} // namespace plk
