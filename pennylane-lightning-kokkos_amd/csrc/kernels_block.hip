// Dense 5-qubit blocks on the matrix cores: v_mfma_f32_16x16x4f32 for
// complex64 states, v_mfma_f64_16x16x4f64 for complex128 states.
//
// A block is a 32x32 complex matrix M acting on five state bits b0 < ... < b4
// (local index s = sum_t bit(b_t) << t). Written over the reals, w = M v is
// a 64x64 real product [wr; wi] = [[Mr, -Mi], [Mi, Mr]] [vr; vi], and over
// all 2^(n-5) groups of amplitudes that share the other bits it is one GEMM
// of a fixed 64x64 matrix with a 64 x 2^(n-5) matrix of gathered amplitudes.
// Each wave takes 16 groups at a time and runs it as 64
// v_mfma_f32_16x16x4f32 (4 output row blocks x 16 steps of K = 4).
//
// The rows of both operands are permuted so that no data is exchanged
// between lanes: lane l = 16 kq + j (j = group of the tile, kq = l / 16)
// loads the eight amplitudes s = 8 kq + t, t = 0..7, of its group. The MFMA
// B operand of lane l at step ks is row 4 ks + kq of column j, so row
// 4 ks + kq is defined to be Re v[8 kq + ks] (ks < 8) or Im v[8 kq + ks - 8]
// (ks >= 8): every lane feeds the values it loaded. The output block rb of
// the 16x16x4 instruction puts row 4 kq + r of column j in register r of lane
// 16 kq + j, so output row 16 rb + 4 kq + r is defined to be
// Re w[8 kq + 4 rb + r] (rb < 2) or Im w[8 kq + 4 (rb - 2) + r] (rb >= 2):
// every lane ends up holding the eight amplitudes it loaded, and stores them
// in place. The host applies both permutations to the 64x64 real matrix and
// lays it out per lane (64 floats a lane, resident in registers).
//
// Bytes per launch: 2 S (each amplitude read and written once); flops:
// 8 * 32 per amplitude (a complex multiply-add is 8 real flops), so 16 flop
// per byte of complex64 state (8 per byte of complex128 state).
// The FP64 instruction has the same A / B layouts and puts output row
// 4 r + kq (rather than 4 kq + r) in register r of lane 16 kq + j; only the
// host's output-row permutation differs.
#include <set>

#include "plk_internal.hpp"

namespace plk {

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef double d2 __attribute__((ext_vector_type(2)));

constexpr int kBlockWaves = 4;

struct BlockArgs {
    uint64_t groups;      // 2^(n-5)
    int bits[5];          // ascending block bits
    int pad;
    uint64_t off_t[8];    // offset of local states t = 0..7 (bits b0, b1, b2)
    uint64_t off_kq[4];   // offset of local states 8 kq (bits b3, b4)
};

template <typename T> struct BlockTypes;
template <> struct BlockTypes<float> {
    using C2 = float2;
    using V2 = f2;
    using Unit = f4;
    using Acc = f4;
    static __device__ __forceinline__ Acc mfma(float a, float b, Acc c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
};
template <> struct BlockTypes<double> {
    using C2 = double2;
    using V2 = d2;
    using Unit = d2;
    using Acc = d4;
    static __device__ __forceinline__ Acc mfma(double a, double b, Acc c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
};

__device__ __forceinline__ uint64_t insert_zero_bit(uint64_t x, int b) {
    const uint64_t lo = x & ((uint64_t{1} << b) - 1);
    return ((x >> b) << (b + 1)) | lo;
}

__device__ __forceinline__ uint64_t group_base(const BlockArgs &a, uint64_t g) {
#pragma unroll
    for (int q = 0; q < 5; q++) {
        g = insert_zero_bit(g, a.bits[q]);
    }
    return g;
}

// One wave: tiles of 16 groups, round-robin over the waves of the grid; the
// next tile's amplitudes are loaded while the current tile's products run.
template <typename T>
__global__ void __launch_bounds__(64 * kBlockWaves)
    block5_kernel(typename BlockTypes<T>::C2 *__restrict__ psi, const T *__restrict__ apack,
                  BlockArgs a) {
    using BT = BlockTypes<T>;
    using C2 = typename BT::C2;
    const int l = threadIdx.x & 63;
    const int j = l & 15;
    const int kq = l >> 4;
    // The lane's 64 matrix values: apack[(rb * 16 + ks) * 64 + l].
    T A[64];
#pragma unroll
    for (int e = 0; e < 64; e++) {
        A[e] = apack[e * 64 + l];
    }
    const uint64_t lane_off = a.off_kq[kq];
    const uint64_t tiles = a.groups >> 4;
    const uint64_t wave = uint64_t{blockIdx.x} * kBlockWaves + (threadIdx.x >> 6);
    const uint64_t nwaves = uint64_t{gridDim.x} * kBlockWaves;
    uint64_t tile = wave;
    if (tile >= tiles) {
        return;
    }
    uint64_t base = group_base(a, tile * 16 + static_cast<uint64_t>(j)) + lane_off;
    C2 v[8];
#pragma unroll
    for (int t = 0; t < 8; t++) {
        v[t] = psi[base + a.off_t[t]];
    }
    while (true) {
        const uint64_t next = tile + nwaves;
        const bool more = next < tiles;
        const uint64_t nbase =
            more ? group_base(a, next * 16 + static_cast<uint64_t>(j)) + lane_off : base;
        C2 nv[8];
        if (more) {
#pragma unroll
            for (int t = 0; t < 8; t++) {
                nv[t] = psi[nbase + a.off_t[t]];
            }
        }
        typename BT::Acc c[4];
#pragma unroll
        for (int rb = 0; rb < 4; rb++) {
            c[rb] = typename BT::Acc{0, 0, 0, 0};
        }
#pragma unroll
        for (int ks = 0; ks < 16; ks++) {
            const T b = ks < 8 ? v[ks].x : v[ks - 8].y;
#pragma unroll
            for (int rb = 0; rb < 4; rb++) {
                c[rb] = BT::mfma(A[rb * 16 + ks], b, c[rb]);
            }
        }
#pragma unroll
        for (int t = 0; t < 8; t++) {
            // Register r of output block rb holds Re (rb < 2) or Im (rb >= 2)
            // of local 8 kq + 4 (rb % 2) + r.
            const int rb = t >> 2, r = t & 3;
            psi[base + a.off_t[t]] = C2{c[rb][r], c[rb + 2][r]};
        }
        if (!more) {
            break;
        }
        tile = next;
        base = nbase;
#pragma unroll
        for (int t = 0; t < 8; t++) {
            v[t] = nv[t];
        }
    }
}

// Two blocks in one pass. One block a pass is bound by HBM (27 qubits
// complex64: 400-480 us for 2 GiB, while its products take 224 us of the
// matrix cores), so the tile that holds both blocks' bits is staged in LDS and
// both products are taken there. The tile has the blocks' bits, at most ten,
// and the lowest other bits up to 128 KB: every run of global memory is then at
// least 128 bytes (with 64 KB and 64 bytes the pass took 840 us where it now
// takes 640). One workgroup a CU; the matrices stay in registers, and the next
// tile is loaded into registers during the first product. The order of the tile
// in LDS is linear over its index bits: the higher bits are folded into the
// lowest so that the lanes of each product's reads lie in different banks (found
// per pair on the host).
// Bound: the matrix cores, busy 437 us of the 640 us that a pass takes at 27
// qubits complex64 (two passes of one block: 800-960 us) and of the 690 us at 26
// qubits complex128 (930 us); the rest is filling and emptying the tile between
// barriers, and column tiles whose first products wait for the last ones' writes.
template <typename T> constexpr int kPairTile = sizeof(T) == 4 ? 14 : 13;     // tile bits: 128 KB
template <typename T> constexpr int kPairWaveBits = sizeof(T) == 4 ? 3 : 2;   // waves of a workgroup
template <typename T> constexpr int kPairUnitBits = sizeof(T) == 4 ? 1 : 0;   // amplitudes of a 16-byte unit

__host__ __device__ constexpr uint64_t pair_xcds(unsigned grid) {
    return grid % 8 == 0 ? 8 : 1;
}

struct PairArgs {
    uint64_t tiles;       // 2^(n - tile bits)
    uint64_t mask;        // the tile's state bits
    uint64_t step;        // a workgroup's step from tile to tile, spread over the other bits
    int tb[14];           // the tile's state bits, ascending
    uint32_t ld[14];      // LDS bytes of each tile bit (exclusive or)
    uint32_t lane[2][6];  // per product: of the lane's bits (four of the column, two of the block)
    uint32_t reg[2][3];   // of the block's other three bits
    uint32_t col[2][5];   // of the other columns: wave bits, then the wave's own
};

template <typename T>
__global__ void __launch_bounds__(64 << kPairWaveBits<T>, sizeof(T) == 4 ? 2 : 1)
    block_pair_kernel(typename BlockTypes<T>::Unit *__restrict__ psi, const T *__restrict__ apack, PairArgs a) {
    using BT = BlockTypes<T>;
    using C2 = typename BT::V2;
    using Unit = typename BT::Unit;
    constexpr int TB = kPairTile<T>, WB = kPairWaveBits<T>, UB = kPairUnitBits<T>;
    constexpr int RB = TB - UB - 6 - WB; // register bits of the load layout
    constexpr int IB = TB - 9 - WB;      // column bits a wave walks
    extern __shared__ __align__(16) unsigned char tile_lds[];
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
    T A[2][64];
#pragma unroll
    for (int e = 0; e < 64; e++) {
        A[0][e] = apack[e * 64 + l];
        A[1][e] = apack[4096 + e * 64 + l];
    }
    // Load layout, in 16-byte units: lane = the lowest tile bits, wave = the highest.
    uint32_t own = 0;
    uint64_t off = 0;
    uint32_t at[2] = {0, 0};
#pragma unroll
    for (int q = 0; q < 6; q++) {
        const bool on = (l >> q) & 1;
        own ^= on ? a.ld[UB + q] : 0u;
        off += on ? uint64_t{1} << a.tb[UB + q] : 0u;
        at[0] ^= on ? a.lane[0][q] : 0u;
        at[1] ^= on ? a.lane[1][q] : 0u;
    }
#pragma unroll
    for (int q = 0; q < WB; q++) {
        const bool on = (w >> q) & 1;
        own ^= on ? a.ld[UB + 6 + RB + q] : 0u;
        off += on ? uint64_t{1} << a.tb[UB + 6 + RB + q] : 0u;
        at[0] ^= on ? a.col[0][q] : 0u;
        at[1] ^= on ? a.col[1][q] : 0u;
    }
    // State offsets of the register bits; hidden from hoisting, which would hold
    // every slot's offset and LDS address in registers.
    uint64_t reg_off[RB];
#pragma unroll
    for (int q = 0; q < RB; q++) {
        reg_off[q] = (uint64_t{1} << a.tb[UB + 6 + q]) >> UB;
    }
    auto keep_here = [&]() {
        asm volatile("" : "+v"(own));
#pragma unroll
        for (int q = 0; q < RB; q++) {
            asm volatile("" : "+s"(reg_off[q]));
        }
    };
    auto slot_lds = [&](int r) {
        uint32_t v = own;
#pragma unroll
        for (int q = 0; q < RB; q++) {
            v ^= ((r >> q) & 1) ? a.ld[UB + 6 + q] : 0u;
        }
        return reinterpret_cast<Unit *>(tile_lds + v);
    };
    auto slot_off = [&](int r) {
        uint64_t v = 0;
#pragma unroll
        for (int q = 0; q < RB; q++) {
            v += ((r >> q) & 1) ? reg_off[q] : 0u;
        }
        return v;
    };
    // Consecutive workgroups run on different XCDs: each XCD takes a contiguous
    // range of tiles.
    const uint64_t xcds = pair_xcds(gridDim.x);
    const uint64_t step = gridDim.x / xcds;
    uint64_t base = (blockIdx.x % xcds) * (a.tiles / xcds) + blockIdx.x / xcds;
    uint64_t left = (a.tiles / xcds - blockIdx.x / xcds + step - 1) / step; // tiles of this workgroup
#pragma unroll 1
    for (int q = 0; q < TB; q++) {
        base = insert_zero_bit(base, a.tb[q]);
    }
    Unit nv[1 << RB];
    Unit *here = psi + ((base + off) >> UB);
#pragma unroll
    for (int r = 0; r < (1 << RB); r++) {
        nv[r] = here[slot_off(r)];
    }
    while (true) {
        // The slots a thread fills are those it read at the end of the last tile.
        keep_here();
#pragma unroll
        for (int r = 0; r < (1 << RB); r++) {
            *slot_lds(r) = nv[r];
        }
        __syncthreads();
        const bool more = --left != 0;
        Unit *there = here;
        if (more) {
            base = ((base | a.mask) + a.step) & ~a.mask;
            there = psi + ((base + off) >> UB);
        }
#pragma unroll
        for (int k = 0; k < 2; k++) {
            auto column = [&](int i) { // LDS bytes of the wave's column tile i
                uint32_t x = at[k];
#pragma unroll
                for (int q = 0; q < IB; q++) {
                    x ^= ((i >> q) & 1) ? a.col[k][WB + q] : 0u;
                }
                return x;
            };
            auto elem = [&](uint32_t x, int t) {
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    x ^= ((t >> q) & 1) ? a.reg[k][q] : 0u;
                }
                return reinterpret_cast<C2 *>(tile_lds + x);
            };
            uint32_t x = column(0);
            C2 v[8];
#pragma unroll
            for (int t = 0; t < 8; t++) {
                v[t] = *elem(x, t);
            }
#pragma unroll
            for (int half = 0; half < 2; half++) {
                // The next tile's loads, a half before each half of the first product's
                // column tiles: issued together they hold the waves up.
                if (k == 0 && more) {
#pragma unroll
                    for (int r = half << (RB - 1); r < (half + 1) << (RB - 1); r++) {
                        nv[r] = there[slot_off(r)];
                    }
                }
#pragma unroll 1
                for (int i = half << (IB - 1); i < (half + 1) << (IB - 1); i++) {
                    const uint32_t xn = column(i + 1 < (1 << IB) ? i + 1 : 0);
                    typename BT::Acc c[4];
#pragma unroll
                    for (int rb = 0; rb < 4; rb++) {
                        c[rb] = typename BT::Acc{0, 0, 0, 0};
                    }
#pragma unroll
                    for (int ks = 0; ks < 16; ks++) {
                        const T b = ks < 8 ? v[ks].x : v[ks - 8].y;
#pragma unroll
                        for (int rb = 0; rb < 4; rb++) {
                            c[rb] = BT::mfma(A[k][rb * 16 + ks], b, c[rb]);
                        }
                        if (ks >= 8) { // last use: the next column tile's value
                            __builtin_amdgcn_sched_barrier(0);
                            v[ks - 8] = *elem(xn, ks - 8);
                        }
                    }
                    asm volatile("" : "+v"(x)); // addresses anew, not kept in registers
#pragma unroll
                    for (int t = 0; t < 8; t++) {
                        *elem(x, t) = C2{c[t >> 2][t & 3], c[(t >> 2) + 2][t & 3]};
                    }
                    x = xn;
                }
            }
            __syncthreads();
        }
        keep_here();
#pragma unroll
        for (int r = 0; r < (1 << RB); r++) {
            here[slot_off(r)] = *slot_lds(r);
        }
        if (!more) {
            break;
        }
        here = there;
    }
}

// Rank over GF(2) of the `count` vectors' low `rows` bits.
int low_rank(const uint32_t *vec, int count, int rows) {
    std::vector<uint32_t> v(vec, vec + count);
    int rank = 0;
    for (int r = 0; r < rows; r++) {
        int p = rank;
        while (p < count && !((v[p] >> r) & 1)) {
            p++;
        }
        if (p == count) {
            continue;
        }
        std::swap(v[rank], v[p]);
        for (int q = 0; q < count; q++) {
            if (q != rank && ((v[q] >> r) & 1)) {
                v[q] ^= v[rank];
            }
        }
        rank++;
    }
    return rank;
}

template <typename T> PairArgs pair_args(int n, const int *bits0, const int *bits1) {
    constexpr int TB = kPairTile<T>, UB = kPairUnitBits<T>;
    PairArgs a{};
    a.tiles = uint64_t{1} << (n - TB);
    std::set<int> bits(bits0, bits0 + 5);
    bits.insert(bits1, bits1 + 5);
    for (int b = 0; static_cast<int>(bits.size()) < TB; b++) {
        bits.insert(b);
    }
    std::copy(bits.begin(), bits.end(), a.tb);
    for (int b : bits) {
        a.mask |= uint64_t{1} << b;
    }
    // Tile positions of each product: block bits, then columns, ascending.
    int block[2][5], cols[2][TB - 5];
    for (int k = 0; k < 2; k++) {
        const int *own = k == 0 ? bits0 : bits1;
        int nb = 0, nc = 0;
        for (int q = 0; q < TB; q++) {
            if (std::find(own, own + 5, a.tb[q]) != own + 5) {
                block[k][nb++] = q;
            } else {
                cols[k][nc++] = q;
            }
        }
    }
    // LDS order: the identity with the higher bits folded into the low four or
    // five, whole units together. The lanes of a group that the LDS serves together (32 of 8 bytes, 16 of
    // 16) have to differ in these: lane bits 0-3 are columns 0-3, 4-5 block bits 3-4.
    constexpr int lanes = sizeof(T) == 4 ? 5 : 4;
    uint32_t best[14];
    int best_rank = -1;
    uint32_t rng = 1;
    for (int tries = 0; tries < 256 && best_rank < 2 * lanes; tries++) {
        uint32_t c[14];
        for (int q = 0; q < TB; q++) {
            rng = rng * 1664525u + 1013904223u;
            c[q] = (uint32_t{1} << q) ^ (q >= lanes ? (rng >> 16) & ((1u << lanes) - (1u << UB)) : 0u);
        }
        int rank = 0;
        for (int k = 0; k < 2; k++) {
            const uint32_t lane[5] = {c[cols[k][0]], c[cols[k][1]], c[cols[k][2]], c[cols[k][3]], c[block[k][3]]};
            rank += low_rank(lane, lanes, lanes);
        }
        if (rank > best_rank) {
            best_rank = rank;
            std::copy(c, c + TB, best);
        }
    }
    constexpr uint32_t bytes = 2 * sizeof(T);
    for (int q = 0; q < TB; q++) {
        a.ld[q] = best[q] * bytes;
    }
    for (int k = 0; k < 2; k++) {
        for (int q = 0; q < 4; q++) {
            a.lane[k][q] = a.ld[cols[k][q]];
        }
        for (int q = 0; q < 2; q++) {
            a.lane[k][4 + q] = a.ld[block[k][3 + q]];
        }
        for (int q = 0; q < 3; q++) {
            a.reg[k][q] = a.ld[block[k][q]];
        }
        for (int q = 0; q < TB - 9; q++) {
            a.col[k][q] = a.ld[cols[k][4 + q]];
        }
    }
    return a;
}

template <typename T> void launch_pair_t(Device &dev, const State &s, const int *bits0, const int *bits1, const void *d) {
    PairArgs a = pair_args<T>(s.n, bits0, bits1);
    constexpr size_t lds = (size_t{2} * sizeof(T)) << kPairTile<T>;
    // One workgroup a CU (LDS); the number of tiles is a power of two and at least 8.
    const unsigned grid = static_cast<unsigned>(std::min(a.tiles, static_cast<uint64_t>(dev.num_cus)));
    uint64_t step = grid / pair_xcds(grid);
    for (int b = 0; b < s.n && step != 0; b++) {
        if (!((a.mask >> b) & 1)) {
            a.step |= (step & 1) << b;
            step >>= 1;
        }
    }
    PLK_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&block_pair_kernel<T>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
    hipLaunchKernelGGL((block_pair_kernel<T>), dim3(grid), dim3(64 << kPairWaveBits<T>), lds, dev.stream,
                       static_cast<typename BlockTypes<T>::Unit *>(s.d), static_cast<const T *>(d), a);
    PLK_HIP(hipGetLastError());
}

} // namespace

template <typename T>
void block5_lane_pack_t(const std::vector<cd> &M, std::vector<T> &out) {
    // Real 64x64 form R[i][k] with logical index x < 32: Re of local x,
    // x >= 32: Im of local x - 32.
    auto R = [&](int i, int k) -> double {
        const int ri = i >> 5, si = i & 31, rk = k >> 5, sk = k & 31;
        const cd m = M[static_cast<size_t>(si) * 32 + sk];
        if (ri == rk) {
            return m.real();
        }
        return ri == 1 ? m.imag() : -m.imag();
    };
    // Output row o of output block rb = o / 16 sits in register r of lane
    // 16 kq + j with (FP32) o % 16 = 4 kq + r or (FP64) o % 16 = 4 r + kq; it
    // is Re / Im of local 8 kq + 4 (rb % 2) + r. Input row k = 4 ks + kq is
    // Re / Im of local 8 kq + ks % 8.
    auto out_row = [](int o) {
        const int rb = o >> 4;
        const int kq = sizeof(T) == 4 ? (o >> 2) & 3 : o & 3;
        const int r = sizeof(T) == 4 ? o & 3 : (o >> 2) & 3;
        return rb < 2 ? 8 * kq + 4 * rb + r : 32 + 8 * kq + 4 * (rb - 2) + r;
    };
    auto in_row = [](int k) {
        const int ks = k >> 2, kq = k & 3;
        return ks < 8 ? 8 * kq + ks : 32 + 8 * kq + (ks - 8);
    };
    out.assign(64 * 64, T(0));
    for (int rb = 0; rb < 4; rb++) {
        for (int ks = 0; ks < 16; ks++) {
            for (int l = 0; l < 64; l++) {
                // A operand of lane l: row 16 rb + l % 16, column 4 ks + l / 16.
                const int o = 16 * rb + (l & 15);
                const int k = 4 * ks + (l >> 4);
                out[static_cast<size_t>((rb * 16 + ks) * 64 + l)] =
                    static_cast<T>(R(out_row(o), in_row(k)));
            }
        }
    }
}

int block5_lane_pack(const std::vector<cd> &M, std::vector<float> &out) {
    block5_lane_pack_t<float>(M, out);
    return 0;
}

int block5_lane_pack(const std::vector<cd> &M, std::vector<double> &out) {
    block5_lane_pack_t<double>(M, out);
    return 0;
}

namespace {

void check_block_bits(const State &s, const int *bits) {
    for (int q = 0; q < 5; q++) {
        if (bits[q] < 0 || bits[q] >= s.n || (q > 0 && bits[q] <= bits[q - 1])) {
            raise(PLK_ERR_INVALID, "block bits must be ascending and inside the state");
        }
    }
}

} // namespace

// Two blocks a pass from a tile per CU on. 22 qubits complex64 (23 blocks, call
// to return): 1092 us a block a pass, 881 us two; 20 qubits 674 and 793 us. 21
// qubits complex128: 960 and 902 us; 20 qubits 836 and 866 us.
bool block_pairs(const Device &dev, const State &s) {
    const int tile = s.dtype == PLK_C64 ? kPairTile<float> : kPairTile<double>;
    return s.n >= tile && (uint64_t{1} << (s.n - tile)) >= static_cast<uint64_t>(dev.num_cus);
}

void launch_block_pair(Device &dev, const State &s, const int *bits0, const int *bits1, const void *d_apack) {
    check_block_bits(s, bits0);
    check_block_bits(s, bits1);
    if (!block_pairs(dev, s)) {
        raise(PLK_ERR_UNSUPPORTED, "the state is too small for two blocks a pass");
    }
    ProfScope prof("apply_block5", 2.0 * static_cast<double>(s.bytes()), dev.stream);
    if (s.dtype == PLK_C64) {
        launch_pair_t<float>(dev, s, bits0, bits1, d_apack);
    } else {
        launch_pair_t<double>(dev, s, bits0, bits1, d_apack);
    }
}

void launch_block5(Device &dev, const State &s, const int *bits, const void *d_apack) {
    if (s.n < 9) {
        raise(PLK_ERR_UNSUPPORTED, "5-qubit MFMA blocks need at least 9 qubits");
    }
    check_block_bits(s, bits);
    BlockArgs a{};
    a.groups = uint64_t{1} << (s.n - 5);
    std::copy(bits, bits + 5, a.bits);
    for (int t = 0; t < 8; t++) {
        uint64_t o = 0;
        for (int q = 0; q < 3; q++) {
            if ((t >> q) & 1) {
                o |= uint64_t{1} << bits[q];
            }
        }
        a.off_t[t] = o;
    }
    for (int kq = 0; kq < 4; kq++) {
        uint64_t o = 0;
        for (int q = 0; q < 2; q++) {
            if ((kq >> q) & 1) {
                o |= uint64_t{1} << bits[3 + q];
            }
        }
        a.off_kq[kq] = o;
    }
    const uint64_t tiles = a.groups >> 4;
    const uint64_t want = (tiles + kBlockWaves - 1) / kBlockWaves;
    const unsigned grid = static_cast<unsigned>(
        std::max<uint64_t>(1, std::min<uint64_t>(want, static_cast<uint64_t>(dev.num_cus) * 8)));
    ProfScope prof("apply_block5", 2.0 * static_cast<double>(s.bytes()), dev.stream);
    if (s.dtype == PLK_C64) {
        hipLaunchKernelGGL(block5_kernel<float>, dim3(grid), dim3(64 * kBlockWaves), 0,
                           dev.stream, static_cast<float2 *>(s.d),
                           static_cast<const float *>(d_apack), a);
    } else {
        hipLaunchKernelGGL(block5_kernel<double>, dim3(grid), dim3(64 * kBlockWaves), 0,
                           dev.stream, static_cast<double2 *>(s.d),
                           static_cast<const double *>(d_apack), a);
    }
    PLK_HIP(hipGetLastError());
}

} // namespace plk
