// Probabilities and sampling (MeasuresKokkos.hpp:389-569,
// MeasuresFunctors.hpp:15-210), FP64 and deterministic.
//
// Marginal probabilities: output bin b collects |psi[i]|^2 over the indices i
// whose bits at the measured positions spell b (first measured wire = most
// significant bit of b). One block sums a contiguous range of the
// complementary index space for the bins that differ in the lowest measured
// bits only: those share cache lines, so a thread reads them together. The
// range is walked with the masked increment x' = ((x | ~mask) + step) & mask, so
// consecutive threads read consecutive amplitudes whenever the low bits are
// unmeasured. A second kernel adds the ranges of each bin, a wave per bin, in
// a fixed order. With few amplitudes per bin a thread owns a bin instead.
// Bound: HBM reads. 25 qubits complex128, call to return: one wire 414 us with a
// thread adding 4096 ranges of its bin, 120 us so; the lowest wire 536 us, 116
// us; the six lowest wires 306 us with a block per bin, 134 us.
//
// Sampling: probabilities of 64-amplitude runs and of 4096-amplitude chunks in
// one pass over the state, an exclusive scan of the chunks, then one wave per
// shot: a SplitMix64 uniform u in (0, 1] (Steele, Lea, Flood 2014; output k of
// the generator seeded with `seed`) and the bin with cdf[k] < u <= cdf[k+1] (the
// reference's binary search, MeasuresFunctors.hpp:74-110), found by a 64-way
// search of the chunk offsets, then of the chunk's runs, then of the run's
// amplitudes. No CDF of the whole register is written or read again.
// Bound: the HBM read of the state. 23 qubits complex128, 2000 shots, call to
// return: 314 us with a scanned CDF, 73 us so; 25 qubits 1189 us and 157 us.
#include "device_common.hpp"

namespace plk {

namespace {

constexpr int PB = 256;          // threads per block
constexpr int MARG_BLOCKS = 2048; // blocks a marginal aims for
constexpr int RUN = 64;           // amplitudes of a run: one per lane
constexpr int CHUNK = 64 * RUN;   // amplitudes of a chunk: a run per lane

struct BinMap {
    int m;        // measured wires
    int g[64];    // global bit of measured wire k (k = 0 most significant)
    int p[64];    // bin bit of measured wire k
};

__device__ __forceinline__ uint64_t bin_bits(const BinMap &bm, uint64_t b) {
    uint64_t v = 0;
    for (int k = 0; k < bm.m; k++) {
        v |= ((b >> (bm.m - 1 - k)) & 1ull) << bm.g[k];
    }
    return v;
}

// The bin bits of group b of the map's wires.
__device__ __forceinline__ uint64_t bin_base(const BinMap &bm, uint64_t b) {
    uint64_t v = 0;
    for (int k = 0; k < bm.m; k++) {
        v |= ((b >> (bm.m - 1 - k)) & 1ull) << bm.p[k];
    }
    return v;
}

__device__ __forceinline__ uint64_t pdep(uint64_t c, uint64_t mask) {
    uint64_t out = 0;
    while (mask) {
        const uint64_t low = mask & (~mask + 1ull);
        if (c & 1ull) {
            out |= low;
        }
        c >>= 1;
        mask &= mask - 1ull;
    }
    return out;
}

template <typename T> __device__ __forceinline__ double prob_of(const Cx<T> &a) {
    const double r = static_cast<double>(a.r), i = static_cast<double>(a.i);
    return r * r + i * i;
}

// One block per (group of 2^K bins, range of `per` complement indices); the
// bins of a group differ in the K lowest measured bits, at offsets off[].
template <int K> struct LowBins {
    uint64_t off[1 << K]; // index bits of the group's bins
    uint32_t bin[1 << K]; // their bin bits
};
template <typename T, int K>
__global__ void __launch_bounds__(PB)
    marg_block_kernel(const Cx<T> *__restrict__ psi, BinMap high, LowBins<K> low, uint64_t cmask, uint64_t step,
                      uint64_t per, uint64_t chunks, double *__restrict__ partial) {
    constexpr int NB = 1 << K;
    __shared__ double lds[NB][PB / 64];
    const uint64_t b = blockIdx.x / chunks;
    const uint64_t chunk = blockIdx.x % chunks;
    const uint64_t base = bin_bits(high, b);
    uint64_t x = pdep(chunk * per + threadIdx.x, cmask);
    double acc[NB];
#pragma unroll
    for (int i = 0; i < NB; i++) {
        acc[i] = 0.0;
    }
    constexpr int U = K >= 3 ? 1 : 4 >> K; // loads in flight per thread
    for (uint64_t r = threadIdx.x; r < per; r += uint64_t{U} * PB) {
        Cx<T> a[U][NB];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const bool on = r + static_cast<uint64_t>(u) * PB < per;
#pragma unroll
            for (int i = 0; i < NB; i++) {
                a[u][i] = on ? psi[base | x | low.off[i]] : Cx<T>{T(0), T(0)};
            }
            x = ((x | ~cmask) + step) & cmask;
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
#pragma unroll
            for (int i = 0; i < NB; i++) {
                acc[i] += prob_of(a[u][i]);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < NB; i++) {
        const double v = wave_sum(acc[i]);
        if ((threadIdx.x & 63) == 0) {
            lds[i][threadIdx.x >> 6] = v;
        }
    }
    __syncthreads();
    const int i = static_cast<int>(threadIdx.x);
    if (i < NB) {
        partial[(bin_base(high, b) | low.bin[i]) * chunks + chunk] = lds[i][0] + lds[i][1] + lds[i][2] + lds[i][3];
    }
}

// One wave per bin.
__global__ void __launch_bounds__(PB)
    marg_finish_kernel(const double *__restrict__ partial, uint64_t bins, uint64_t chunks,
                       double *__restrict__ out) {
    const uint64_t b = uint64_t{blockIdx.x} * (PB / 64) + (threadIdx.x >> 6);
    if (b >= bins) {
        return;
    }
    double s = 0.0;
#pragma unroll 8
    for (uint64_t c = threadIdx.x & 63; c < chunks; c += 64) {
        s += partial[b * chunks + c];
    }
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) {
        out[b] = s;
    }
}

// One thread per bin (few amplitudes per bin).
template <typename T>
__global__ void __launch_bounds__(PB)
    marg_thread_kernel(const Cx<T> *__restrict__ psi, BinMap bm, uint64_t cmask, uint64_t count,
                       uint64_t bins, double *__restrict__ out) {
    const uint64_t b = uint64_t{blockIdx.x} * PB + threadIdx.x;
    if (b >= bins) {
        return;
    }
    const uint64_t base = bin_bits(bm, b);
    uint64_t x = 0;
    double s = 0.0;
    for (uint64_t c = 0; c < count; c++) {
        s += prob_of(psi[base | x]);
        x = ((x | ~cmask) + 1ull) & cmask;
    }
    out[b] = s;
}

// Probability of every run and chunk: a block per chunk, a wave per 16 runs.
template <typename T>
__global__ void __launch_bounds__(PB)
    run_totals_kernel(const Cx<T> *__restrict__ psi, uint64_t len, double *__restrict__ runs,
                      double *__restrict__ chunks) {
    constexpr int PER = CHUNK / PB; // runs of a wave
    __shared__ double lds[64];
    const int lane = static_cast<int>(threadIdx.x) & 63, wave = static_cast<int>(threadIdx.x) >> 6;
    const uint64_t first = uint64_t{blockIdx.x} * CHUNK + static_cast<uint64_t>(wave * PER * RUN + lane);
    Cx<T> a[PER];
#pragma unroll
    for (int r = 0; r < PER; r++) {
        const uint64_t i = first + static_cast<uint64_t>(r) * RUN;
        a[r] = i < len ? psi[i] : Cx<T>{T(0), T(0)};
    }
    double mine = 0.0; // lane r keeps run r
#pragma unroll
    for (int r = 0; r < PER; r++) {
        const double t = wave_sum(prob_of(a[r])); // DPP; halving exchanges through LDS take longer
        mine = lane == r ? t : mine;
    }
    if (lane < PER) {
        lds[wave * PER + lane] = mine;
    }
    __syncthreads();
    if (threadIdx.x < 64) {
        const double t = lds[threadIdx.x];
        runs[uint64_t{blockIdx.x} * 64 + threadIdx.x] = t;
        const double s = wave_sum(t);
        if (threadIdx.x == 0) {
            chunks[blockIdx.x] = s;
        }
    }
}

// Inclusive prefix sum over the wave.
__device__ __forceinline__ double wave_scan(double v, int lane) {
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const double o = __shfl_up(v, off, 64);
        v = lane >= off ? v + o : v;
    }
    return v;
}

// In-place exclusive scan of the chunk totals by one block, SCAN at a time.
constexpr int SCAN = 1024;
__global__ void __launch_bounds__(SCAN) scan_top_kernel(double *__restrict__ totals, uint64_t nb) {
    __shared__ double part[SCAN / 64];
    const int lane = static_cast<int>(threadIdx.x) & 63, wave = static_cast<int>(threadIdx.x) >> 6;
    double carry = 0.0;
    for (uint64_t at = 0; at < nb; at += SCAN) {
        const uint64_t i = at + threadIdx.x;
        const double v = i < nb ? totals[i] : 0.0;
        const double inc = wave_scan(v, lane);
        if (lane == 63) {
            part[wave] = inc;
        }
        __syncthreads();
        double before = carry, all = carry;
        for (int w = 0; w < SCAN / 64; w++) {
            before += w < wave ? part[w] : 0.0;
            all += part[w];
        }
        const double exc = __shfl_up(inc, 1, 64);
        if (i < nb) {
            totals[i] = before + (lane == 0 ? 0.0 : exc);
        }
        carry = all;
        __syncthreads();
    }
}

__device__ __forceinline__ uint64_t splitmix64(uint64_t z) {
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// The last lane whose value lies below u (lane 0's always does).
__device__ __forceinline__ int last_below(double v, double u) {
    const uint64_t m = __ballot(v < u);
    return m == 0 ? 0 : 63 - __clzll(static_cast<long long>(m));
}

// One wave per shot: the last k with cdf[k] < u; bits of the bin written most
// significant (wire 0) first.
template <typename T>
__global__ void __launch_bounds__(PB)
    sample_kernel(const Cx<T> *__restrict__ psi, uint64_t len, const double *__restrict__ runs,
                  const double *__restrict__ chunks, uint64_t nb, int n, uint64_t shots, uint64_t seed,
                  uint64_t *__restrict__ out) {
    const uint64_t s = uint64_t{blockIdx.x} * (PB / 64) + (threadIdx.x >> 6);
    if (s >= shots) {
        return;
    }
    const int lane = static_cast<int>(threadIdx.x) & 63;
    const uint64_t z = splitmix64(seed + (s + 1) * 0x9E3779B97F4A7C15ull);
    const double u = static_cast<double>((z >> 11) + 1) * 0x1.0p-53;
    // Chunk: the last whose offset lies below u, 64 candidates at a time.
    uint64_t lo = 0, count = nb;
    while (count > 1) {
        const uint64_t step = (count + 63) / 64;
        const uint64_t at = static_cast<uint64_t>(lane) * step;
        const double v = at < count ? chunks[lo + at] : 2.0;
        const uint64_t k = static_cast<uint64_t>(last_below(v, u)) * step;
        lo += k;
        count = count - k < step ? count - k : step;
    }
    double below = chunks[lo];
    // Run of the chunk, then amplitude of the run.
    double t = runs[lo * 64 + static_cast<uint64_t>(lane)];
    double exc = __shfl_up(wave_scan(t, lane), 1, 64);
    exc = lane == 0 ? below : below + exc;
    const uint64_t first_run = lo * CHUNK + static_cast<uint64_t>(lane) * RUN;
    const int run = last_below(first_run < len ? exc : 2.0, u);
    below = __shfl(exc, run, 64);
    const uint64_t i = lo * CHUNK + static_cast<uint64_t>(run * RUN + lane);
    t = i < len ? prob_of(psi[i]) : 0.0;
    exc = __shfl_up(wave_scan(t, lane), 1, 64);
    exc = lane == 0 ? below : below + exc;
    const uint64_t index = lo * CHUNK + static_cast<uint64_t>(run * RUN + last_below(i < len ? exc : 2.0, u));
    for (int j = lane; j < n; j += 64) {
        out[s * static_cast<uint64_t>(n) + static_cast<uint64_t>(j)] = (index >> (n - 1 - j)) & 1ull;
    }
}

// The same for a state of one chunk and many shots, a thread a shot: every block
// forms the offsets of all amplitudes in LDS (as sample_kernel does for the run
// it needs, in the same order) and its threads search those. With 64 times as many
// threads as shots 300000 shots of 1 qubit took 286 us, of 6 qubits 1100, so 191
// and 990; 10000 shots of 10 qubits 73 and 70, of 12 qubits 81 and 85: used from
// four shots an amplitude on.
template <typename T>
__global__ void __launch_bounds__(PB)
    sample_chunk_kernel(const Cx<T> *__restrict__ psi, uint32_t len, const double *__restrict__ runs, int n,
                        uint64_t shots, uint64_t seed, uint64_t *__restrict__ out) {
    __shared__ double offset[CHUNK];
    __shared__ double run_offset[64];
    const int lane = static_cast<int>(threadIdx.x) & 63, wave = static_cast<int>(threadIdx.x) >> 6;
    const uint32_t nruns = (len + RUN - 1) / RUN;
    const double t = runs[lane];
    const double exc = __shfl_up(wave_scan(t, lane), 1, 64);
    const double mine = lane == 0 ? 0.0 : exc; // of run `lane`
    if (wave == 0) {
        run_offset[lane] = mine;
    }
    for (uint32_t r = static_cast<uint32_t>(wave); r < nruns; r += PB / 64) {
        const uint32_t i = r * RUN + static_cast<uint32_t>(lane);
        const double p = i < len ? prob_of(psi[i]) : 0.0;
        const double below = __shfl(mine, static_cast<int>(r), 64);
        const double e = __shfl_up(wave_scan(p, lane), 1, 64);
        offset[i] = lane == 0 ? below : below + e;
    }
    __syncthreads();
    // The last of `count` (a power of two) ascending offsets that lies below u, or the first.
    auto last = [](const double *v, uint32_t count, double u) {
        uint32_t at = 0;
        for (uint32_t step = count / 2; step > 0; step /= 2) {
            at += v[at + step] < u ? step : 0;
        }
        return at;
    };
    const uint32_t per = len < RUN ? len : RUN;
    for (uint64_t s = uint64_t{blockIdx.x} * PB + threadIdx.x; s < shots; s += uint64_t{gridDim.x} * PB) {
        const uint64_t z = splitmix64(seed + (s + 1) * 0x9E3779B97F4A7C15ull);
        const double u = static_cast<double>((z >> 11) + 1) * 0x1.0p-53;
        const uint32_t r = last(run_offset, nruns, u);
        const uint32_t index = r * RUN + last(offset + r * RUN, per, u);
        for (int j = 0; j < n; j++) {
            out[s * static_cast<uint64_t>(n) + static_cast<uint64_t>(j)] = (index >> (n - 1 - j)) & 1u;
        }
    }
}

template <typename T, int K>
void launch_marg(Device &dev, const Cx<T> *psi, const BinMap &bm, uint64_t cmask, uint64_t step, uint64_t per,
                 uint64_t chunks, double *partial) {
    BinMap high{};
    LowBins<K> low{};
    // The K measured wires on the lowest bits leave the map.
    std::vector<int> order;
    for (int k = 0; k < bm.m; k++) {
        order.push_back(k);
    }
    std::sort(order.begin(), order.end(), [&](int a, int b) { return bm.g[a] < bm.g[b]; });
    for (int i = 0; i < (1 << K); i++) {
        for (int q = 0; q < K; q++) {
            if ((i >> q) & 1) {
                low.off[i] |= uint64_t{1} << bm.g[order[q]];
                low.bin[i] |= uint32_t{1} << (bm.m - 1 - order[q]);
            }
        }
    }
    for (int k = 0; k < bm.m; k++) {
        if (std::find(order.begin(), order.begin() + K, k) == order.begin() + K) {
            high.g[high.m] = bm.g[k];
            high.p[high.m] = bm.m - 1 - k;
            high.m++;
        }
    }
    const uint64_t grid = (uint64_t{1} << high.m) * chunks;
    if (grid > (uint64_t{1} << 31)) {
        raise(PLK_ERR_UNSUPPORTED, "probability grid too large");
    }
    hipLaunchKernelGGL((marg_block_kernel<T, K>), dim3(static_cast<unsigned>(grid)), dim3(PB), 0, dev.stream, psi,
                       high, low, cmask, step, per, chunks, partial);
    PLK_HIP(hipGetLastError());
}

template <typename T>
void probs_t(Device &dev, const State &s, const std::vector<int> &gbits, double *host_out) {
    const int m = static_cast<int>(gbits.size());
    BinMap bm{};
    bm.m = m;
    uint64_t wmask = 0;
    for (int k = 0; k < m; k++) {
        bm.g[k] = gbits[k];
        wmask |= uint64_t{1} << gbits[k];
    }
    const uint64_t full = s.n >= 64 ? ~uint64_t{0} : (uint64_t{1} << s.n) - 1;
    const uint64_t cmask = full & ~wmask;
    const uint64_t bins = uint64_t{1} << m;
    const uint64_t count = uint64_t{1} << (s.n - m);
    const auto *psi = static_cast<const Cx<T> *>(s.d);
    ProfScope prof("probs", static_cast<double>(s.bytes()), dev.stream);
    if (count <= 64) {
        double *out = static_cast<double *>(ensure_work(dev, bins * sizeof(double)));
        const unsigned grid = static_cast<unsigned>((bins + PB - 1) / PB);
        hipLaunchKernelGGL((marg_thread_kernel<T>), dim3(grid), dim3(PB), 0, dev.stream, psi, bm,
                           cmask, count, bins, out);
        PLK_HIP(hipGetLastError());
        PLK_HIP(hipMemcpyAsync(host_out, out, bins * sizeof(double), hipMemcpyDeviceToHost,
                               dev.stream));
    } else {
        // Measured bits inside a 128-byte line: their bins are summed together.
        const int line = sizeof(T) == 8 ? 3 : 4;
        int K = 0;
        for (int k = 0; k < m; k++) {
            K += gbits[k] < line ? 1 : 0;
        }
        // A state of at most 4 MiB stays in the L2s, where bins apart cost nothing and
        // more blocks hide more latency (16 qubits complex128, the five lowest wires: 31
        // us together, 28 apart; 20 qubits complex64, the lowest wire: 29 and 39).
        K = s.bytes() <= (size_t{4} << 20) ? 0 : std::min(K, 3);
        // A power of two of ranges per bin: enough blocks to fill the device, of at
        // least 1024 amplitudes a bin, or a block a CU of at least one a thread.
        uint64_t chunks = 1;
        while ((bins >> K) * chunks < MARG_BLOCKS && count / (2 * chunks) >= 1024) {
            chunks *= 2;
        }
        while ((bins >> K) * chunks < static_cast<uint64_t>(dev.num_cus) && count / (2 * chunks) >= PB) {
            chunks *= 2;
        }
        const uint64_t per = count / chunks;
        double *partial = static_cast<double *>(
            ensure_work(dev, (bins * chunks + bins) * sizeof(double)));
        double *out = chunks == 1 ? partial : partial + bins * chunks;
        const uint64_t step = [&] {
            uint64_t v = 0, c = PB, mk = cmask;
            while (mk) {
                const uint64_t low = mk & (~mk + 1);
                if (c & 1) {
                    v |= low;
                }
                c >>= 1;
                mk &= mk - 1;
            }
            return v;
        }();
        switch (K) {
        case 0: launch_marg<T, 0>(dev, psi, bm, cmask, step, per, chunks, partial); break;
        case 1: launch_marg<T, 1>(dev, psi, bm, cmask, step, per, chunks, partial); break;
        case 2: launch_marg<T, 2>(dev, psi, bm, cmask, step, per, chunks, partial); break;
        default: launch_marg<T, 3>(dev, psi, bm, cmask, step, per, chunks, partial); break;
        }
        if (chunks > 1) {
            hipLaunchKernelGGL(marg_finish_kernel, dim3(static_cast<unsigned>((bins + PB / 64 - 1) / (PB / 64))),
                               dim3(PB), 0, dev.stream, partial, bins, chunks, out);
            PLK_HIP(hipGetLastError());
        }
        PLK_HIP(hipMemcpyAsync(host_out, out, bins * sizeof(double), hipMemcpyDeviceToHost,
                               dev.stream));
    }
    PLK_HIP(hipStreamSynchronize(dev.stream));
}

template <typename T>
void sample_t(Device &dev, const State &s, size_t shots, uint64_t seed, size_t *host_out) {
    const uint64_t len = s.len;
    const uint64_t nb = (len + CHUNK - 1) / CHUNK;
    const size_t run_bytes = nb * 64 * sizeof(double);
    const size_t tot_bytes = ((nb * sizeof(double)) + 255) & ~size_t{255};
    const size_t out_bytes = static_cast<size_t>(shots) * s.n * sizeof(uint64_t);
    unsigned char *w = static_cast<unsigned char *>(ensure_work(dev, run_bytes + tot_bytes + out_bytes));
    double *runs = reinterpret_cast<double *>(w);
    double *totals = reinterpret_cast<double *>(w + run_bytes);
    uint64_t *out = reinterpret_cast<uint64_t *>(w + run_bytes + tot_bytes);
    const auto *psi = static_cast<const Cx<T> *>(s.d);
    if (shots > 0) {
        ProfScope prof("sample", static_cast<double>(s.bytes()), dev.stream);
        hipLaunchKernelGGL((run_totals_kernel<T>), dim3(static_cast<unsigned>(nb)), dim3(PB), 0,
                           dev.stream, psi, len, runs, totals);
        PLK_HIP(hipGetLastError());
        hipLaunchKernelGGL(scan_top_kernel, dim3(1), dim3(SCAN), 0, dev.stream, totals, nb);
        PLK_HIP(hipGetLastError());
        if (nb == 1 && shots >= std::max<size_t>(8192, 4 * static_cast<size_t>(len))) {
            const uint64_t blocks = std::min<uint64_t>((shots + PB - 1) / PB, static_cast<uint64_t>(dev.num_cus) * 4);
            hipLaunchKernelGGL((sample_chunk_kernel<T>), dim3(static_cast<unsigned>(blocks)), dim3(PB), 0, dev.stream,
                               psi, static_cast<uint32_t>(len), runs, s.n, static_cast<uint64_t>(shots), seed, out);
        } else {
            hipLaunchKernelGGL((sample_kernel<T>), dim3(static_cast<unsigned>((shots + PB / 64 - 1) / (PB / 64))),
                               dim3(PB), 0, dev.stream, psi, len, runs, totals, nb, s.n,
                               static_cast<uint64_t>(shots), seed, out);
        }
        PLK_HIP(hipGetLastError());
        PLK_HIP(hipMemcpyAsync(host_out, out, out_bytes, hipMemcpyDeviceToHost, dev.stream));
    }
    PLK_HIP(hipStreamSynchronize(dev.stream));
}

} // namespace

void probs(Device &dev, const State &s, const std::vector<int> &gbits, double *host_out) {
    if (s.dtype == PLK_C64) {
        probs_t<float>(dev, s, gbits, host_out);
    } else {
        probs_t<double>(dev, s, gbits, host_out);
    }
}

void sample(Device &dev, const State &s, size_t shots, uint64_t seed, size_t *host_out) {
    if (s.dtype == PLK_C64) {
        sample_t<float>(dev, s, shots, seed, host_out);
    } else {
        sample_t<double>(dev, s, shots, seed, host_out);
    }
}

} // namespace plk
