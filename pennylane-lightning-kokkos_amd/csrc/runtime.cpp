// Device context, error plumbing and kernel statistics.
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

#include <chrono>

#include "plk_internal.hpp"

namespace plk {

[[noreturn]] void raise(int code, const std::string &msg) { throw Error{code, msg}; }

void check_hip(hipError_t e, const char *what) {
    if (e != hipSuccess) {
        const int code = (e == hipErrorOutOfMemory) ? PLK_ERR_OOM : PLK_ERR_HIP;
        raise(code, std::string("HIP error ") + hipGetErrorString(e) + " in " + what);
    }
}

namespace {
std::mutex g_dev_mutex;
std::map<int, std::unique_ptr<Device>> g_devices;
} // namespace

std::recursive_mutex &engine_mutex() {
    static std::recursive_mutex m;
    return m;
}

void set_device(int id) { PLK_HIP(hipSetDevice(id)); }

Device &device(int id) {
    std::lock_guard<std::mutex> lock(g_dev_mutex);
    auto it = g_devices.find(id);
    if (it != g_devices.end()) {
        set_device(id);
        return *it->second;
    }
    int count = 0;
    PLK_HIP(hipGetDeviceCount(&count));
    if (id < 0 || id >= count) {
        raise(PLK_ERR_INVALID, "device id " + std::to_string(id) + " out of range (" +
                                   std::to_string(count) + " devices)");
    }
    auto d = std::make_unique<Device>();
    d->id = id;
    set_device(id);
    PLK_HIP(hipStreamCreateWithFlags(&d->stream, hipStreamNonBlocking));
    int cus = 0;
    PLK_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, id));
    d->num_cus = cus > 0 ? cus : 256;
    Device &ref = *d;
    g_devices[id] = std::move(d);
    ensure_red(ref, static_cast<size_t>(ref.num_cus) * 8 * SEG_PMAX * SEG_NJMAX, 256);
    return ref;
}

void ensure_red(Device &d, size_t partial_doubles, size_t out_doubles) {
    if (partial_doubles > d.red_cap) {
        PLK_HIP(hipStreamSynchronize(d.stream));
        if (d.red) {
            PLK_HIP(hipFree(d.red));
            d.red = nullptr;
        }
        d.red = static_cast<double *>(dev_malloc(d.id, partial_doubles * sizeof(double), "partials"));
        d.red_cap = partial_doubles;
    }
    if (out_doubles > d.red_out_cap) {
        PLK_HIP(hipStreamSynchronize(d.stream));
        if (d.red_out) {
            PLK_HIP(hipFree(d.red_out));
            d.red_out = nullptr;
        }
        d.red_out = static_cast<double *>(dev_malloc(d.id, out_doubles * sizeof(double), "reductions"));
        d.red_out_cap = out_doubles;
    }
}

void ensure_parts(Device &d, size_t doubles) {
    if (doubles > d.parts_cap) {
        PLK_HIP(hipStreamSynchronize(d.stream));
        if (d.parts) {
            PLK_HIP(hipFree(d.parts));
            d.parts = nullptr;
            d.parts_cap = 0;
        }
        const size_t cap = std::max<size_t>(doubles, size_t{1} << 16);
        d.parts = static_cast<double *>(dev_malloc(d.id, cap * sizeof(double), "partials"));
        d.parts_cap = cap;
    }
}

namespace {
uint64_t g_call = 1;
} // namespace

void begin_call() { g_call++; }

void *arena_alloc(Device &d, size_t bytes) {
    if (d.arena_call != g_call) {
        d.arena_call = g_call;
        d.arena_used = 0;
        if (!d.arena_retired.empty()) {
            PLK_HIP(hipStreamSynchronize(d.stream));
            for (void *p : d.arena_retired) {
                PLK_HIP(hipFree(p));
            }
            d.arena_retired.clear();
        }
    }
    const size_t need = (bytes + 255) & ~size_t{255};
    if (d.arena_used + need > d.arena_cap) {
        // Earlier regions of this call may still be read by queued kernels:
        // the outgrown chunk is retired, not freed.
        if (d.arena) {
            d.arena_retired.push_back(d.arena);
        }
        const size_t cap = std::max(need + (size_t{1} << 20), 2 * d.arena_cap);
        d.arena = dev_malloc(d.id, cap, "plan tables");
        d.arena_cap = cap;
        d.arena_used = 0;
    }
    void *p = static_cast<unsigned char *>(d.arena) + d.arena_used;
    d.arena_used += need;
    return p;
}

void *ensure_work(Device &d, size_t bytes) {
    if (bytes > d.work_cap) {
        PLK_HIP(hipStreamSynchronize(d.stream));
        if (d.work) {
            PLK_HIP(hipFree(d.work));
            d.work = nullptr;
            d.work_cap = 0;
        }
        d.work = dev_malloc(d.id, bytes, "workspace");
        d.work_cap = bytes;
    }
    return d.work;
}

double *ensure_jac(Device &d, size_t doubles) {
    if (doubles > d.jac_cap) {
        PLK_HIP(hipStreamSynchronize(d.stream));
        if (d.jac) {
            PLK_HIP(hipFree(d.jac));
            d.jac = nullptr;
            d.jac_cap = 0;
        }
        const size_t cap = std::max<size_t>(doubles, 4096);
        d.jac = static_cast<double *>(dev_malloc(d.id, cap * sizeof(double), "Jacobian"));
        d.jac_cap = cap;
    }
    return d.jac;
}

// ---------------------------------------------------------------------------
// Kernel statistics. Events are recorded around launches without blocking;
// their durations are resolved when statistics are read.
// ---------------------------------------------------------------------------
namespace {
struct Pending {
    std::string family;
    double bytes;
    hipEvent_t e0, e1;
};
std::mutex g_prof_mutex;
bool g_prof_on = false;
std::vector<Pending> g_pending;
std::map<std::string, KernelStats> g_stats;

void resolve_pending() {
    for (auto &p : g_pending) {
        PLK_HIP(hipEventSynchronize(p.e1));
        float ms = 0.f;
        PLK_HIP(hipEventElapsedTime(&ms, p.e0, p.e1));
        auto &s = g_stats[p.family];
        s.launches += 1;
        s.ms += ms;
        s.bytes += p.bytes;
        PLK_HIP(hipEventDestroy(p.e0));
        PLK_HIP(hipEventDestroy(p.e1));
    }
    g_pending.clear();
}
} // namespace

bool profiling_on() { return g_prof_on; }

namespace {
bool g_capturing = false;
} // namespace

void set_capturing(bool on) { g_capturing = on; }

ProfScope::ProfScope(const char *f, double b, hipStream_t s) : family(f), bytes(b), stream(s) {
    // Event timing does not apply to work recorded into a graph.
    if (!g_prof_on || g_capturing) {
        return;
    }
    PLK_HIP(hipEventCreate(&e0));
    PLK_HIP(hipEventCreate(&e1));
    PLK_HIP(hipEventRecord(e0, stream));
}

ProfScope::~ProfScope() {
    if (!e0) {
        return;
    }
    if (hipEventRecord(e1, stream) != hipSuccess) {
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        return;
    }
    std::lock_guard<std::mutex> lock(g_prof_mutex);
    g_pending.push_back({family, bytes, e0, e1});
}

namespace {
double host_ms() {
    return std::chrono::duration<double, std::milli>(
               std::chrono::steady_clock::now().time_since_epoch())
        .count();
}
} // namespace

HostScope::HostScope(const char *f) : family(f) {
    if (g_prof_on) {
        t0 = host_ms();
    }
}

HostScope::~HostScope() {
    if (t0 >= 0.0) {
        record_kernel(family, static_cast<float>(host_ms() - t0), 0.0);
    }
}

void record_kernel(const char *family, float ms, double bytes) {
    std::lock_guard<std::mutex> lock(g_prof_mutex);
    auto &s = g_stats[family];
    s.launches += 1;
    s.ms += ms;
    s.bytes += bytes;
}

// Temporary states and observables' tables are recycled per device instead of
// being freed: every kernel of the library runs on the device's one stream,
// so a buffer handed out again is written (on that stream) only after the work
// that last used it. States and tables have a pool each, so that the tables of
// many observables do not keep states out; an allocation that fails releases
// both.
namespace {
struct TmpPool {
    std::multimap<size_t, void *> free;
    size_t held = 0;
};

// What a device's pool holds at most.
struct PoolLimit {
    size_t bytes, buffers;
};
constexpr PoolLimit kPoolLimit[] = {{size_t{32} << 30, SIZE_MAX}, // Pool::States
                                    {size_t{1} << 30, 4096}};     // Pool::Tables

std::mutex g_pool_mutex;
std::map<int, TmpPool> g_pools[2];

void release_pool(int dev) {
    std::vector<void *> bufs;
    {
        std::lock_guard<std::mutex> lock(g_pool_mutex);
        for (auto &pools : g_pools) {
            TmpPool &p = pools[dev];
            for (auto &kv : p.free) {
                bufs.push_back(kv.second);
            }
            p.free.clear();
            p.held = 0;
        }
    }
    if (!bufs.empty()) {
        (void)hipDeviceSynchronize();
        for (void *b : bufs) {
            (void)hipFree(b);
        }
    }
}
} // namespace

void *dev_malloc(int device, size_t bytes, const char *what) {
    void *p = nullptr;
    hipError_t e = hipMalloc(&p, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        release_pool(device);
        e = hipMalloc(&p, bytes);
    }
    if (e == hipSuccess) {
        if (g_prof_on) {
            record_kernel("device_alloc", 0.f, static_cast<double>(bytes));
        }
        return p;
    }
    (void)hipGetLastError();
    raise(PLK_ERR_OOM, "device allocation of " + std::to_string(bytes) + " bytes failed (" + what + ")");
}

void *pool_take(Pool kind, int dev, size_t bytes, const char *what) {
    {
        std::lock_guard<std::mutex> lock(g_pool_mutex);
        TmpPool &p = g_pools[static_cast<int>(kind)][dev];
        auto it = p.free.find(bytes);
        if (it != p.free.end()) {
            void *d = it->second;
            p.held -= bytes;
            p.free.erase(it);
            return d;
        }
    }
    return dev_malloc(dev, bytes, what);
}

void pool_give(Pool kind, int dev, size_t bytes, void *d) {
    {
        std::lock_guard<std::mutex> lock(g_pool_mutex);
        TmpPool &p = g_pools[static_cast<int>(kind)][dev];
        const PoolLimit &most = kPoolLimit[static_cast<int>(kind)];
        if (p.held + bytes <= most.bytes && p.free.size() < most.buffers) {
            p.free.emplace(bytes, d);
            p.held += bytes;
            return;
        }
    }
    // Kernels enqueued on this buffer must finish before it is released.
    (void)hipDeviceSynchronize();
    (void)hipFree(d);
}

TmpState::TmpState(int n, int dtype, int dev) {
    s.n = n;
    s.dtype = dtype;
    s.len = size_t{1} << n;
    s.device = dev;
    s.d = pool_take(Pool::States, dev, s.bytes(), "temporary state");
}

TmpState::~TmpState() {
    if (s.d) {
        pool_give(Pool::States, s.device, s.bytes(), s.d);
    }
}

} // namespace plk

namespace plk {

void profiling_enable_impl(bool on) {
    std::lock_guard<std::mutex> lock(g_prof_mutex);
    resolve_pending();
    g_stats.clear();
    g_prof_on = on;
}

KernelStats profiling_get_impl(const std::string &kernel) {
    std::lock_guard<std::mutex> lock(g_prof_mutex);
    resolve_pending();
    auto it = g_stats.find(kernel);
    return it == g_stats.end() ? KernelStats{} : it->second;
}

std::string profiling_names_impl() {
    std::lock_guard<std::mutex> lock(g_prof_mutex);
    resolve_pending();
    std::string s;
    for (auto &kv : g_stats) {
        if (!s.empty()) {
            s += ",";
        }
        s += kv.first;
    }
    return s;
}

} // namespace plk

namespace plk {

namespace {
// f(variant of the chunk nj).
template <typename F> void with_chunk(int nj, F &&f) {
    switch (nj) {
    case 0: f(std::integral_constant<int, 0>{}); return;
    case 1: f(std::integral_constant<int, 1>{}); return;
    case 2: f(std::integral_constant<int, 2>{}); return;
    case 3: f(std::integral_constant<int, 3>{}); return;
    case 4: f(std::integral_constant<int, 4>{}); return;
    default: break;
    }
    static_assert(RT_NJMAX == 4, "one case per chunk");
    raise(PLK_ERR_INVALID, "unsupported register-tile observable chunk " + std::to_string(nj));
}
} // namespace

int rtile_blocks(const Device &dev, int dtype, const RtLaunch &L) {
    int blocks = 0;
    if (L.nslots < 0 || L.nslots > RT_SLOTS_MAX) {
        raise(PLK_ERR_INVALID, "register-tile pass with too many sums");
    }
    with_chunk(L.nj, [&](auto NJ) {
        constexpr int nj = decltype(NJ)::value;
        blocks = dtype == PLK_C64 ? rtile_blocks_t<float, nj>(dev, L, L.nc)
                                  : rtile_blocks_t<double, nj>(dev, L, L.nc);
    });
    return blocks;
}

void launch_rtile(Device &dev, const State &phi, const State *phi_out, void *const *h_ptrs,
                  const void *d_prog, const RtLaunch &L, double *partials) {
    if (L.wide != (phi.dtype == PLK_C128 ? 1 : 0) && !(L.wide == 1 && L.nj == 0)) {
        raise(PLK_ERR_INVALID, "register-tile pass of another precision than the state's");
    }
    if (L.R < rt_reg_min(phi.dtype, L.nj) || L.R > rt_reg_max(phi.dtype, L.nj) || L.T != L.R + RT_LANE_BITS || L.T > L.n || L.n != phi.n || L.nslots > RT_SLOTS_MAX || L.nj < 0 ||
        L.nc < 1 || L.nc * std::max(1, L.nj) > RT_OBS_MAX || (L.nc > 1 && L.nj == 0) || L.nbig < 0 ||
        L.nbig > L.nc || (L.nj == 1 && L.nbig < L.nc) || (L.nslots > 0 && partials == nullptr)) {
        raise(PLK_ERR_INVALID, "register-tile pass does not match the state");
    }
    if (phi_out != nullptr && (phi_out->len != phi.len || phi_out->dtype != phi.dtype)) {
        raise(PLK_ERR_INVALID, "register-tile pass: output state of another shape");
    }
    if (L.nc > 1 && L.write_phi && (phi_out == nullptr || phi_out->d == phi.d)) {
        raise(PLK_ERR_INVALID, "register-tile pass: chunks side by side need a separate output");
    }
    void *out = phi_out ? phi_out->d : phi.d;
    const int blocks = rtile_blocks(dev, phi.dtype, L);
    with_chunk(L.nj, [&](auto NJ) {
        constexpr int nj = decltype(NJ)::value;
        if (phi.dtype == PLK_C64) {
            rtile_launch_t<float, nj>(dev, phi, out, h_ptrs, d_prog, L, blocks, partials);
        } else {
            rtile_launch_t<double, nj>(dev, phi, out, h_ptrs, d_prog, L, blocks, partials);
        }
    });
}

} // namespace plk
