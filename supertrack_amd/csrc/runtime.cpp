// runtime.cpp -- status strings, device memory helpers, geometry and bin
// edges of libsupertrack_amd (host code).
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdarg>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <set>
#include <vector>

#include "st_common.hpp"
#include "st_internal.hpp"
#include "transfer.hpp"

namespace st {

namespace {
thread_local std::string g_last_error;
}

int set_error(int code, const char *fmt, ...)
{
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    std::vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_last_error = buf;
    return code;
}

void clear_error() { g_last_error.clear(); }

namespace {
// st_debug_fail_allocation: allocations left before the one that fails (0: off)
std::atomic<int64_t> g_fail_countdown{0};

bool injected_failure()
{
    int64_t c = g_fail_countdown.load();
    while (c > 0) {
        if (g_fail_countdown.compare_exchange_weak(c, c - 1)) return c == 1;
    }
    return false;
}
}  // namespace

namespace {
// Device blocks given back and kept for the next taker of their size.  A track
// or a small library makes and frees a handful of them; hipMalloc and hipFree
// take 2-5 us each at 80 kB, but 150-220 us at 2-8 MB.  Blocks of up to
// kPoolBlock are kept, kPoolBytes of them at most; a taker waits until the
// device is done with what used the block before it was given back, as hipFree
// would have.  A block given back to a full pool takes the place of those kept
// longest; an allocation that fails gives all of them back and tries again.
constexpr size_t kPoolBlock = (size_t)16 << 20, kPoolBytes = (size_t)32 << 20;
struct Kept {
    void *p;
    uint64_t given;   // g_pool_clock when it was given back
};
std::mutex g_pool_mu;
// (the maps are never destroyed: objects may be freed at exit)
auto &g_pool = *new std::map<std::pair<int, size_t>, std::vector<Kept>>;          // (device, size)
struct Live {
    int dev;
    size_t size, asked;   // bytes of the block, and those its taker asked for
};
auto &g_pool_live = *new std::map<uintptr_t, Live>;   // blocks handed out
auto &g_pool_synced = *new std::map<int, uint64_t>;   // device: blocks given back before this are free of work
size_t g_pool_bytes = 0;
uint64_t g_pool_clock = 0;

// Four sizes to an octave.
size_t pool_size(size_t bytes)
{
    size_t step = 256;
    while (bytes > step * 4) step *= 2;
    return (bytes + step - 1) / step * step;
}

// The handed-out block that holds p (g_pool_mu held).
std::map<uintptr_t, Live>::iterator live_block(const void *p)
{
    auto it = g_pool_live.upper_bound((uintptr_t)p);
    if (it == g_pool_live.begin()) return g_pool_live.end();
    --it;
    return (uintptr_t)p - it->first < it->second.size ? it : g_pool_live.end();
}

// Notes that [p, p + bytes) was allocated anew: handed-out blocks noted there
// were freed by other means (g_pool_mu held).
void forget_blocks(const void *p, size_t bytes)
{
    auto it = g_pool_live.lower_bound((uintptr_t)p);
    while (it != g_pool_live.end() && it->first - (uintptr_t)p < bytes) it = g_pool_live.erase(it);
    if (it == g_pool_live.begin()) return;
    --it;
    if (it->first + it->second.size > (uintptr_t)p) g_pool_live.erase(it);
}

// Whether p lies in a kept block, one given back already (g_pool_mu held).
bool in_kept_block(const void *p)
{
    for (const auto &size : g_pool)
        for (const Kept &k : size.second)
            if (p >= k.p && (uintptr_t)p - (uintptr_t)k.p < size.first.second) return true;
    return false;
}

// Waits until the device is done with all that was queued, as hipFree does
// before it frees anything.  (hipDeviceSynchronize, which costs 0.3 us where
// this costs 1.3, is not allowed while any thread captures a stream, and ends
// that capture; hipMalloc and hipFree are, unless this thread forbids them.)
hipError_t wait_for_device()
{
    void *p = nullptr;
    hipError_t e = hipMalloc(&p, 256);
    if (e == hipSuccess) e = hipFree(p);
    return e;
}

// All kept blocks back to the device (g_pool_mu held).
void pool_trim()
{
    for (auto &size : g_pool)
        for (const Kept &k : size.second) (void)hipFree(k.p);
    g_pool.clear();
    g_pool_bytes = 0;
}
}  // namespace

hipError_t dev_malloc(void **p, size_t bytes)
{
    *p = nullptr;
    if (injected_failure()) return hipErrorOutOfMemory;
    int dev = 0;
    if (bytes == 0 || bytes > kPoolBlock || hipGetDevice(&dev) != hipSuccess) {
        hipError_t e = hipMalloc(p, bytes);
        if (e == hipErrorOutOfMemory) {
            std::lock_guard<std::mutex> lock(g_pool_mu);
            if (g_pool_bytes > 0) {
                (void)hipGetLastError();
                pool_trim();
                e = hipMalloc(p, bytes);
            }
        }
        if (e == hipSuccess) {
            std::lock_guard<std::mutex> lock(g_pool_mu);
            forget_blocks(*p, bytes);
        }
        return e;
    }
    const size_t size = pool_size(bytes);
    Kept got{nullptr, 0};
    uint64_t now = 0;
    bool clean = false;
    {
        std::lock_guard<std::mutex> lock(g_pool_mu);
        auto it = g_pool.find({dev, size});
        if (it != g_pool.end() && !it->second.empty()) {
            got = it->second.back();
            it->second.pop_back();
            g_pool_bytes -= size;
            now = ++g_pool_clock;
            auto synced = g_pool_synced.find(dev);
            clean = synced != g_pool_synced.end() && got.given < synced->second;
        }
    }
    if (got.p && !clean) {
        const hipError_t e = wait_for_device();
        if (e != hipSuccess && hipFree(got.p) == hipSuccess) {
            (void)hipGetLastError();   // (a full device, say: a block of its own)
            got.p = nullptr;
        } else {
            std::lock_guard<std::mutex> lock(g_pool_mu);
            try {
                if (e == hipSuccess) {
                    uint64_t &synced = g_pool_synced[dev];
                    synced = std::max(synced, now);
                } else {   // (under a capture that forbids both: the block stays)
                    g_pool[{dev, size}].push_back(got);
                    g_pool_bytes += size;
                }
            } catch (const std::bad_alloc &) {   // (waited for again the next time)
            }
            if (e != hipSuccess) return e;
        }
    }
    if (!got.p) {
        hipError_t e = hipMalloc(&got.p, size);
        if (e == hipErrorOutOfMemory) {
            (void)hipGetLastError();
            std::lock_guard<std::mutex> lock(g_pool_mu);
            pool_trim();
            e = hipMalloc(&got.p, size);
        }
        if (e != hipSuccess) return e;
    }
    try {
        std::lock_guard<std::mutex> lock(g_pool_mu);
        forget_blocks(got.p, size);
        g_pool_live[(uintptr_t)got.p] = {dev, size, bytes};
    } catch (const std::bad_alloc &) {   // no host memory to note it in: freed straight away later
    }
    *p = got.p;
    return hipSuccess;
}

hipError_t dev_free(void *p)
{
    if (!p) return hipSuccess;
    std::vector<void *> evicted;   // the blocks kept longest make room
    bool kept = false;
    {
        std::lock_guard<std::mutex> lock(g_pool_mu);
        auto it = live_block(p);
        // (a block given back twice would be handed out twice)
        if (it == g_pool_live.end() ? in_kept_block(p) : (uintptr_t)p - it->first >= it->second.asked)
            return hipErrorInvalidValue;
        if (it != g_pool_live.end()) {
            const std::pair<int, size_t> where{it->second.dev, it->second.size};
            p = (void *)it->first;   // (as hipFree, which takes any address inside an allocation)
            g_pool_live.erase(it);
            try {
                while (g_pool_bytes + where.second > kPoolBytes) {
                    auto oldest = g_pool.end();
                    for (auto k = g_pool.begin(); k != g_pool.end(); ++k)
                        if (!k->second.empty() &&
                            (oldest == g_pool.end() || k->second.front().given < oldest->second.front().given))
                            oldest = k;
                    if (oldest == g_pool.end()) break;
                    evicted.push_back(oldest->second.front().p);
                    oldest->second.erase(oldest->second.begin());
                    g_pool_bytes -= oldest->first.second;
                }
                if (g_pool_bytes + where.second <= kPoolBytes) {
                    g_pool[where].push_back({p, ++g_pool_clock});
                    g_pool_bytes += where.second;
                    kept = true;
                }
            } catch (const std::bad_alloc &) {
            }
        }
    }
    for (void *old : evicted) (void)hipFree(old);
    if (kept) return hipSuccess;
    return hipFree(p);
}

hipError_t dev_check(const void *p, size_t bytes)
{
    std::lock_guard<std::mutex> lock(g_pool_mu);
    auto it = live_block(p);
    return it != g_pool_live.end() && (uintptr_t)p - it->first + bytes > it->second.asked ? hipErrorInvalidValue
                                                                                          : hipSuccess;
}

bool dev_known(const void *p)
{
    {
        std::lock_guard<std::mutex> lock(g_pool_mu);
        if (live_block(p) != g_pool_live.end()) return true;
    }
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
    (void)hipGetLastError();
    return false;
}

bool dev_writable(const void *p, size_t bytes)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    {
        std::lock_guard<std::mutex> lock(g_pool_mu);
        auto it = live_block(p);
        if (it != g_pool_live.end())
            return it->second.dev == dev && (uintptr_t)p - it->first + bytes <= it->second.asked;
    }
    hipPointerAttribute_t a{};
    hipDeviceptr_t start = nullptr;
    size_t size = 0;
    if (hipPointerGetAttributes(&a, p) != hipSuccess || a.type != hipMemoryTypeDevice || a.device != dev ||
        hipMemGetAddressRange(&start, &size, const_cast<void *>(p)) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return (uintptr_t)p >= (uintptr_t)start && (uintptr_t)p - (uintptr_t)start + bytes <= size;
}

namespace {
// Slots of pinned, mapped host memory that the device reports into, kept for
// the next caller: making one costs about 25 us.  At most kKeptSlots of a
// size wait unused; st_shutdown gives them back.
constexpr size_t kSlotBytes[] = {4096, 65536};
constexpr size_t kKeptSlots = 8;
std::mutex g_slot_mu;
struct SlotLists {
    std::vector<void *> of[2];
};
// (never destroyed, as above)
auto &g_slots = (new SlotLists)->of;
auto &g_slots_live = *new std::set<void *>;   // slots handed out

int slot_class(size_t bytes) { return bytes <= kSlotBytes[0] ? 0 : 1; }
}  // namespace

void *report_slot_take(size_t bytes, bool counted)
{
    if (bytes > kSlotBytes[1] || (counted && injected_failure())) return nullptr;
    const int c = slot_class(bytes);
    {
        std::lock_guard<std::mutex> lock(g_slot_mu);
        if (!g_slots[c].empty()) {
            void *p = g_slots[c].back();
            try {
                g_slots_live.insert(p);
            } catch (const std::bad_alloc &) {
                return nullptr;
            }
            g_slots[c].pop_back();
            return p;
        }
    }
    void *p = nullptr;
    void *mapped = nullptr;   // kernels store through the same address (unified addressing)
    if (hipHostMalloc(&p, kSlotBytes[c], hipHostMallocMapped | hipHostMallocPortable | hipHostMallocCoherent) !=
        hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    bool ok = hipHostGetDevicePointer(&mapped, p, 0) == hipSuccess && mapped == p;
    try {
        std::lock_guard<std::mutex> lock(g_slot_mu);
        if (ok) g_slots_live.insert(p);
    } catch (const std::bad_alloc &) {
        ok = false;
    }
    if (!ok) (void)hipHostFree(p);
    return ok ? p : nullptr;
}

void report_slot_give(void *p, size_t bytes)
{
    if (!p) return;
    const int c = slot_class(bytes);
    {
        std::lock_guard<std::mutex> lock(g_slot_mu);
        if (g_slots_live.erase(p) == 0) {
            // given back already, or not one of these slots
            for (const std::vector<void *> &kept : g_slots)
                if (std::find(kept.begin(), kept.end(), p) != kept.end()) return;
        } else if (g_slots[c].size() < kKeptSlots) {
            try {
                g_slots[c].push_back(p);
                return;
            } catch (const std::bad_alloc &) {
            }
        }
    }
    (void)hipHostFree(p);
}

namespace {
// per-device default streams, created on first use, destroyed by st_shutdown
std::mutex g_stream_mu;
std::vector<hipStream_t> g_streams;
}  // namespace

hipStream_t default_stream()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    std::lock_guard<std::mutex> lock(g_stream_mu);
    if ((int)g_streams.size() <= dev) g_streams.resize(dev + 1, nullptr);
    if (!g_streams[dev]) {
        hipStream_t s = nullptr;
        if (hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess) return nullptr;
        g_streams[dev] = s;
    }
    return g_streams[dev];
}

int device_cu_count()
{
    static int cached = 0;
    if (cached) return cached;
    int dev = 0;
    hipDeviceProp_t p;
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&p, dev) != hipSuccess) return 256;
    cached = p.multiProcessorCount;
    return cached;
}

// SphericalGeometry::SphericalGeometry (SphericalGeometry.cu:34-58).
void make_geometry(double half_length_ini, double diameter_ini, st_geometry *g)
{
    const double D = diameter_ini;
    const double r = D / 2;
    int N = (int)std::floor((half_length_ini * 2) / D);
    double L = N * D;
    double H = L / 2;
    double gso = -H + r;
    if (r > H) {  // sphere larger than the voxel
        H = r;
        N = 1;
        L = H * 2;
        gso = -H + r;
    }
    g->half_length = H;
    g->length = L;
    g->diameter = D;
    g->radius = r;
    g->gso = gso;
    g->n_linear = N;
    g->pad = 0;
}

// utils::LinSpace / utils::LogSpace (utils.cc:8-31).  The limits arrive as
// floats (Histogram.cu:34-35 reads them with GetFloat) and the width is a
// float quotient widened to double, so edges carry the float truncation.
void make_edges(int type, float lo, float hi, int nbins, double *edges)
{
    if (type == ST_HIST_LIN) {
        const float wf = (hi - lo) / (float)nbins;
        const double w = wf;
        for (int i = 0; i <= nbins; ++i) edges[i] = (double)lo + (double)i * w;
    } else {
        const float bo = (float)std::log10((double)lo);
        const float to = (float)std::log10((double)hi);
        const float wf = (to - bo) / (float)nbins;
        const double w = wf;
        for (int i = 0; i <= nbins; ++i) edges[i] = std::pow(10.0, (double)bo + (double)i * w);
    }
}

}  // namespace st

using namespace st;

extern "C" {

const char *st_last_error(void) { return g_last_error.c_str(); }

const char *st_version(void) { return "supertrack_amd 0.1 (gfx950)"; }

int st_device_count(int *count)
{
    if (!count) return set_error(ST_EINVAL, "st_device_count: null pointer");
    ST_HIP_TRY(hipGetDeviceCount(count));
    return ST_OK;
}

int st_malloc(void **ptr, size_t bytes)
{
    if (!ptr) return set_error(ST_EINVAL, "st_malloc: null pointer");
    *ptr = nullptr;
    if (bytes == 0) return ST_OK;
    hipError_t e = dev_malloc(ptr, bytes);
    if (e != hipSuccess) {
        *ptr = nullptr;
        return set_error(ST_ENOMEM, "hipMalloc(%zu) failed: %s", bytes, hipGetErrorString(e));
    }
    return ST_OK;
}

int st_free(void *ptr)
{
    if (ptr) ST_HIP_TRY(dev_free(ptr));
    return ST_OK;
}

// The helpers below are ordered after all device work queued so far on any
// stream (the library's streams are non-blocking, so a plain hipMemcpy on the
// null stream would not wait for them) and complete before returning.
int st_memcpy_htod(void *dst, const void *src, size_t bytes)
{
    if (!bytes) return ST_OK;
    ST_HIP_TRY(hipDeviceSynchronize());
    const UploadPart part{dst, src, bytes};
    ST_HIP_TRY(upload(&part, 1));
    return ST_OK;
}

int st_memcpy_dtoh(void *dst, const void *src, size_t bytes)
{
    if (!bytes) return ST_OK;
    ST_HIP_TRY(hipDeviceSynchronize());
    ST_HIP_TRY(download(dst, src, bytes));
    return ST_OK;
}

int st_memcpy_dtod(void *dst, const void *src, size_t bytes)
{
    if (!bytes) return ST_OK;
    ST_HIP_TRY(dev_check(dst, bytes));
    ST_HIP_TRY(dev_check(src, bytes));
    ST_HIP_TRY(hipDeviceSynchronize());
    ST_HIP_TRY(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToDevice));
    ST_HIP_TRY(hipDeviceSynchronize());
    return ST_OK;
}

int st_memset(void *dst, int value, size_t bytes)
{
    if (!bytes) return ST_OK;
    ST_HIP_TRY(dev_check(dst, bytes));
    ST_HIP_TRY(hipDeviceSynchronize());
    ST_HIP_TRY(hipMemset(dst, value, bytes));
    ST_HIP_TRY(hipDeviceSynchronize());
    return ST_OK;
}

int st_device_synchronize(void)
{
    ST_HIP_TRY(hipDeviceSynchronize());
    return ST_OK;
}

int st_debug_fail_allocation(int64_t countdown)
{
    if (countdown < 0) return set_error(ST_EINVAL, "st_debug_fail_allocation: countdown < 0");
    g_fail_countdown.store(countdown);
    return ST_OK;
}

int st_shutdown(void)
{
    staging_shutdown();
    {
        std::lock_guard<std::mutex> pool(g_pool_mu);
        pool_trim();
    }
    {
        std::lock_guard<std::mutex> slots(g_slot_mu);
        for (std::vector<void *> &kept : g_slots) {
            for (void *p : kept) (void)hipHostFree(p);
            kept.clear();
        }
    }
    std::lock_guard<std::mutex> lock(g_stream_mu);
    int cur = 0;
    const bool have_cur = hipGetDevice(&cur) == hipSuccess;
    int rc = ST_OK;
    for (int dev = 0; dev < (int)g_streams.size(); ++dev) {
        if (!g_streams[dev]) continue;
        hipError_t e = hipSetDevice(dev);
        if (e == hipSuccess) e = hipStreamSynchronize(g_streams[dev]);
        if (e == hipSuccess) e = hipStreamDestroy(g_streams[dev]);
        if (e != hipSuccess && rc == ST_OK)
            rc = set_error(ST_EHIP, "st_shutdown: device %d: %s", dev, hipGetErrorString(e));
        g_streams[dev] = nullptr;
    }
    if (have_cur) (void)hipSetDevice(cur);
    return rc;
}

int st_default_stream(void **hip_stream)
{
    if (!hip_stream) return set_error(ST_EINVAL, "st_default_stream: null pointer");
    hipStream_t s = default_stream();
    if (!s) return set_error(ST_EHIP, "st_default_stream: could not create a stream");
    *hip_stream = (void *)s;
    return ST_OK;
}

int st_geometry_make(double half_length_ini, double diameter_ini, st_geometry *out)
{
    if (!out) return set_error(ST_EINVAL, "st_geometry_make: null output");
    if (!(diameter_ini > 0) || !(half_length_ini >= 0) || !std::isfinite(diameter_ini) ||
        !std::isfinite(half_length_ini))
        return set_error(ST_EINVAL, "st_geometry_make: need finite half length >= 0 and diameter > 0 "
                                    "(got %g, %g)", half_length_ini, diameter_ini);
    make_geometry(half_length_ini, diameter_ini, out);
    if ((double)out->n_linear * out->n_linear * (double)out->n_linear > 1.8e19)
        return set_error(ST_ERANGE, "st_geometry_make: %d spheres per axis overflow 64-bit keys",
                         out->n_linear);
    return ST_OK;
}

}  // extern "C"
