// transfer.hip -- staged copies between host and device (transfer.hpp).
//
// hipMemcpy from ordinary memory stages or pins pages itself: 22 us for 8 B,
// 28 us for 16 kB, 14 us for 80 kB, 67 us for 1 MB and 30 GB/s for 590 MB,
// where the link carries 57 GB/s.  Here the caller's data go through pinned
// buffers kept from call to call, where that is faster:
//   * small uploads and several columns of up to 512 KiB in all (a track): one
//     kernel reads the buffer over the link and writes them where they belong
//     (8 B 15 us, 32 kB 16 us; tracks of 500, 7000, 16000 points 24, 30 and
//     42 us, where four hipMemcpy take 64, 52 and 65 us);
//   * several columns above that, and uploads from 16 MiB on: up to kMaxWorkers
//     threads fill large buffers while the copy engine empties those filled
//     before (one thread's memcpy runs at 28 GB/s; a copy costs the engine 14 us
//     however small, hence the large buffers): 590 MB 20.7 -> 12 ms, four
//     columns of 0.16, 0.48 and 1.2 MB 67, 106 and 230 us against 67, 132 and 330;
//   * small downloads (8 B 15 us, 32 kB 19 us against 22 and 24; 64 kB 20 us,
//     where hipMemcpy takes 13 or 36).
// In between hipMemcpy is the faster one: one column of 80 kB 14 us against 17
// by the kernel, of 3 MB 147 against 192 by the buffers, of 8 MB 345 against
// 475; 80 kB down 14 against 21.
#include "transfer.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "parallel.hpp"
#include "st_common.hpp"

namespace st {

namespace {

constexpr int kMaxWorkers = 2;
// Where the lines above lie: bytes that the kernel takes of one column and that a
// small download has at most, and from which one column uses the large buffers
// (one worker more for each kPerWorker).
constexpr size_t kSmall = (size_t)64 << 10, kLargeFrom = (size_t)16 << 20;
constexpr size_t kPerWorker = (size_t)8 << 20;
constexpr size_t kSlot[2] = {(size_t)512 << 10, (size_t)8 << 20};   // bytes of a buffer (small, large)
constexpr size_t kKeep[2] = {16, kMaxWorkers};   // pairs of buffers kept for a device (16 + 32 MiB)

// A pair of buffers, filled and copied in turn on the null stream, as
// hipMemcpy copies.
struct Stage {
    int dev = 0, kind = 0;
    char *slot[2] = {nullptr, nullptr};
    hipEvent_t ev[2] = {nullptr, nullptr};   // the last copy from each buffer
};

std::mutex g_stage_mu;
struct StageLists {
    std::vector<Stage *> of[2];
};
auto &g_stages = (new StageLists)->of;   // (never destroyed: objects may be freed at exit)

void destroy(Stage *s)
{
    if (s->slot[0]) (void)hipHostFree(s->slot[0]);
    for (hipEvent_t e : s->ev)
        if (e) (void)hipEventDestroy(e);
    delete s;
}

// A stage on the current device (null: none to be had).
Stage *take(int kind)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    {
        std::lock_guard<std::mutex> lock(g_stage_mu);
        std::vector<Stage *> &kept = g_stages[kind];
        for (size_t i = kept.size(); i-- > 0;)
            if (kept[i]->dev == dev) {
                Stage *s = kept[i];
                kept.erase(kept.begin() + (std::ptrdiff_t)i);
                return s;
            }
    }
    Stage *s = new (std::nothrow) Stage;
    if (!s) return nullptr;
    s->dev = dev;
    s->kind = kind;
    bool ok = hipHostMalloc((void **)&s->slot[0], 2 * kSlot[kind], hipHostMallocDefault) == hipSuccess;
    if (!ok) s->slot[0] = nullptr;
    for (hipEvent_t &e : s->ev) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
    if (!ok) {
        (void)hipGetLastError();
        destroy(s);
        return nullptr;
    }
    s->slot[1] = s->slot[0] + kSlot[kind];
    return s;
}

// (no copy from it is under way)
void give(Stage *s)
{
    {
        std::lock_guard<std::mutex> lock(g_stage_mu);
        std::vector<Stage *> &kept = g_stages[s->kind];
        const size_t same =
            (size_t)std::count_if(kept.begin(), kept.end(), [&](const Stage *k) { return k->dev == s->dev; });
        try {
            if (same < kKeep[s->kind]) {
                kept.push_back(s);
                return;
            }
        } catch (const std::bad_alloc &) {
        }
    }
    destroy(s);
}

// What [p, p + bytes), which the caller names as host memory, is.  Staging reads
// and writes it with memcpy: all else (device memory, a range past its pinned
// allocation) is left to hipMemcpy, which copies or refuses it.
enum class HostRange { ordinary, pinned, other };
HostRange host_range(const void *p, size_t bytes)
{
    if (!p) return HostRange::other;
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return HostRange::ordinary;
    }
    if (a.type == hipMemoryTypeUnregistered) return HostRange::ordinary;
    if (a.type != hipMemoryTypeHost && a.type != hipMemoryTypeManaged) return HostRange::other;
    hipDeviceptr_t start = nullptr;
    size_t size = 0;
    if (hipMemGetAddressRange(&start, &size, const_cast<void *>(p)) != hipSuccess) {
        (void)hipGetLastError();
        return HostRange::other;
    }
    const bool inside = (uintptr_t)p >= (uintptr_t)start && (uintptr_t)p - (uintptr_t)start + bytes <= size;
    return inside ? HostRange::pinned : HostRange::other;
}

hipError_t plain_upload(const UploadPart *parts, int n)
{
    for (int i = 0; i < n; ++i) {
        if (parts[i].bytes == 0) continue;
        const hipError_t e = hipMemcpy(parts[i].dst, parts[i].src, parts[i].bytes, hipMemcpyHostToDevice);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// A buffer's parts to where they belong, blockIdx.y a part.
constexpr int kGatherParts = 4;
struct GatherArgs {
    struct {
        char *dst;
        const char *src;   // 256-byte aligned
        size_t bytes;
    } part[kGatherParts];
};

template <typename Word>
__device__ __forceinline__ void copy_words(char *dst, const char *src, size_t bytes)
{
    const size_t i0 = (size_t)blockIdx.x * 256 + threadIdx.x, stride = (size_t)gridDim.x * 256;
    const size_t words = bytes / sizeof(Word);
    for (size_t i = i0; i < words; i += stride) ((Word *)dst)[i] = ((const Word *)src)[i];
    for (size_t i = words * sizeof(Word) + i0; i < bytes; i += stride) dst[i] = src[i];
}

__global__ __launch_bounds__(256) void gather_kernel(GatherArgs a)
{
    char *const dst = a.part[blockIdx.y].dst;
    const char *const src = a.part[blockIdx.y].src;
    const size_t bytes = a.part[blockIdx.y].bytes;
    if (((uintptr_t)dst & 15) == 0) copy_words<uint4>(dst, src, bytes);
    else copy_words<uint2>(dst, src, bytes);
}

// Copies up to kGatherParts parts, which fit a small buffer together, with the
// kernel.
hipError_t gather_upload(Stage *s, const UploadPart *parts, int n)
{
    GatherArgs a{};
    size_t used = 0, most = 0;
    int k = 0;
    for (int i = 0; i < n; ++i) {
        if (parts[i].bytes == 0) continue;
        std::memcpy(s->slot[0] + used, parts[i].src, parts[i].bytes);
        a.part[k++] = {(char *)parts[i].dst, s->slot[0] + used, parts[i].bytes};
        used += (parts[i].bytes + 255) / 256 * 256;
        most = std::max(most, parts[i].bytes);
    }
    const dim3 grid((unsigned)((most / 16 + 255) / 256 + 1), (unsigned)k);
    hipError_t e = launch(gather_kernel, grid, 256, 0, nullptr, a);
    if (e != hipSuccess) return e;
    e = hipEventRecord(s->ev[0], nullptr);
    const hipError_t waited = e == hipSuccess ? hipEventSynchronize(s->ev[0]) : hipStreamSynchronize(nullptr);
    return e == hipSuccess ? waited : e;
}

// The parts cut into pieces of at most a buffer, small neighbours sharing one.
struct Piece {
    int part;
    size_t at, bytes, slot_at;
};

// Copies the parts through large buffers, several threads filling them.
hipError_t large_upload(const UploadPart *parts, int n, size_t total)
{
    const size_t cap = kSlot[1];
    std::vector<Piece> pieces;
    std::vector<size_t> fills;   // first piece of each buffer's fill
    size_t used = cap;
    for (int i = 0; i < n; ++i)
        for (size_t at = 0; at < parts[i].bytes;) {
            if (used + 256 > cap) {
                fills.push_back(pieces.size());
                used = 0;
            }
            const size_t b = std::min(parts[i].bytes - at, cap - used);
            pieces.push_back({i, at, b, used});
            at += b;
            used += (b + 255) / 256 * 256;
        }
    const size_t n_fills = fills.size();
    fills.push_back(pieces.size());

    std::vector<std::thread> pool;
    std::vector<Stage *> stages;
    pool.reserve(kMaxWorkers);
    stages.reserve(kMaxWorkers);
    Stage *first = take(1);
    if (!first) return plain_upload(parts, n);
    stages.push_back(first);
    std::atomic<size_t> next{0};
    std::atomic<int> failed{(int)hipSuccess};
    auto work = [&](Stage *s) {
        hipError_t e = hipSuccess;
        int used = 0;
        for (int k = 0; e == hipSuccess && failed.load() == (int)hipSuccess; ++k) {
            const size_t f = next.fetch_add(1);
            if (f >= n_fills) break;
            char *buf = s->slot[k & 1];
            if (k >= 2) e = hipEventSynchronize(s->ev[k & 1]);
            used = std::max(used, (k & 1) + 1);
            for (size_t i = fills[f]; e == hipSuccess && i < fills[f + 1]; ++i) {
                const Piece &p = pieces[i];
                std::memcpy(buf + p.slot_at, (const char *)parts[p.part].src + p.at, p.bytes);
                e = hipMemcpyAsync((char *)parts[p.part].dst + p.at, buf + p.slot_at, p.bytes, hipMemcpyHostToDevice,
                                   nullptr);
            }
            const hipError_t noted = hipEventRecord(s->ev[k & 1], nullptr);
            if (e == hipSuccess) e = noted;
        }
        for (int k = 0; k < used; ++k) {
            const hipError_t waited = hipEventSynchronize(s->ev[k]);
            if (e == hipSuccess) e = waited;
        }
        if (e != hipSuccess) failed.store((int)e);
    };
    const size_t helpers = std::min<size_t>({(size_t)std::min(kMaxWorkers, host_threads()) - 1, total / kPerWorker,
                                             n_fills - 1});
    for (size_t w = 0; w < helpers; ++w) {
        Stage *s = take(1);
        if (!s) break;
        try {
            pool.emplace_back([&work, s] {
                if (hipSetDevice(s->dev) == hipSuccess) work(s);
            });
        } catch (const std::exception &) {
            give(s);   // the others do its share
            break;
        }
        stages.push_back(s);
    }
    work(first);
    for (std::thread &t : pool) t.join();
    for (Stage *s : stages) give(s);
    return (hipError_t)failed.load();
}

hipError_t staged_upload(const UploadPart *parts, int n, size_t total)
{
    int columns = 0;
    size_t padded = 0;
    bool aligned = true;
    for (int i = 0; i < n; ++i) {
        if (parts[i].bytes == 0) continue;
        ++columns;
        padded += (parts[i].bytes + 255) / 256 * 256;
        aligned = aligned && ((uintptr_t)parts[i].dst & 7) == 0;
    }
    const bool gather = aligned && columns <= kGatherParts && padded <= kSlot[0] && (columns > 1 || total <= kSmall);
    if (!gather && (columns > 1 ? total <= kSlot[0] : total < kLargeFrom)) return plain_upload(parts, n);
    for (int i = 0; i < n; ++i) {
        if (parts[i].bytes == 0) continue;
        const HostRange range = host_range(parts[i].src, parts[i].bytes);
        // (the copy engine reads pinned memory itself; host memory in the device's
        // place is for hipMemcpy to refuse; the kernel's stores are checked by no
        // one else)
        if (range == HostRange::other) return plain_upload(parts, n);
        if (gather ? !dev_writable(parts[i].dst, parts[i].bytes)
                   : range == HostRange::pinned || !dev_known(parts[i].dst))
            return plain_upload(parts, n);
    }
    if (!gather) return large_upload(parts, n, total);
    Stage *s = take(0);
    if (!s) return plain_upload(parts, n);
    const hipError_t e = gather_upload(s, parts, n);
    give(s);
    return e;
}

}  // namespace

hipError_t upload(const UploadPart *parts, int n)
{
    size_t total = 0;
    for (int i = 0; i < n; ++i) {
        total += parts[i].bytes;
        const hipError_t e = dev_check(parts[i].dst, parts[i].bytes);
        if (e != hipSuccess) return e;
    }
    if (total == 0) return hipSuccess;
    try {
        return staged_upload(parts, n, total);
    } catch (const std::bad_alloc &) {   // (thrown before anything is queued)
        return plain_upload(parts, n);
    }
}

hipError_t download(void *dst, const void *src, size_t bytes)
{
    if (bytes == 0) return hipSuccess;
    hipError_t e = dev_check(src, bytes);
    if (e != hipSuccess) return e;
    Stage *s = bytes <= kSmall && host_range(dst, bytes) != HostRange::other && dev_known(src) ? take(0) : nullptr;
    if (!s) return hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost);
    e = hipMemcpyAsync(s->slot[0], src, bytes, hipMemcpyDeviceToHost, nullptr);
    if (e == hipSuccess) e = hipEventRecord(s->ev[0], nullptr);
    const hipError_t waited = e == hipSuccess ? hipEventSynchronize(s->ev[0]) : hipStreamSynchronize(nullptr);
    if (e == hipSuccess) e = waited;
    if (e == hipSuccess) std::memcpy(dst, s->slot[0], bytes);
    give(s);
    return e;
}

void staging_shutdown()
{
    std::lock_guard<std::mutex> lock(g_stage_mu);
    for (std::vector<Stage *> &kept : g_stages) {
        for (Stage *s : kept) destroy(s);
        kept.clear();
    }
}

}  // namespace st
