// wave_kernel.hpp -- the batched form's default kernel (included by batch.hip
// only): one wavefront scores a (track, oversample) segment, or a part of one,
// on its own, with its own sphere table in LDS.
//
// What bounds it: instruction issue (256 tracks, 2 nm spheres, x 1000: about 85
// vector and 80 scalar instructions per row of 64 points, vector units busy
// 0.8 of the time), whatever a point's bytes (points are re-read from L2 by the
// track's other oversamples), so the layout below is chosen to leave out
// instructions and waits, not bytes:
//   * no workgroup barrier between the start and the end of the kernel: the
//     occupancy check of the table is a scalar compare, a flush runs on 64
//     dense list entries per step, and segment set-up is done once per wave
//     and segment instead of by every wave of a workgroup;
//   * table keys are bit fields (x | y << bx | z << by), formed by three
//     shift-adds (the last may hold a copy number below them);
//     the hash is a rank-1 lattice over the three indices (24-bit multiply-adds,
//     constants of the R3 low-discrepancy sequence): neighbouring spheres land
//     far apart, 2.5 probes for the longest lane of a row where a
//     multiplicative hash of the key takes 3.0 (2 nm spheres, a quarter full);
//   * large segments are cut into parts at sphere layers, so that one
//     segment's points spread over several waves when there are few segments;
//   * workgroup histograms go to a slab of their own and are summed by
//     slab_sum_kernel: merging with atomics makes every workgroup wait on the
//     few hot bins (a library of 16 small tracks spent 0.35 of 0.42 ms there).
// Tracks whose flush survivors or key box do not fit (TrackDesc::wave unset) are
// scored by batch_kernel.
#pragma once

#include "batch_kernel.hpp"

namespace st {
namespace {

static_assert(kQueues == 8, "one work queue per XCD");

// The work queues.  Track positions of the order are dealt to the queues in
// turn (queue q: positions q, q + 8, ...); each track is cut into chunks of
// about the points it names, and prefix counts the chunks before it in its
// queue.
struct PlanTrack {
    int64_t prefix;
    int32_t track;
    int32_t chunk_points;
};
struct WavePlan {
    const PlanTrack *tracks;   // queue q's from tracks + q * stride
    const int64_t *total;      // chunks per queue
    int64_t stride;
    int32_t n_tracks;
    unsigned long long *tickets;   // [kQueues * kTicketPad], cleared per pass
};

// What the host reads of a pass's control block.
struct CtlReport {
    unsigned long long rec_count;
    unsigned long long stats[kStats];
    int error, pad;
};

struct WaveArgs {
    BatchArgs b;
    WavePlan plan;
    CtlReport *report;              // where slab_sum_kernel reports the pass (host memory; null: nowhere)
    unsigned int *slab;             // [workgroup][hist_lds_words]; null: merge with atomics
    unsigned long long *slab_stats; // [workgroup][kStats]
};

// Oversamples per chunk (tracks of at most chunk_points points) and parts per
// segment (larger ones).
__host__ __device__ inline int chunk_oversamples(int n, int chunk_points)
{
    if (n >= chunk_points) return 1;
    const int c = chunk_points / (n > 0 ? n : 1);
    return c > 64 ? 64 : c;
}

__host__ __device__ inline int segment_parts(int n, int chunk_points)
{
    return n <= chunk_points ? 1 : (n + chunk_points - 1) / chunk_points;
}

__host__ __device__ inline int64_t track_chunks(int n, int n_os, int chunk_points)
{
    const int c = chunk_oversamples(n, chunk_points);
    return (int64_t)((n_os + c - 1) / c) * segment_parts(n, chunk_points);
}

// Largest chunk: larger ones add nothing to the share of a segment's set-up, and
// an oversample more per chunk makes the waves uneven (4096 tracks of up to 1e6
// points, no bound: x 100 in FP64 20.1 ms, x 1000 at 2 nm 165.0; 2^20: 19.3 and
// 162.1; 2^18: 17.7 and 160.7; 2^16: 17.7 and 168.4).
constexpr int kMaxChunk = 1 << 18;

// Builds the queues.  A chunk holds a fixed share of the points still to come
// in the order (largest tracks first), at least min_points: large chunks while
// much is left, small ones at the end, so that the last wave to finish is not
// late.  As first written: fixed chunks, 24 per wave: 6.8 ms on a mixed library of 96 tracks x
// 1000 oversamples and 1.11 ms on 256 tracks x 100; 48 per wave: 6.2 and 1.28
// ms; this: 5.9 and 1.06 ms.
__global__ __launch_bounds__(64 * kQueues) void wave_plan_kernel(const TrackDesc *tracks, const int32_t *order,
                                                                 int32_t n_tracks, int32_t n_os, int64_t points,
                                                                 double per_point, int32_t min_points,
                                                                 int64_t stride, PlanTrack *plan, int64_t *total)
{
    __shared__ int64_t s_wave[kQueues];
    __shared__ int64_t s_chunks[64 * kQueues];
    const int tid = threadIdx.x, q = tid >> 6, lane = tid & 63;
    int64_t before = 0;   // points of the tracks before this block of positions
    int64_t base = 0;     // queue q's chunks before it
    auto scan = [&](int64_t v) {
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int64_t t = __shfl_up(v, d, 64);
            if (lane >= d) v += t;
        }
        return v;
    };
    for (int64_t p0 = 0; p0 < n_tracks; p0 += 64 * kQueues) {
        const int64_t p = p0 + tid;
        const int n = p < n_tracks ? tracks[order[p]].n : 0;
        const int64_t incl = scan(n);
        if (lane == 63) s_wave[q] = incl;
        __syncthreads();
        int64_t left = points - before - (incl - n);
        for (int w = 0; w < q; ++w) left -= s_wave[w];
        const int per = (int)fmin(fmax((double)left * per_point, (double)min_points), (double)kMaxChunk);
        s_chunks[tid] = p < n_tracks ? track_chunks(n, n_os, per) : 0;
        if (p < n_tracks) {
            PlanTrack &e = plan[(p % kQueues) * stride + p / kQueues];
            e.track = order[p];
            e.chunk_points = per;
        }
        for (int w = 0; w < kQueues; ++w) before += s_wave[w];
        __syncthreads();
        const int64_t mine = p0 + q + (int64_t)kQueues * lane;   // position of this queue's lane-th track of the block
        const int64_t c = s_chunks[q + kQueues * lane];
        const int64_t sum = scan(c);
        if (mine < n_tracks) plan[q * stride + mine / kQueues].prefix = base + sum - c;
        base += __shfl(sum, 63, 64);
        __syncthreads();
    }
    if (lane == 0) total[q] = base;
}

__device__ __forceinline__ double uniform_f64(double v)
{
    return __longlong_as_double(uniform_i64(__double_as_longlong(v)));
}

// Orders this wave's LDS accesses for the compiler (a wave's LDS instructions
// execute in order).
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ int lanes_below(unsigned long long mask)
{
    return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
}

// Table slots of a wave, flush threshold and list capacity.  A flush at a
// quarter full keeps the probe chains short, and its entries then mostly fill
// the two rows of 64 that it handles together (256 tracks x 1000, 2 nm spheres,
// as first written: 320 slots 14.1 ms, 384 13.8, 416 13.6, 432 13.9; 416 slots
// now: a flush at 88 entries 11.3 ms, 104 10.8, 120 11.6); the list holds what a flush
// keeps (at most kWaveWindow, or fewer than the threshold) and one row of 64
// points.
constexpr int kWaveSlots = 416;
constexpr int wave_flush_at(int slots) { return slots / 4; }
constexpr int wave_list(int slots)
{
    const int keep = wave_flush_at(slots) - 1 > (int)kWaveWindow ? wave_flush_at(slots) - 1 : (int)kWaveWindow;
    return keep + 64;
}
// Hot tracks flush at 64 entries: before a flush they hold at most the larger
// of 63 and kHotCopies * kHotWindow entries and one row's, and merging copies
// may add an entry for each of at most 63 + 64 spheres.
constexpr int kHotFlushAt = 64;
static_assert(kHotCopies * kHotWindow + 64 + 127 <= wave_list(kWaveSlots), "the list holds a hot track's entries");
// LDS bytes of one wave's table and list
constexpr int wave_lds(int words, int slots)
{
    return (slots * (8 * words + 4) + wave_list(slots) * 2 + 15) / 16 * 16;
}

// What the wave's rare paths need of the current segment: in LDS, so that it
// holds no registers through the point loop.
struct WaveRare {
    ExactParams e;
    const double *x, *y, *z;   // the track's FP64 points
    int64_t seg;               // track * oversamples + oversample (recording)
    double ox, oy, oz;         // lattice-unit offsets that make the rounded coordinates local indices
    float fx, fy, fz;          // ST_F32: the rest of ox.. beside its nearest integer,
    int kx, ky, kz;            // and the integer
};

__device__ __forceinline__ bool lane_of(unsigned long long mask)
{
    return __builtin_amdgcn_inverse_ballot_w64(mask);
}

// a * b + c of 24-bit a, b
__device__ __forceinline__ unsigned mad24(unsigned a, unsigned b, unsigned c)
{
    unsigned r;
    asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(b), "v"(c));
    return r;
}

// Slots are named by the byte offset of their key (four times their number).
// Home slot: the low 24 bits of lx * a + ly * b + lz * c (a, b, c the R3
// sequence's fractions in 2^24ths) scaled to the table size.
// copy: kCopyHash times the entry's copy number (0 unless the track is hot).
constexpr unsigned kLatticeX = 13743434u, kLatticeY = 11258244u, kLatticeZ = 9222436u;
constexpr unsigned kCopyHash = 7555035u;
// Rounds an FP32 number below 2^22 to an integer when added: the low bits of
// the sum are the integer, above them this number's.
constexpr float kMagic32 = 12582912.0f;   // 1.5 * 2^23
constexpr int kMagic32Bits = 0x4B400000;
template <int SLOTS>
__device__ __forceinline__ unsigned lattice_slot(unsigned lx, unsigned ly, unsigned lz, unsigned copy)
{
    const unsigned h = mad24(lx, kLatticeX, mad24(ly, kLatticeY, mad24(lz, kLatticeZ, copy)));
    return (unsigned)(((unsigned long long)(h & 0xFFFFFFu) * (unsigned)(SLOTS << 10)) >> 32) & ~3u;
}

// The slot after (the last one wraps: the smaller of the two as unsigned numbers).
template <int SLOTS>
__device__ __forceinline__ unsigned lattice_next(unsigned slot)
{
    return min(slot + 4u, slot + 4u - 4u * (unsigned)SLOTS);
}

// First i in [0, n) with pred(i), else n, by one wave (n uniform, the answer
// too); 64-way steps.
template <typename Pred>
__device__ __forceinline__ int wave_first(int n, Pred pred)
{
    const int lane = threadIdx.x & 63;
    int lo = 0, hi = n;
#pragma unroll 1
    while (lo < hi) {
        const int step = (hi - lo + 63) >> 6;
        const int i = lo + lane * step;
        bool p = true;
        if (i < hi) p = pred(i);
        const unsigned long long mask = __ballot(p);
        // lane f: the first that holds; the answer lies in (its predecessor, it]
        const int f = mask ? __ffsll((long long)mask) - 1 : 64;
        const int top = f < 64 ? lo + f * step : hi;
        lo = f > 0 ? lo + (f - 1) * step + 1 : lo;
        hi = min(top, hi);
    }
    return lo;
}

// The same pointer, opaque to the compiler: what is loaded through it is
// loaded here again (scalar cache), not kept in registers from an earlier use.
template <typename T>
__device__ __forceinline__ const T *reload(const T *p)
{
    asm volatile("" : "+s"(p));
    return p;
}

// The same value in scalar registers of its own (a member of a loaded record
// would keep the whole record's registers alive).
__device__ __forceinline__ double detach(double v)
{
    double r;
    asm("s_mov_b64 %0, %1" : "=s"(r) : "s"(v));
    return r;
}

// The same value in every lane's vector registers (scalar ones are spilled
// around the point loop and read back for each row).
__device__ __forceinline__ float to_lanes(float v)
{
    float r;
    asm("v_mov_b32 %0, %1" : "=v"(r) : "s"(v));
    return r;
}

__device__ __forceinline__ double to_lanes(double v)
{
    double r;
    asm("v_mov_b64 %0, %1" : "=v"(r) : "s"(v));
    return r;
}

template <typename T>
__device__ __forceinline__ const T *detach(const T *p)
{
    const T *r;
    asm("s_mov_b64 %0, %1" : "=s"(r) : "s"(p));
    return r;
}

// A load from device memory at a byte offset from a uniform base.  (Through a
// pointer whose memory the compiler does not know it would be a flat load,
// which the wait for any LDS operation waits for too: 256 tracks, 10 nm
// spheres, x 100 in FP64 1.52 ms, this 1.42.)
template <typename T>
__device__ __forceinline__ T load_global(const void *base, uint64_t offset)
{
    using Bytes = const __attribute__((address_space(1))) char *;
    return *(const __attribute__((address_space(1))) T *)((Bytes)base + offset);
}
typedef float Float4 __attribute__((ext_vector_type(4)));
typedef double Double2 __attribute__((ext_vector_type(2), aligned(8)));

// Acc<ST_F32>::value of a sum below 2^52 units: its bits under the exponent
// whose unit is 2^-32, less that exponent's value.
__device__ __forceinline__ double small_value(unsigned long long v0)
{
    return __longlong_as_double((long long)(v0 | 0x4130000000000000ull)) - 1048576.0;
}
constexpr unsigned kMerged32 = 0xFFFFFFFEu;   // key of a merged copy (above every sphere key)

// wave_kernel's arguments (its only parameter) in the argument segment, read
// where they are used: scalar loads, not registers held through the point loop.
typedef const __attribute__((address_space(4))) WaveArgs *ArgsPtr;
__device__ __forceinline__ ArgsPtr args_here()
{
    ArgsPtr q = (ArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(q));
    return q;
}

// Counts two sums per lane (those of the masks) in histogram h.
__device__ __forceinline__ void bin_two(ArgsPtr args, int h, const double (&v)[2], const unsigned long long (&mask)[2],
                                        unsigned int *lhist)
{
    const auto &hd = args->b.hist[h];
    // what the common case needs of the histogram, in one wait (as the code
    // came to need them they were five scalar waits and two rounds of edge
    // loads: 2 nm spheres, 256 tracks x 1000, 11.21 -> 10.76 ms, with a branch
    // in place of both conversions of the sums)
    int type = hd.guess.type, nbins = hd.guess.nbins;
    float log2_origin = hd.guess.log2_origin, log2_inv_width = hd.guess.log2_inv_width;
    const double *edges = hd.edges;
    int in_lds = args->b.hist_lds_words, lds_offset = hd.lds_offset;
    asm volatile("" : "+s"(type), "+s"(nbins), "+s"(log2_origin), "+s"(log2_inv_width), "+s"(edges), "+s"(in_lds),
                 "+s"(lds_offset));
    // closed-form guesses, clamped into [0, nbins - 1]: always a valid load
    float f[2];
    if (type == ST_HIST_LIN) {
#pragma unroll
        for (int u = 0; u < 2; ++u) f[u] = (float)((v[u] - hd.guess.origin) * hd.guess.inv_width);
    } else {
#pragma unroll
        for (int u = 0; u < 2; ++u) f[u] = (__log2f((float)v[u]) - log2_origin) * log2_inv_width;
    }
    asm volatile("" : "+v"(f[0]), "+v"(f[1]));   // (one branch for both)
    const float top = (float)(nbins - 1);
    int b[2];
    double lo[2], hi[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        b[u] = (int)__builtin_amdgcn_fmed3f(f[u], 0.0f, top);
        const Double2 pair = load_global<Double2>(edges, (unsigned)b[u] * 8u);
        lo[u] = pair.x;
        hi[u] = pair.y;
    }
    unsigned long long miss[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) miss[u] = mask[u] & ~(__ballot(v[u] >= lo[u]) & __ballot(v[u] < hi[u]));
    if ((miss[0] | miss[1]) != 0ull) {   // the guess missed: exact search (-1: outside)
        BinGuess g;
        g.type = hd.guess.type;
        g.nbins = hd.guess.nbins;
        g.origin = hd.guess.origin;
        g.inv_width = hd.guess.inv_width;
        g.log2_origin = hd.guess.log2_origin;
        g.log2_inv_width = hd.guess.log2_inv_width;
        g.e0 = hd.guess.e0;
        g.en = hd.guess.en;
#pragma unroll 1
        for (int u = 0; u < 2; ++u) {
            if (!lane_of(u ? miss[1] : miss[0])) continue;
            const int f = bin_fast(hd.edges, g, u ? v[1] : v[0]);
            if (u) b[1] = f;
            else b[0] = f;
        }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        if (lane_of(mask[u]) && b[u] >= 0) {
            if (in_lds) atomicAdd(&lhist[lds_offset + b[u]], 1u);
            else atomicAdd(&hd.bins[b[u]], 1ull);
        }
    }
}

template <int MODE, int SLOTS, int WPE>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(WPE)))
void wave_kernel(WaveArgs wa)
{
    const BatchArgs &a = wa.b;
    constexpr int kFlushAt = wave_flush_at(SLOTS);
    constexpr int kList = wave_list(SLOTS);
    constexpr int kWords = Acc<MODE>::words;
    static_assert(kList <= SLOTS * 9 / 10, "the table must hold the survivors of a flush plus one row");
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ WaveRare s_rare[16];
    __shared__ unsigned long long s_stats[kStats];
    __shared__ unsigned s_empty;   // queues found empty (bit mask)

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = uniform_i32(tid >> 6);
    const int n_waves = blockDim.x >> 6;
    unsigned char *const mine = smem + wave * wave_lds(kWords, SLOTS);
    unsigned long long *const tacc0 = reinterpret_cast<unsigned long long *>(mine);
    unsigned long long *const tacc1 = tacc0 + SLOTS;   // kWords == 2
    unsigned int *const tkey = reinterpret_cast<unsigned int *>(mine + SLOTS * 8 * kWords);
    // a slot's key and sums
    auto key_of = [&](unsigned slot) -> unsigned & { return *(unsigned *)((char *)tkey + slot); };
    auto acc0_of = [&](unsigned slot) -> unsigned long long & { return *(unsigned long long *)((char *)tacc0 + 2u * slot); };
    auto acc1_of = [&](unsigned slot) -> unsigned long long & { return *(unsigned long long *)((char *)tacc1 + 2u * slot); };
    unsigned short *const tlist = reinterpret_cast<unsigned short *>(mine + SLOTS * (8 * kWords + 4));
    unsigned int *const lhist = reinterpret_cast<unsigned int *>(smem + n_waves * wave_lds(kWords, SLOTS));
    WaveRare &rare = s_rare[wave];
    ExactParams &ex = rare.e;

    for (int s = lane; s < SLOTS; s += 64) {
        tkey[s] = kEmpty32;
        tacc0[s] = 0;
        if (kWords == 2) tacc1[s] = 0;
    }
    for (int w = tid; w < a.hist_lds_words; w += blockDim.x) lhist[w] = 0;
    if (tid < kStats) s_stats[tid] = 0;
    if (tid == 0) s_empty = 0;
    __syncthreads();

    // statistics (BatchCtl::stats): per lane, or per wave where uniform
    // (n_in, n_created, n_retired: of the current segment, added to s_stats at
    // its end)
    unsigned int n_flagged = 0;
    unsigned long long bal_in = 0, bal_out = 0;
    unsigned int n_in = 0, n_created = 0, n_retired = 0, unspilled = 0;
    int cnt = 0;            // entries in the table (uniform)

    int queue = blockIdx.x & (kQueues - 1);   // workgroups are dealt to the XCDs in turn
    int j_last = 0;         // the queue's track position of the last chunk
    bool first = true;
    for (;;) {
        // ---- take a chunk ----
        // (queues known to be empty, by any wave of the workgroup, cost no
        // further ticket)
        const unsigned empty = uniform_u32(__hip_atomic_load(&s_empty, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
        if (!first && empty == (1u << kQueues) - 1u) break;
        if (!first && ((empty >> queue) & 1u)) {
            queue = (queue + 1) & (kQueues - 1);
            j_last = 0;
            continue;
        }
        // A queue's first chunks, one for each wave of its own workgroups, are
        // dealt out without tickets (tickets on one address pass at about one
        // per 10 ns: 6144 waves asking at once cost 0.06 ms).
        const int64_t n_chunks = wa.plan.total[queue];
        const int64_t dealt = (int64_t)(((int)gridDim.x - queue + kQueues - 1) / kQueues) * n_waves;
        int64_t tk;
        if (first) {
            tk = (int64_t)(blockIdx.x / kQueues) * n_waves + wave;
            first = false;
        } else if (n_chunks > dealt) {
            unsigned long long ticket = 0;
            if (lane == 0) ticket = atomicAdd(&wa.plan.tickets[queue * kTicketPad], 1ull);
            tk = dealt + uniform_i64((long long)ticket);
        } else {
            tk = n_chunks;
        }
        if (tk >= n_chunks) {
            if (lane == 0) atomicOr(&s_empty, 1u << queue);
            continue;
        }
        // the track holding chunk tk: the last prefix entry <= tk
        int32_t t, chunk, chunk_points;
        {
            const PlanTrack *q = wa.plan.tracks + queue * wa.plan.stride;
            const int nq = (wa.plan.n_tracks - queue + kQueues - 1) / kQueues;
            const int from = j_last + 1;
            j_last += wave_first(nq - from, [&](int i) { return q[from + i].prefix > tk; });
            t = uniform_i32(q[j_last].track);
            chunk_points = uniform_i32(q[j_last].chunk_points);
            chunk = (int)(tk - uniform_i64(q[j_last].prefix));
        }
        int os0, part, parts;
        unsigned long long alive;
        {
            const TrackDesc td = load_uniform(a.tracks + t);
            const GeomDev g = load_uniform(a.geoms + td.geom);
            const int per = uniform_i32(chunk_oversamples(td.n, chunk_points));
            parts = uniform_i32(segment_parts(td.n, chunk_points));
            os0 = uniform_i32(chunk / parts);
            part = chunk - os0 * parts;
            os0 *= per;
            const double zmin = load_uniform(a.zfirst + td.block0);
            // the chunk's oversamples that reach the voxel (exact: fl(x + s) is
            // monotone in x), one lane each
            bool ok = false;
            const int os = os0 + lane;
            if (lane < per && os < a.n_os) {
                const Shift sh = shift_for(a.seed, a.track_index_base + (uint32_t)t, (uint32_t)os, a.shift_xy,
                                           a.shift_z, g.L, g.H);
                ok = (td.xmax + sh.x) > -g.H && (td.xmin + sh.x) < g.H && (td.ymax + sh.y) > -g.H &&
                     (td.ymin + sh.y) < g.H && ((td.zmax + g.H) + sh.z) > -g.H && ((zmin + g.H) + sh.z) < g.H;
            }
            alive = __ballot(ok);
        }
        while (alive != 0ull) {
            const int os = os0 + __ffsll((long long)alive) - 1;
            alive &= alive - 1ull;
            // (records read again per segment: kept in registers from the
            // chunk's start they would be spilled around the point loop)
            const TrackDesc td = load_uniform(reload(a.tracks + t));
            const GeomDev g = load_uniform(reload(a.geoms + td.geom));
            const double zmin = load_uniform(a.zfirst + td.block0);
            // what the point loop needs of the segment (uniform)
            unsigned nx, ny, nz;
            int k_first, row, r_end;
            // key = copy | lx << bits_c | ly << bits_x | lz << bits_xy
            int bits_c, bits_x, bits_xy;
            int in_lo, in_hi;   // rows [in_lo, in_hi) are full and hold only points inside the key box
            {
                const Shift sh = shift_for(a.seed, a.track_index_base + (uint32_t)t, (uint32_t)os, a.shift_xy,
                                           a.shift_z, g.L, g.H);
                // The segment's box of sphere indices (as in batch_kernel).
                const unsigned N = (unsigned)g.N;
                const double fN1 = (double)(N - 1u);
                const double bx0 = fmax(0.0, floor(((td.xmin + sh.x) - g.gso) * g.invD) - 1.0);
                const double bx1 = fmin(fN1, ceil(((td.xmax + sh.x) - g.gso) * g.invD) + 1.0);
                const double by0 = fmax(0.0, floor(((td.ymin + sh.y) - g.gso) * g.invD) - 1.0);
                const double by1 = fmin(fN1, ceil(((td.ymax + sh.y) - g.gso) * g.invD) + 1.0);
                const double bz0 = fmax(0.0, floor((((zmin + g.H) + sh.z) - g.gso) * g.invD) - 1.0);
                const double bz1 = fmin(fN1, ceil((((td.zmax + g.H) + sh.z) - g.gso) * g.invD) + 1.0);
                if (__ballot(bx0 <= bx1 && by0 <= by1 && bz0 <= bz1) == 0ull) continue;
                const unsigned kx0 = uniform_u32((unsigned)bx0), ky0 = uniform_u32((unsigned)by0);
                nx = uniform_u32((unsigned)bx1) - kx0 + 1u;
                ny = uniform_u32((unsigned)by1) - ky0 + 1u;
                const int kz_lo = uniform_i32((int)bz0), kz_hi = uniform_i32((int)bz1);
                // block range of the segment (blocks whose z span can reach
                // the voxel's layers)
                const double *zf = a.zfirst + td.block0;
                const double zlo = fmax(-g.H, g.gso + ((double)kz_lo - 1.0) * g.D);
                const double zhi = fmin(g.H, g.gso + ((double)kz_hi + 1.0) * g.D);
                const int b_hi = wave_first(td.nblocks, [&](int b) { return !(((zf[b] + g.H) + sh.z) < zhi); });
                const int b_lo = wave_first(b_hi, [&](int b) {
                    const double zhb = (b + 1 < td.nblocks) ? zf[b + 1] : td.zmax;
                    return ((zhb + g.H) + sh.z) > zlo;
                });
                if (b_lo >= b_hi) continue;
                if (part == 0 && lane == 0)
                    atomicAdd(&s_stats[0], (unsigned long long)(min(b_hi * kBlk, td.n) - b_lo * kBlk));
                // The segment's parts: block cut points, and between them the
                // sphere layers above the layer of the cut's first point
                // (points of that layer, before and after the cut, belong to
                // the part before it).  A point's layer, rounded as the
                // reference rounds it, never decreases along the track.  A key
                // box that spans the voxel in y stays whole: there a face
                // point's carried index may name a sphere of the next layer.
                const int parts_here = (ky0 == 0u && ny == N) ? 1 : min(parts, b_hi - b_lo);
                if (part >= parts_here) continue;
                auto layer_of = [&](int b) {
                    return (int)nearest_index(((zf[b] + g.H) + sh.z) - g.gso, g.D, g.invD);
                };
                int c0 = b_lo, c1 = b_hi, k_last = kz_hi;
                k_first = kz_lo;
                if (parts_here > 1) {
                    const int64_t len = b_hi - b_lo;
                    c0 = b_lo + uniform_i32((int)(len * part / parts_here));
                    if (part > 0) k_first = max(kz_lo, uniform_i32(layer_of(c0)) + 1);
                    if (part < parts_here - 1) {
                        const int next = b_lo + uniform_i32((int)(len * (part + 1) / parts_here));
                        const int cut = uniform_i32(layer_of(next));
                        k_last = min(kz_hi, cut);
                        c1 = next + wave_first(b_hi - next, [&](int b) { return layer_of(next + b) > cut; });
                    }
                    if (k_first > k_last) continue;
                }
                nz = uniform_u32((unsigned)(k_last - k_first + 1));
                row = uniform_i32(c0 * kBlk);
                r_end = uniform_i32(min(c1 * kBlk, td.n));   // both relative to the track's first point
                // Blocks whose points all lie in the key box (their rows need
                // no box test): where the track's x/y bounds lie inside the
                // voxel, so does every index; in z, blocks that start at the
                // part's first layer or later and end before the first block
                // above its last layer.  (Decisions near a boundary are made
                // exactly in any case.)
                in_lo = in_hi = 0;
                if ((td.xmin + sh.x) > -g.H && (td.xmax + sh.x) < g.H && (td.ymin + sh.y) > -g.H &&
                    (td.ymax + sh.y) < g.H) {
                    const int i0 = c0 + wave_first(c1 - c0, [&](int b) { return layer_of(c0 + b) >= k_first; });
                    const int i1 = i0 + wave_first(c1 - i0, [&](int b) { return layer_of(i0 + b) > k_last; });
                    in_lo = uniform_i32(i0 * kBlk);
                    in_hi = uniform_i32((i1 - 1) * kBlk);
                }
                bits_c = uniform_i32((td.wave & kFlagHot) ? 2 : 0);
                bits_x = uniform_i32(bits_c + 32 - __builtin_clz(nx | 1u));
                bits_xy = uniform_i32(bits_x + (32 - __builtin_clz(ny | 1u)));
                wave_lds_fence();
                if (lane == 0) {
                    ex.H = g.H;
                    ex.gso = g.gso;
                    ex.D = g.D;
                    ex.invD = g.invD;
                    ex.r2 = g.r2;
                    ex.sx = sh.x;
                    ex.sy = sh.y;
                    ex.sz = sh.z;
                    ex.N = N;
                    ex.kx0 = kx0;
                    ex.ky0 = ky0;
                    ex.nx = nx;
                    ex.ny = ny;
                    ex.kz_lo = (unsigned)kz_lo;
                    ex.nz_all = (unsigned)(kz_hi - kz_lo + 1);
                    ex.multi = parts_here > 1 ? 1u : 0u;
                    ex.kz0 = (unsigned)k_first;
                    ex.nz = nz;
                    rare.x = a.x64 + td.offset;
                    rare.y = a.y64 + td.offset;
                    rare.z = a.z64 + td.offset;
                    rare.seg = (int64_t)t * a.n_os + os;
                    const double sqx = sh.x * g.invD, sqy = sh.y * g.invD, sqz = sh.z * g.invD;
                    rare.ox = (MODE == ST_F64 ? sqx - g.qc : sqx) - (double)kx0;
                    rare.oy = (MODE == ST_F64 ? sqy - g.qc : sqy) - (double)ky0;
                    rare.oz = (MODE == ST_F64 ? (sqz + g.H * g.invD) - g.qc : sqz) - (double)k_first;
                    if constexpr (MODE == ST_F32) {
                        const double kx = rint(rare.ox), ky = rint(rare.oy), kz = rint(rare.oz);
                        rare.kx = (int)kx;
                        rare.ky = (int)ky;
                        rare.kz = (int)kz;
                        rare.fx = (float)(rare.ox - kx);
                        rare.fy = (float)(rare.oy - ky);
                        rare.fz = (float)(rare.oz - kz);
                    }
                }
                wave_lds_fence();
            }

            // ---- stream the part's points, 64 per row ----
            using PointT = typename std::conditional<MODE == ST_F64, double4, float4>::type;
            // (the point arrays are padded: a row may be read past the last point)
            const char *const p0 = detach((const char *)(MODE == ST_F64 ? (const void *)(a.x64 + td.offset)
                                                                        : (const void *)(a.p32 + td.offset)));
            const char *const p1 = detach((const char *)(a.y64 + td.offset));
            const char *const p2 = detach((const char *)(a.z64 + td.offset));
            const char *const p3 = detach((const char *)(a.e64 + td.offset));
            unsigned at = (unsigned)(row + lane) * (MODE == ST_F64 ? 8u : 16u);   // byte offset of the lane's next point
            auto fetch = [&](PointT &dst) __attribute__((always_inline)) {
                if constexpr (MODE == ST_F64) {
                    dst = make_double4(load_global<double>(p0, at), load_global<double>(p1, at),
                                       load_global<double>(p2, at), load_global<double>(p3, at));
                } else {
                    const Float4 v = load_global<Float4>(p0, at);
                    dst = make_float4(v.x, v.y, v.z, v.w);
                }
                at += 64u * (MODE == ST_F64 ? 8u : 16u);
            };
            // the lane's copy number and its part of the hash (hot tracks: lanes
            // that share a sphere spread over kHotCopies entries, merged when
            // the sphere is complete)
            const int flush_at = uniform_i32(bits_c ? kHotFlushAt : kFlushAt);
            static_assert(kHotCopies == 4, "two key bits");
            const unsigned copy = lane & ((1u << bits_c) - 1u), copy_hash = copy * kCopyHash;
            // ST_F32: the rounded coordinates carry kMagic32's bits and count
            // from the block's sphere; these make them local indices, and the
            // key and the hash of what they carry are folded into the terms of
            // the copy (all modulo 2^32, the hash modulo 2^24)
            int cx = 0, cy = 0, cz = 0;
            unsigned key0 = copy, hash0 = copy_hash;
            auto home = [&](unsigned k) {
                return lattice_slot<SLOTS>((k >> bits_c) & ((1u << (bits_x - bits_c)) - 1u),
                                           (k >> bits_x) & ((1u << (bits_xy - bits_x)) - 1u), k >> bits_xy,
                                           (k & ((1u << bits_c) - 1u)) * kCopyHash);
            };
            const double invD = detach(g.invD), yscale = detach(g.yscale);   // (ST_F32)
            using Real = typename std::conditional<MODE == ST_F64, double, float>::type;
            constexpr Real kMagic = MODE == ST_F64 ? (Real)kRoundMagic : (Real)kMagic32;
            Real bqx, bqy, bqz, sure, maybe;
            const Real inv = MODE == ST_F64 ? (Real)invD : (Real)__int_as_float(uniform_i32(__float_as_int((float)invD)));
            if constexpr (MODE == ST_F64) {
                bqx = rare.ox;
                bqy = rare.oy;
                bqz = rare.oz;
                sure = to_lanes(g.sure);
                maybe = to_lanes(g.maybe);
            }
            const BlockF32 *blk = detach(a.blocks + td.block0);
            bool edge = false;   // the block's rows need the box and count tests
            auto new_block = [&]() __attribute__((always_inline)) {
                edge = row < in_lo || row >= in_hi;
                // block-uniform terms of the row's block (scalar loads)
                if constexpr (MODE == ST_F32) {
                    const BlockF32 bk = load_uniform(blk + row / kBlk);
                    bqx = bk.fx + rare.fx;
                    bqy = bk.fy + rare.fy;
                    bqz = bk.fz + rare.fz;
                    sure = to_lanes(bk.sure32);
                    maybe = to_lanes(bk.maybe32);
                    cx = bk.kx + uniform_i32(rare.kx) - kMagic32Bits;
                    cy = bk.ky + uniform_i32(rare.ky) - kMagic32Bits;
                    cz = bk.kz + uniform_i32(rare.kz) - kMagic32Bits;
                    key0 = copy + (((unsigned)cx << bits_c) + ((unsigned)cy << bits_x) + ((unsigned)cz << bits_xy));
                    hash0 = copy_hash + ((unsigned)cx * kLatticeX + (unsigned)cy * kLatticeY + (unsigned)cz * kLatticeZ);
                }
            };
            // Scores the row at `row`, then flushes if the table is a quarter
            // full or the part ends; returns true at its end.  (Parts start at
            // a block's first row.)
            auto step = [&](Real qx, Real qy, Real qz, double w) __attribute__((always_inline)) -> bool {
                // ST_F32: FP32 arithmetic, relative to a sphere near the block's
                // origin so that its error stays below the block's own; rows
                // with a point in doubt (0.9 % at 2 nm) go on to FP64.  19 FP64
                // instructions of a row became FP32 ones, additions and
                // products at nearly twice the rate: 256 tracks x 1000, 2 nm
                // spheres, 11.59 -> 11.21 ms; x 100, 10 nm, 1.064 -> 1.040.
                // (Decisions are kept as lane masks in scalar registers.)
                const Real tx = qx + kMagic, ty = qy + kMagic, tz = qz + kMagic;
                const Real ux = (tx - kMagic) - qx, uy = (ty - kMagic) - qy, uz = (tz - kMagic) - qz;
                unsigned lx, ly, lz;   // local indices less cx, cy, cz
                Real distq;
                if constexpr (MODE == ST_F64) {
                    distq = fma(ux, ux, fma(uy, uy, uz * uz));
                    lx = (unsigned)__double2loint(tx);
                    ly = (unsigned)__double2loint(ty);
                    lz = (unsigned)__double2loint(tz);
                } else {
                    distq = fmaf(ux, ux, fmaf(uy, uy, uz * uz));
                    lx = __float_as_uint(tx);
                    ly = __float_as_uint(ty);
                    lz = __float_as_uint(tz);
                }
                const int layer0 = (int)lz;
                unsigned long long m_in = __ballot(distq < sure);
                unsigned long long m_near = __ballot(distq <= maybe) & ~m_in;
                if (edge) {
                    const int left = r_end - row;
                    const unsigned long long m_valid = left >= 64 ? ~0ull : (1ull << left) - 1ull;
                    m_in &= m_valid & __ballot(lx + (unsigned)cx < nx) & __ballot(ly + (unsigned)cy < ny) &
                            __ballot(lz + (unsigned)cz < nz);
                    m_near &= m_valid;
                }
                if (m_near != 0ull) {
                    bool in = false;
                    if (lane_of(m_near)) {
                        bool near = true;
                        if constexpr (MODE == ST_F32) {
                            // within the error bound of FP32 arithmetic: again
                            // in FP64, from the FP32 offsets
                            const Float4 p = load_global<Float4>(p0, (uint64_t)(unsigned)(row + lane) * 16u);
                            const BlockF32 bk = load_uniform(blk + row / kBlk);
                            const double qx = fma((double)p.x, invD, bk.oqx + rare.ox);
                            const double qy = fma((double)p.y, invD, bk.oqy + rare.oy);
                            const double qz = fma((double)p.z, invD, bk.oqz + rare.oz);
                            const double tx = qx + kRoundMagic, ty = qy + kRoundMagic, tz = qz + kRoundMagic;
                            const double ux = (tx - kRoundMagic) - qx, uy = (ty - kRoundMagic) - qy,
                                         uz = (tz - kRoundMagic) - qz;
                            const double distq = fma(ux, ux, fma(uy, uy, uz * uz));
                            lx = (unsigned)__double2loint(tx);
                            ly = (unsigned)__double2loint(ty);
                            lz = (unsigned)__double2loint(tz);
                            in = distq < bk.sure && lx < nx && ly < ny && lz < nz;
                            near = distq <= bk.maybe && !(distq < bk.sure);
                        }
                        const int layer = (int)lz;
                        // any decision within the error bound is redone exactly
                        // from FP64, unless clearly outside (an index beyond the
                        // box by more than one)
                        const ExactParams &e = ex;
                        const bool in_xy = near && lx + 1u <= nx + 1u && ly + 1u <= ny + 1u;
                        if constexpr (MODE == ST_F32) {
                            // (statistic: counted against the whole segment's
                            // box, by the part that holds the layer)
                            const int k0 = (int)e.kz0 - (int)e.kz_lo;
                            const int lza = layer + k0;
                            n_flagged += in_xy && (unsigned)(lza + 1) <= e.nz_all + 1u && (layer >= 0 || k0 == 0) &&
                                         (layer < (int)nz || k0 + nz == e.nz_all);
                        }
                        if (in_xy && lz + 1u <= nz + 1u) {
                            // (batch_kernel's exact_local for bit-field keys: an
                            // index N is carried into the next one)
                            const uint64_t i8 = (uint64_t)(unsigned)(row + lane) * 8u;
                            const double x = load_global<double>(rare.x, i8), y = load_global<double>(rare.y, i8),
                                         z = load_global<double>(rare.z, i8);
                            unsigned gx, gy, gz;
                            if (exact_member(x, y, z, e, gx, gy, gz)) {
                                if (gx >= e.N) {
                                    gx -= e.N;
                                    ++gy;
                                }
                                const bool up = gy >= e.N;   // carried into the next layer
                                if (up) {
                                    gy -= e.N;
                                    ++gz;
                                }
                                lx = gx - e.kx0;
                                ly = gy - e.ky0;
                                lz = gz - e.kz0;
                                // every in-sphere point lies in the segment's box
                                // by construction; only a carried index can leave
                                // it, or its part: reported, never scored wrong
                                if (lx >= nx || ly >= ny || gz - e.kz_lo >= e.nz_all || (up && e.multi))
                                    atomicOr(&args_here()->b.ctl->error, 4);
                                in = lx < nx && ly < ny && lz < nz;
                            }
                        }
                        lx -= (unsigned)cx;
                        ly -= (unsigned)cy;
                        lz -= (unsigned)cz;
                    }
                    m_in |= __ballot(in);
                }
                n_in += (unsigned)__popcll(m_in);
                unsigned h = 0, prev = 0;
                if (lane_of(m_in)) {
                    unsigned long long v0, v1 = 0;
                    if constexpr (MODE == ST_F64) {
                        long long s0, s1;
                        Acc<ST_F64>::split(w, s0, s1);
                        v0 = (unsigned long long)s0;
                        v1 = (unsigned long long)s1;
                    } else {
                        // rint of w (the low word of the magic constant is zero)
                        const double tw = w + kRoundMagic;
                        v0 = ((unsigned long long)((unsigned)__double2hiint(tw) - 0x43380000u) << 32) |
                             (unsigned)__double2loint(tw);
                    }
                    const unsigned key = (lz << bits_xy) + ((ly << bits_x) + ((lx << bits_c) + key0));
                    h = lattice_slot<SLOTS>(lx, ly, lz, hash0);
                    prev = atomicCAS(&key_of(h), kEmpty32, key);
#pragma unroll 1
                    while (prev != kEmpty32 && prev != key) {
                        h = lattice_next<SLOTS>(h);
                        prev = atomicCAS(&key_of(h), kEmpty32, key);
                    }
                    atomicAdd(&acc0_of(h), v0);
                    if (kWords == 2) atomicAdd(&acc1_of(h), v1);
                    bal_in += Acc<MODE>::balance(v0, v1);
                }
                asm("" : "+v"(prev));   // compared once, here
                const unsigned long long m_fresh = __ballot(prev == kEmpty32);
                if (lane_of(m_fresh)) tlist[cnt + lanes_below(m_fresh)] = (unsigned short)h;
                const int added = __popcll(m_fresh);
                cnt += added;
                n_created += (unsigned)added;
                const bool last = row + 64 >= r_end;
                if (!last && cnt < flush_at) return false;
                // ---- flush: entries below `bound` are complete ----
                unsigned bound = kEmpty32;
                if (!last) {
                    // Every later point lies in a layer >= that of this row's
                    // last point; a key's layer is never below its point's.
                    // (its rounding is certain below fm, and sure <= fm^2)
                    int lb = __builtin_amdgcn_readlane(layer0, 63) + cz;
                    if (__ballot(!(uz * uz < sure)) >> 63) {
                        // rare: the exact layer, as the reference rounds it
                        const ExactParams &e = ex;
                        lb = uniform_i32((int)nearest_index(((load_global<double>(rare.z, (uint64_t)(unsigned)(row + 63) * 8u) + e.H) + e.sz) - e.gso, e.D, e.invD) -
                                         (int)e.kz0);
                    }
                    if (lb <= 0) return false;   // nothing is complete
                    if (lb < (int)nz) bound = (unsigned)lb << bits_xy;
                }
                wave_lds_fence();
                const ArgsPtr args = args_here();
                if (bits_c != 0) {
                    // the copies of complete spheres are added to copy 0 (their
                    // slots keep a key that matches no point, so no probe path
                    // breaks, until they are cleared below)
#pragma unroll 1
                    for (int r = 0; r < min(cnt, kList); r += 64) {
                        bool fresh = false;
                        unsigned h = 0;
                        if (lane < cnt - r) {
                            const unsigned sl = tlist[r + lane];
                            const unsigned k = key_of(sl);
                            if (k < bound && (k & (kHotCopies - 1u)) != 0u) {
                                const unsigned k0 = k & ~(kHotCopies - 1u);
                                h = home(k0);
                                unsigned prev = atomicCAS(&key_of(h), kEmpty32, k0);
#pragma unroll 1
                                while (prev != kEmpty32 && prev != k0) {
                                    h = lattice_next<SLOTS>(h);
                                    prev = atomicCAS(&key_of(h), kEmpty32, k0);
                                }
                                fresh = prev == kEmpty32;
                                atomicAdd(&acc0_of(h), acc0_of(sl));
                                acc0_of(sl) = 0;
                                if (kWords == 2) {
                                    atomicAdd(&acc1_of(h), acc1_of(sl));
                                    acc1_of(sl) = 0;
                                }
                                key_of(sl) = kMerged32;
                            }
                        }
                        const unsigned long long m = __ballot(fresh);
                        if (fresh && cnt + lanes_below(m) < kList) tlist[cnt + lanes_below(m)] = (unsigned short)h;
                        cnt += __popcll(m);
                        n_created += (unsigned)__popcll(m);
                        wave_lds_fence();
                    }
                }
                if (cnt > kList) {   // cannot happen (the bound above)
                    if (lane == 0) atomicOr(&args->b.ctl->error, 2);
                }
                const int n = min(cnt, kList);
                cnt = 0;
                // two rows of 64 entries at a time: their LDS and edge loads overlap
#pragma unroll 1
                for (int r = 0; r < n; r += 128) {
                    unsigned k[2];
                    unsigned sl[2];
                    unsigned long long m_done[2], m_keep[2], v0[2] = {}, v1[2] = {};
                    double v[2];
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        k[u] = kEmpty32;
                        sl[u] = 0;
                        m_keep[u] = __ballot(lane < n - r - 64 * u);
                        if (lane_of(m_keep[u])) sl[u] = tlist[r + 64 * u + lane];
                    }
#pragma unroll
                    for (int u = 0; u < 2; ++u)
                        if (lane_of(m_keep[u])) k[u] = key_of(sl[u]);
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        m_done[u] = __ballot(k[u] < bound) & m_keep[u];
                        if (bits_c != 0) {   // merged copies: cleared, not binned
                            const unsigned long long m_merged = __ballot(k[u] == kMerged32) & m_keep[u];
                            m_done[u] &= ~m_merged;
                            m_keep[u] &= ~m_merged;
                            n_retired += (unsigned)__popcll(m_merged);
                            if (lane_of(m_merged)) key_of(sl[u]) = kEmpty32;
                        }
                        m_keep[u] &= ~m_done[u];
                        n_retired += (unsigned)__popcll(m_done[u]);
                        // entries that stay: listed again from the front (already read)
                        if (lane_of(m_keep[u])) tlist[cnt + lanes_below(m_keep[u])] = (unsigned short)sl[u];
                        cnt += __popcll(m_keep[u]);
                        if (lane_of(m_done[u])) {
                            v0[u] = acc0_of(sl[u]);
                            key_of(sl[u]) = kEmpty32;
                            acc0_of(sl[u]) = 0;
                            if (kWords == 2) {
                                v1[u] = acc1_of(sl[u]);
                                acc1_of(sl[u]) = 0;
                            }
                        }
                    }
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        bal_out += Acc<MODE>::balance(v0[u], v1[u]);
                        if constexpr (MODE == ST_F32) v[u] = small_value(v0[u]);
                        else v[u] = Acc<MODE>::value(v0[u], v1[u]);
                    }
                    if (MODE == ST_F32 && __ballot(((unsigned)(v0[0] >> 32) | (unsigned)(v0[1] >> 32)) >= 1u << 20) != 0ull) {
                        // a sum of 2^20 or more, or a negative one
                        asm volatile("");   // (a branch: not both forms and a select)
#pragma unroll
                        for (int u = 0; u < 2; ++u) v[u] = Acc<MODE>::value(v0[u], v1[u]);
                    }
                    if (args->b.rec != nullptr) {
                        const RecArgs rc = load_uniform(args->b.rec);
#pragma unroll 1
                        for (int u = 0; u < 2; ++u) {
                            if (!lane_of(u ? m_done[1] : m_done[0])) continue;
                            const unsigned ku = u ? k[1] : k[0];
                            const unsigned long long pos = atomicAdd(&args->b.ctl->rec_count, 1ull);
                            if ((int64_t)pos < rc.cap) {   // test hook only; bit 62: a wave_kernel record
                                rc.seg[pos] = rare.seg | (1ll << 62);
                                rc.key[pos] = lattice_key(ex.kx0 + ((ku >> bits_c) & ((1u << (bits_x - bits_c)) - 1u)),
                                                          ex.ky0 + ((ku >> bits_x) & ((1u << (bits_xy - bits_x)) - 1u)),
                                                          ex.kz0 + (ku >> bits_xy), ex.N);
                                rc.sum[pos] = u ? v[1] : v[0];
                            }
                        }
                    }
#pragma unroll 1
                    for (int hh = 0; hh < args->b.n_hists; ++hh) bin_two(args, hh, v, m_done, lhist);
                }
                wave_lds_fence();
                if (last) return true;
                // The entries that stay keep their slots, except those whose
                // probe path may now have an empty slot.
                if (cnt <= 64) {
                    // all at once: those not in their home slot leave the
                    // table, then enter it again
                    if (lane < cnt) {
                        const unsigned sl = tlist[lane];
                        const unsigned k = key_of(sl);
                        unsigned to = home(k);
                        if (to != sl) {
                            const unsigned long long v0 = acc0_of(sl);
                            acc0_of(sl) = 0;
                            unsigned long long v1 = 0;
                            if (kWords == 2) {
                                v1 = acc1_of(sl);
                                acc1_of(sl) = 0;
                            }
                            key_of(sl) = kEmpty32;
#pragma unroll 1
                            while (atomicCAS(&key_of(to), kEmpty32, k) != kEmpty32) to = lattice_next<SLOTS>(to);
                            acc0_of(to) = v0;
                            if (kWords == 2) acc1_of(to) = v1;
                            tlist[lane] = (unsigned short)to;
                        }
                    }
                    wave_lds_fence();
                    return false;
                }
                // more than one row: entries move into empty slots on their
                // paths until none can (each move shortens a path, so this ends)
                bool moved = true;
#pragma unroll 1
                while (moved) {
                    moved = false;
#pragma unroll 1
                    for (int r = 0; r < cnt; r += 64) {
                        bool mv = false;
                        if (lane < cnt - r) {
                            const unsigned sl = tlist[r + lane];
                            const unsigned k = key_of(sl);
                            unsigned to = home(k);
#pragma unroll 1
                            while (to != sl) {
                                if (atomicCAS(&key_of(to), kEmpty32, k) == kEmpty32) {
                                    acc0_of(to) = acc0_of(sl);
                                    acc0_of(sl) = 0;
                                    if (kWords == 2) {
                                        acc1_of(to) = acc1_of(sl);
                                        acc1_of(sl) = 0;
                                    }
                                    key_of(sl) = kEmpty32;
                                    tlist[r + lane] = (unsigned short)to;
                                    mv = true;
                                    break;
                                }
                                to = lattice_next<SLOTS>(to);
                            }
                        }
                        moved |= __ballot(mv) != 0ull;
                        wave_lds_fence();
                    }
                }
                return false;
            };
            // the next row's points are loaded before the current ones are
            // scored, but after these are in lattice units relative to the box
            // corner (batch_kernel): the load's registers are free by then (2 nm
            // spheres, 256 tracks x 1000: 11.76 -> 11.59 ms against moving them)
            PointT ahead;
            fetch(ahead);
            row -= 64;
            bool last = false;
#pragma unroll 1
            while (!last) {
                row += 64;
                if ((row & (kBlk - 1)) == 0) new_block();
                Real qx, qy, qz;
                double w = (double)ahead.w;
                if constexpr (MODE == ST_F64) {
                    qx = fma(ahead.x, inv, bqx);
                    qy = fma(ahead.y, inv, bqy);
                    qz = fma(ahead.z, inv, bqz);
                } else {
                    qx = fmaf(ahead.x, inv, bqx);
                    qy = fmaf(ahead.y, inv, bqy);
                    qz = fmaf(ahead.z, inv, bqz);
                }
                if constexpr (MODE == ST_F32) w *= yscale;
                asm volatile("" : "+v"(qx), "+v"(qy), "+v"(qz), "+v"(w));
                fetch(ahead);
                last = step(qx, qy, qz, w);
            }
            if (lane == 0) {
                atomicAdd(&s_stats[2], (unsigned long long)n_in);
                atomicAdd(&s_stats[5], (unsigned long long)n_created);
                atomicAdd(&s_stats[6], (unsigned long long)n_retired);
            }
            unspilled += n_retired;
            n_in = n_created = n_retired = 0;
            if (a.hist_lds_words && unspilled > (1u << 27)) {
                // keep the workgroup's 32-bit counters far from overflow: each
                // wave adds at most 2^27 + one segment's entries between two
                // of its own spills
                for (int hh = 0; hh < a.n_hists; ++hh)
                    for (int b = lane; b < a.hist[hh].guess.nbins; b += 64) {
                        const unsigned v = atomicExch(&lhist[a.hist[hh].lds_offset + b], 0u);
                        if (v) atomicAdd(&a.hist[hh].bins[b], (unsigned long long)v);
                    }
                unspilled = 0;
            }
        }
    }
    {
        unsigned long long c[3] = {n_flagged, bal_in, bal_out};
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1)
#pragma unroll
            for (int k = 0; k < 3; ++k) c[k] += __shfl_xor(c[k], d, 64);
        if (lane == 0) {
            atomicAdd(&s_stats[1], c[0]);
            atomicAdd(&s_stats[3], c[1]);
            atomicAdd(&s_stats[4], c[2]);
        }
    }
    __syncthreads();
    if (wa.slab) {
        if (tid < kStats) wa.slab_stats[(size_t)blockIdx.x * kStats + tid] = s_stats[tid];
        for (int w = tid; w < a.hist_lds_words; w += blockDim.x)
            wa.slab[(size_t)blockIdx.x * a.hist_lds_words + w] = lhist[w];
        return;
    }
    if (tid < kStats) atomicAdd(&a.ctl->stats[tid], s_stats[tid]);
#pragma unroll
    for (int hh = 0; hh < kMaxHists; ++hh) {
        if (a.hist_lds_words == 0 || hh >= a.n_hists) break;
        for (int b = tid; b < a.hist[hh].guess.nbins; b += blockDim.x) {
            const unsigned v = lhist[a.hist[hh].lds_offset + b];
            if (v) atomicAdd(&a.hist[hh].bins[b], (unsigned long long)v);
        }
    }
}

// Adds the workgroups' histograms and statistics to the device counters: 16
// bins per workgroup, its 64 groups of 16 lanes over the slab's rows (the last
// workgroup: the statistics, and the report to the host).  Launched with
// slab_blocks(hist_lds_words) workgroups.  Bound by latency: 64 bins per
// workgroup, a wave a row, 10.8 us for 512 rows of 1000 bins; this 4.6 us.
constexpr int kSlabBins = 16;
__host__ __device__ inline int slab_blocks(int words) { return (words + kSlabBins - 1) / kSlabBins + 1; }

__global__ __launch_bounds__(1024) void slab_sum_kernel(WaveArgs wa, int rows)
{
    constexpr int kGroups = 1024 / kSlabBins;
    __shared__ unsigned long long s_sum[16][kSlabBins];
    const int lane = threadIdx.x % kSlabBins, group = threadIdx.x / kSlabBins;
    const int words = wa.b.hist_lds_words;
    const bool stats = blockIdx.x == gridDim.x - 1;
    const int w = (int)blockIdx.x * kSlabBins + lane;
    unsigned long long sum = 0;
    if (stats) {
        if (lane < kStats) {
#pragma unroll 4
            for (int r = group; r < rows; r += kGroups) sum += wa.slab_stats[(size_t)r * kStats + lane];
        }
    } else if (w < words) {
#pragma unroll 8
        for (int r = group; r < rows; r += kGroups) sum += wa.slab[(size_t)r * words + w];
    }
    // the groups of a wave, then the waves
#pragma unroll
    for (int d = 32; d >= kSlabBins; d >>= 1) sum += __shfl_xor(sum, d, 64);
    if ((threadIdx.x & 63) < kSlabBins) s_sum[threadIdx.x >> 6][lane] = sum;
    __syncthreads();
    if (threadIdx.x >= kSlabBins) return;
#pragma unroll
    for (int k = 1; k < 16; ++k) sum += s_sum[k][lane];
    if (stats) {
        // the last kernel of the pass: the control block is complete
        if (lane < kStats) {
            sum += wa.b.ctl->stats[lane];
            wa.b.ctl->stats[lane] = sum;
        }
        if (wa.report) {
            if (lane < kStats) wa.report->stats[lane] = sum;
            if (lane == kStats) wa.report->rec_count = wa.b.ctl->rec_count;
            if (lane == kStats + 1) wa.report->error = wa.b.ctl->error;
        }
        return;
    }
    if (sum == 0) return;
    for (int h = 0; h < wa.b.n_hists; ++h) {
        const int b = w - wa.b.hist[h].lds_offset;
        if (b >= 0 && b < wa.b.hist[h].guess.nbins) atomicAdd(&wa.b.hist[h].bins[b], sum);
    }
}

}  // namespace
}  // namespace st
