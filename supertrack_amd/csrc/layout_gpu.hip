// layout_gpu.hip -- device-side library layout (layout_gpu.hpp).
//
// Laying a library out is the larger part of a job on new tracks (18.5e6
// points, 100 oversamples: 336 of 340 ms on the host: a stable sort per track,
// two sliding windows, FP32 records).  Here the points go to the device as
// they come and everything else is done there; the upload then bounds it: 14.2 ms
// for the library, 12 of them the copy (24 tracks, 119e3 points: 1.76 -> 0.34 ms,
// of which 0.2 are the sort's launches).
//   * sort: a stable LSD radix sort of (z, index) over the whole run, 8 bits a
//     pass, then by track number: tile histograms, one scan workgroup per
//     digit, a ranking scatter (wave ballots), all without spinning;
//   * one workgroup per 256-point block gathers the sorted points and forms
//     the block's FP32 record, as fill_chunk does, with the same operations;
//   * the sliding-window bounds are only ever compared with a limit: a row of
//     64 windows passes if no window holds more points than the limit (one
//     load and compare per point), else if the row's joint bounding box holds
//     few enough cells, else window by window.
#include <algorithm>
#include <cmath>

#include "layout_gpu.hpp"
#include "st_common.hpp"
#include "transfer.hpp"

namespace st {
namespace {

constexpr int kMaxGeoms = 16;
constexpr int kThreads = 256;
// Rows of 256 keys a workgroup sorts: few of them where there are few tiles
// (125e3 points: 62 tiles of 8 rows, 244 of 2).
constexpr int kRowsMany = 8, kRowsFew = 2;
constexpr int64_t kFewPoints = (int64_t)1 << 19;
constexpr int kDigits = 256;

struct Geoms {
    st_geometry g[kMaxGeoms];
};

// Window tests a track asks for and failed (bits).
constexpr uint32_t kTestFast = 1u, kTestWave = 2u, kTestHot = 4u;

struct BlockSum {
    double xmin, xmax, ymin, ymax, esum, emax;
    int32_t finite, pad;
};

struct TrackTests {
    uint32_t asked;    // tests whose outcome the flags depend on
    uint32_t run;      // those that the track's own box does not already pass
    uint32_t failed;
    int32_t spans;
};

// ---------------------------------------------------------------------------
// keys
// ---------------------------------------------------------------------------
// Ascending order of doubles as unsigned integers; both zeros alike, NaN with
// +infinity (fill_chunk's order).
__device__ __forceinline__ unsigned long long z_key(double z)
{
    if (z != z) z = HUGE_VAL;
    if (z == 0.0) z = 0.0;
    const unsigned long long u = (unsigned long long)__double_as_longlong(z);
    return (u >> 63) ? ~u : u | 0x8000000000000000ull;
}

__global__ __launch_bounds__(kThreads) void block_track_kernel(const TrackDesc *tds, int64_t n_tracks, int64_t bbase,
                                                               int32_t *block_track)
{
    const int lane = threadIdx.x & 63;
    const int64_t wave = ((int64_t)blockIdx.x * kThreads + threadIdx.x) >> 6;
    const int64_t waves = ((int64_t)gridDim.x * kThreads) >> 6;
    for (int64_t t = wave; t < n_tracks; t += waves) {
        const int64_t b0 = tds[t].block0 - bbase;
        for (int b = lane; b < tds[t].nblocks; b += 64) block_track[b0 + b] = (int32_t)t;
    }
}

__global__ __launch_bounds__(kThreads) void keys_kernel(const TrackDesc *tds, const int32_t *block_track, int64_t pbase,
                                                        int64_t bbase, const double *z, unsigned long long *key,
                                                        uint32_t *index, uint32_t *track)
{
    const int64_t b = blockIdx.x;
    const int32_t t = block_track[b];
    const int64_t r = (b - (tds[t].block0 - bbase)) * kBlk + threadIdx.x;
    if (r >= tds[t].n) return;
    const int64_t i = tds[t].offset - pbase + r;
    key[i] = z_key(z[i]);
    index[i] = (uint32_t)i;
    track[i] = (uint32_t)t;
}

// ---------------------------------------------------------------------------
// radix sort pass
// ---------------------------------------------------------------------------
struct SortArgs {
    const unsigned long long *key;   // null: the digit comes from the point's track
    const uint32_t *index;
    const uint32_t *track;
    unsigned long long *key_out;
    uint32_t *index_out;
    uint32_t *counts;                // [kDigits][tiles]
    uint32_t *totals;                // [kDigits]
    int64_t n;
    int tiles;
    int shift;
};

__device__ __forceinline__ uint32_t digit_of(const SortArgs &a, unsigned long long key, uint32_t index)
{
    return a.key ? (uint32_t)(key >> a.shift) & 255u : (a.track[index] >> a.shift) & 255u;
}

template <int kRows>
__global__ __launch_bounds__(kThreads) void sort_count_kernel(SortArgs a)
{
    constexpr int kTile = kThreads * kRows;
    __shared__ uint32_t s_c[kDigits];
    const int tid = threadIdx.x;
    s_c[tid] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * kTile;
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        const int64_t i = base + r * kThreads + tid;
        if (i < a.n) atomicAdd(&s_c[digit_of(a, a.key ? a.key[i] : 0, a.key ? 0 : a.index[i])], 1u);
    }
    __syncthreads();
    a.counts[(size_t)tid * a.tiles + blockIdx.x] = s_c[tid];
}

// Workgroup d: exclusive scan of digit d's counts over the tiles, and its total.
__global__ __launch_bounds__(kThreads) void sort_scan_kernel(uint32_t *counts, uint32_t *totals, int tiles)
{
    __shared__ uint32_t s_w[kThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint32_t *row = counts + (size_t)blockIdx.x * tiles;
    uint32_t base = 0;
    for (int t0 = 0; t0 < tiles; t0 += kThreads) {
        const uint32_t c = t0 + tid < tiles ? row[t0 + tid] : 0u;
        uint32_t incl = c;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t v = __shfl_up(incl, d, 64);
            if (lane >= d) incl += v;
        }
        if (lane == 63) s_w[wave] = incl;
        __syncthreads();
        uint32_t before = base, all = 0;
        for (int w = 0; w < kThreads / 64; ++w) {
            before += w < wave ? s_w[w] : 0u;
            all += s_w[w];
        }
        if (t0 + tid < tiles) row[t0 + tid] = before + incl - c;
        base += all;
        __syncthreads();
    }
    if (tid == 0) totals[blockIdx.x] = base;
}

template <int kRows>
__global__ __launch_bounds__(kThreads) void sort_scatter_kernel(SortArgs a)
{
    constexpr int kTile = kThreads * kRows;
    __shared__ uint16_t s_cnt[kRows][kThreads / 64][kDigits];
    __shared__ uint32_t s_off[kDigits];
    __shared__ uint32_t s_w[kThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int i = tid; i < kRows * (kThreads / 64) * kDigits / 2; i += kThreads)
        reinterpret_cast<uint32_t *>(&s_cnt[0][0][0])[i] = 0;
    // start of digit tid's output: the totals of the digits below it, then this
    // tile's share
    {
        const uint32_t c = a.totals[tid];
        uint32_t incl = c;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t v = __shfl_up(incl, d, 64);
            if (lane >= d) incl += v;
        }
        if (lane == 63) s_w[wave] = incl;
        __syncthreads();
        uint32_t off = incl - c + a.counts[(size_t)tid * a.tiles + blockIdx.x];
        for (int w = 0; w < wave; ++w) off += s_w[w];
        s_off[tid] = off;
    }
    const int64_t base = (int64_t)blockIdx.x * kTile;
    unsigned long long key[kRows];
    uint32_t index[kRows], digit[kRows], rank[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        const int64_t i = base + r * kThreads + tid;
        key[r] = 0;
        index[r] = 0;
        digit[r] = 0;
        if (i < a.n) {
            index[r] = a.index[i];
            if (a.key) key[r] = a.key[i];
            digit[r] = digit_of(a, key[r], index[r]);
        }
    }
    const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        const bool valid = base + r * kThreads + tid < a.n;
        unsigned long long same = __ballot(valid);
#pragma unroll
        for (int bit = 0; bit < 8; ++bit) {
            const unsigned long long m = __ballot((digit[r] >> bit) & 1u);
            same &= ((digit[r] >> bit) & 1u) ? m : ~m;
        }
        rank[r] = (uint32_t)__popcll(same & below);
        if (valid && rank[r] == 0) s_cnt[r][wave][digit[r]] = (uint16_t)__popcll(same);
    }
    __syncthreads();
    uint32_t run = 0;
    for (int r = 0; r < kRows; ++r)
        for (int w = 0; w < kThreads / 64; ++w) {
            const uint32_t c = s_cnt[r][w][tid];
            s_cnt[r][w][tid] = (uint16_t)run;
            run += c;
        }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        if (base + r * kThreads + tid >= a.n) continue;
        const uint32_t pos = s_off[digit[r]] + s_cnt[r][wave][digit[r]] + rank[r];
        a.index_out[pos] = index[r];
        if (a.key) a.key_out[pos] = key[r];
    }
}

// ---------------------------------------------------------------------------
// blocks and tracks
// ---------------------------------------------------------------------------
template <typename Op>
__device__ __forceinline__ double block_reduce(double v, double *s, Op op)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v = op(v, __shfl_xor(v, d, 64));
    __syncthreads();
    if (lane == 0) s[wave] = v;
    __syncthreads();
    v = s[0];
    for (int w = 1; w < kThreads / 64; ++w) v = op(v, s[w]);
    return v;
}

struct BlockArgs {
    const TrackDesc *tds;
    const int32_t *block_track;
    const uint32_t *order;        // source of each sorted position
    const double *x, *y, *z, *e;  // the run's points as uploaded
    LayoutDst dst;
    BlockSum *sums;
    int64_t pbase, bbase;
    Geoms geoms;
};

__global__ __launch_bounds__(kThreads) void block_kernel(BlockArgs a)
{
    __shared__ double s[kThreads / 64];
    const int tid = threadIdx.x;
    const int64_t b = blockIdx.x;
    const TrackDesc td = a.tds[a.block_track[b]];
    const int64_t r = (b - (td.block0 - a.bbase)) * kBlk + tid;
    const bool act = r < td.n;
    const int64_t p = td.offset - a.pbase + r;
    double v[3] = {0.0, 0.0, 0.0}, e = 0.0;
    if (act) {
        const uint32_t src = a.order[p];
        v[0] = a.x[src];
        v[1] = a.y[src];
        v[2] = a.z[src];
        e = a.e[src];
        a.dst.x[p] = v[0];
        a.dst.y[p] = v[1];
        a.dst.z[p] = v[2];
        a.dst.e[p] = e;
        if (tid == 0) a.dst.zfirst[b] = v[2];
    }
    auto lower = [](double p1, double p2) { return fmin(p1, p2); };
    auto upper = [](double p1, double p2) { return fmax(p1, p2); };
    double lo[3], hi[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        lo[k] = block_reduce(act ? v[k] : HUGE_VAL, s, lower);
        hi[k] = block_reduce(act ? v[k] : -HUGE_VAL, s, upper);
    }
    const double esum = block_reduce(act ? fabs(e) : 0.0, s, [](double p1, double p2) { return p1 + p2; });
    const double emax = block_reduce(act ? fabs(e) : 0.0, s, upper);
    const bool fin = !act || (isfinite(v[0]) && isfinite(v[1]) && isfinite(v[2]) && isfinite(e));
    const int finite = __syncthreads_and(fin ? 1 : 0);
    if (tid == 0) a.sums[b] = BlockSum{lo[0], hi[0], lo[1], hi[1], esum, emax, finite, 0};
    if (!a.dst.p32) return;
    // the block's FP32 record (fill_chunk's operations)
    const st_geometry g = a.geoms.g[td.geom];
    double org[3], err = 0.0, extent = 0.0;
    float f[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        org[k] = (isfinite(lo[k]) && isfinite(hi[k])) ? 0.5 * (lo[k] + hi[k]) : 0.0;
        const double d = v[k] - org[k];
        f[k] = (float)d;
        const double e1 = fabs((double)f[k] - d) + fabs(d) * 2.3e-16;
        if (act) {
            err = isfinite(e1) ? fmax(err, e1) : HUGE_VAL;
            extent = fmax(extent, (double)fabsf(f[k]));
        }
    }
    if (act) a.dst.p32[p] = PointF32{f[0], f[1], f[2], (float)e};
    err = block_reduce(err, s, upper);
    extent = block_reduce(extent, s, upper);
    if (tid != 0) return;
    const double invD = 1.0 / g.diameter;
    BlockF32 bk;
    bk.oqx = (org[0] - g.gso) * invD;
    bk.oqy = (org[1] - g.gso) * invD;
    bk.oqz = ((org[2] + g.half_length) - g.gso) * invD;
    double dl = err + kTwoM44 * (fabs(org[0]) + fabs(org[1]) + fabs(org[2]) + 7.0 * g.half_length + fabs(g.gso) +
                                 g.diameter + 16.0);
    if (!isfinite(dl)) dl = HUGE_VAL;
    const double dlq = dl * invD;
    const double r2q = (g.radius * g.radius) / (g.diameter * g.diameter);
    bk.dl = dl;
    bk.fm = 0.5 - (dlq + 1e-12);
    bk.mrgq = 3.0 * dlq * (1.0 + 2.0 * dlq) + 1e-14 * r2q;
    sphere_thresholds(r2q, bk.fm, bk.mrgq, &bk.sure, &bk.maybe);
    single_terms(bk, extent * invD, g);
    a.dst.blocks[b] = bk;
}

// One wave per track: bounds and the window tests the track's flags need
// (fill_chunk's and wave_flags' rules).
__global__ __launch_bounds__(64) void track_kernel(TrackDesc *tds, const BlockSum *sums, const double *z, int64_t pbase,
                                                   int64_t bbase, int precision, Geoms geoms, TrackTests *tests)
{
    const int lane = threadIdx.x;
    TrackDesc &td = tds[blockIdx.x];
    double xmin = HUGE_VAL, xmax = -HUGE_VAL, ymin = HUGE_VAL, ymax = -HUGE_VAL, esum = 0.0, emax = 0.0;
    bool finite = true;
    for (int b = lane; b < td.nblocks; b += 64) {
        const BlockSum v = sums[td.block0 - bbase + b];
        xmin = fmin(xmin, v.xmin);
        xmax = fmax(xmax, v.xmax);
        ymin = fmin(ymin, v.ymin);
        ymax = fmax(ymax, v.ymax);
        esum += v.esum;
        emax = fmax(emax, v.emax);
        finite = finite && v.finite;
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        xmin = fmin(xmin, __shfl_xor(xmin, d, 64));
        xmax = fmax(xmax, __shfl_xor(xmax, d, 64));
        ymin = fmin(ymin, __shfl_xor(ymin, d, 64));
        ymax = fmax(ymax, __shfl_xor(ymax, d, 64));
        esum += __shfl_xor(esum, d, 64);
        emax = fmax(emax, __shfl_xor(emax, d, 64));
    }
    finite = __ballot(!finite) == 0ull;
    if (lane != 0) return;
    const int64_t n = td.n, o = td.offset - pbase;
    const st_geometry &g = geoms.g[td.geom];
    const double D = g.diameter, z0 = n ? z[o] : 0.0, z1 = n ? z[o + n - 1] : 0.0;
    td.xmin = xmin;
    td.xmax = xmax;
    td.ymin = ymin;
    td.ymax = ymax;
    td.zmax = z1;
    const double denom = (2. / 3.) * D;
    const double ylim = (precision == ST_F64) ? 2.7e11 : 1.0e9;
    const double ypoint = (precision == ST_F64) ? kMaxPointY64 : kMaxPointY32;
    bool fast = finite && n <= kMaxFastPoints && esum / denom < ylim && emax / denom < ypoint;
    const double nl = (double)g.n_linear;
    if (fast && n > 0) {
        const double cmax = fmax(fmax(fmax(fabs(xmin), fabs(xmax)), fmax(fabs(ymin), fabs(ymax))),
                                 fmax(fabs(z0 + g.half_length), fabs(z1 + g.half_length)));
        fast = (cmax + g.half_length + fabs(g.gso)) / D < 1073741824.0;
        const double cx = fmin(nl, floor((xmax - xmin) / D) + 6.0);
        const double cy = fmin(nl, floor((ymax - ymin) / D) + 6.0);
        fast = fast && cx * cy <= 4294967294.0;
    }
    TrackTests q{0u, 0u, 0u, 0};
    if (fast && n > 0) {
        q.asked = kTestFast;
        const double range[3] = {xmax - xmin, ymax - ymin, z1 - z0};
        int bits = 0;
        bool narrow = true;
        for (int k = 0; k < 3; ++k) {
            const double c = fmin(nl, floor(range[k] / D) + 6.0);
            int b = 1;
            while (ldexp(1.0, b) <= c) ++b;
            bits += b;
            narrow = narrow && b <= 24;
        }
        if (narrow && bits <= kWaveKeyBits) {
            q.asked |= kTestWave;
            if ((double)n * D >= 64.0 * (z1 - z0) && bits + 2 <= kWaveKeyBits) q.asked |= kTestHot;
        }
        const double wide = g.length - 4.0 * D;
        q.spans = xmax - xmin >= wide || ymax - ymin >= wide;
        // every window's box lies in the track's
        const double cells = (floor((xmax - xmin) / D) + 2.0) * (floor((ymax - ymin) / D) + 2.0);
        const double kept = cells * (q.spans ? 3.0 : 1.0);
        q.run = q.asked & ((cells * 3.0 > (double)kMaxWindow ? kTestFast : 0u) |
                           (kept > (double)kWaveWindow ? kTestWave : 0u) | (kept > (double)kHotWindow ? kTestHot : 0u));
    }
    td.flags = fast ? 0u : kFlagExact;
    td.wave = fast && n == 0 ? kFlagWave : 0u;
    tests[blockIdx.x] = q;
}

// Whether a z-window of width w starting at one of a row's points holds more
// than `limit` spheres, by window_bound's rule min(points, x-cells * y-cells *
// layers).  One wave; i0: the row's first point of the track's n.
__device__ bool row_exceeds(const double *x, const double *y, const double *z, int64_t n, int64_t i0, double D,
                            double w, int64_t layers, int64_t limit)
{
    const int lane = threadIdx.x & 63;
    const int64_t i = i0 + lane;
    const bool over = i + limit < n && z[i + limit] - z[i] <= w;   // more points than the limit
    unsigned long long todo = __ballot(over);
    if (todo == 0ull) return false;
    // first point beyond the window of point s, at or after `from`
    auto window_end = [&](int64_t s, int64_t from) {
        const double zs = z[s];
        int64_t lo = from, step = 64;
        while (lo < n) {   // steps of 64 points per lane-wide look, doubling
            const int64_t j = lo + (int64_t)lane * (step / 64);
            const unsigned long long out = __ballot(j >= n || !(z[j] - zs <= w));
            if (out != 0ull) {
                const int f = __ffsll((long long)out) - 1;
                const int64_t gap = step / 64;
                const int64_t hi = lo + (int64_t)f * gap;   // beyond the window (or the track)
                if (gap == 1) return hi < n ? hi : n;
                lo = f > 0 ? hi - gap + 1 : lo;
                if (f == 0) return lo;
                step = 64;   // the answer lies in (hi - gap, hi]
                continue;
            }
            lo += 63 * (step / 64) + 1;
            if (step < (int64_t)1 << 20) step *= 2;
        }
        return n;
    };
    auto cells = [&](int64_t s, int64_t end) {
        double xl = HUGE_VAL, xh = -HUGE_VAL, yl = HUGE_VAL, yh = -HUGE_VAL;
        for (int64_t j = s + lane; j < end; j += 64) {
            xl = fmin(xl, x[j]);
            xh = fmax(xh, x[j]);
            yl = fmin(yl, y[j]);
            yh = fmax(yh, y[j]);
        }
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) {
            xl = fmin(xl, __shfl_xor(xl, d, 64));
            xh = fmax(xh, __shfl_xor(xh, d, 64));
            yl = fmin(yl, __shfl_xor(yl, d, 64));
            yh = fmax(yh, __shfl_xor(yh, d, 64));
        }
        return (floor((xh - xl) / D) + 2.0) * (floor((yh - yl) / D) + 2.0) * (double)layers;
    };
    const int64_t first = i0 + __ffsll((long long)todo) - 1, last = i0 + 63 - __clzll((long long)todo);
    if (cells(first, window_end(last, last)) <= (double)limit) return false;
    int64_t end = first;
    while (todo != 0ull) {
        const int64_t s = i0 + __ffsll((long long)todo) - 1;
        todo &= todo - 1ull;
        end = window_end(s, end > s ? end : s);
        if (cells(s, end) > (double)limit) return true;   // (its points exceed the limit too)
    }
    return false;
}

__global__ __launch_bounds__(kThreads) void window_kernel(const TrackDesc *tds, const int32_t *block_track, LayoutDst d,
                                                          int64_t pbase, int64_t bbase, Geoms geoms, TrackTests *tests)
{
    const int64_t b = blockIdx.x;
    const int32_t t = block_track[b];
    const TrackDesc &td = tds[t];
    TrackTests &q = tests[t];
    const uint32_t run = q.run;
    if (run == 0u) return;
    const int64_t o = td.offset - pbase, n = td.n;
    const int64_t i0 = (b - (td.block0 - bbase)) * kBlk + (threadIdx.x & ~63);
    if (i0 >= n) return;
    const double D = geoms.g[td.geom].diameter;
    const double w1 = D * (1.0 + 1e-12) + 1e-9, w2 = 2.0 * D * (1.0 + 1e-12) + 1e-9;
    const bool spans = q.spans != 0;
    const struct {
        uint32_t bit;
        double w;
        int64_t layers, limit;
    } test[3] = {{kTestFast, w2, 3, kMaxWindow},
                 {kTestWave, spans ? w2 : w1, spans ? 3 : 1, kWaveWindow},
                 {kTestHot, spans ? w2 : w1, spans ? 3 : 1, kHotWindow}};
#pragma unroll   // (a table walked at run time would lie in scratch memory)
    for (const auto &c : test) {
        // (a test already failed by another row needs no more rows)
        if (!(run & c.bit) || (__hip_atomic_load(&q.failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & c.bit))
            continue;
        if (row_exceeds(d.x + o, d.y + o, d.z + o, n, i0, D, c.w, c.layers, c.limit) && (threadIdx.x & 63) == 0)
            atomicOr(&q.failed, c.bit);
    }
}

__global__ __launch_bounds__(kThreads) void flags_kernel(TrackDesc *tds, const TrackTests *tests, int64_t n_tracks)
{
    const int64_t t = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (t >= n_tracks) return;
    const TrackTests q = tests[t];
    const uint32_t passed = q.asked & ~q.failed;
    if (!(q.asked & kTestFast)) return;   // track_kernel's flags stand
    const bool fast = (passed & kTestFast) != 0;
    tds[t].flags = fast ? 0u : kFlagExact;
    tds[t].wave = fast && (passed & kTestWave) ? kFlagWave | ((passed & kTestHot) ? kFlagHot : 0u) : 0u;
}

// ST_F64: the fast-path tracks' energies become lineal energies (scored once
// per oversample, where a division is a dozen instructions: 256 tracks x 100,
// 10 nm spheres, 1.40 -> 1.34 ms).
__global__ __launch_bounds__(kThreads) void lineal_kernel(const TrackDesc *tds, const int32_t *block_track, double *e,
                                                          int64_t pbase, int64_t bbase, Geoms geoms)
{
    const int64_t b = blockIdx.x;
    const TrackDesc &td = tds[block_track[b]];
    const int64_t r = (b - (td.block0 - bbase)) * kBlk + threadIdx.x;
    if ((td.flags & kFlagExact) || r >= td.n) return;
    double &v = e[td.offset - pbase + r];
    v = lineal_energy(v, geoms.g[td.geom]);
}

}  // namespace

int layout_chunk_device(const double *x, const double *y, const double *z, const double *edep, int64_t n_points,
                        int64_t n_tracks, const st_geometry *geoms, int n_geoms, int precision, int64_t pbase,
                        int64_t bbase, int64_t nblocks, TrackDesc *tds, const LayoutDst &dst)
{
    if (n_points >= ((int64_t)1 << 31) || n_geoms > kMaxGeoms)
        return set_error(ST_ENOMEM, "device layout: run of %lld points", (long long)n_points);
    hipStream_t stream = default_stream();
    const size_t n = (size_t)n_points;
    const bool few = n_points <= kFewPoints;
    const int tile = kThreads * (few ? kRowsFew : kRowsMany);
    const int tiles = (int)((n_points + tile - 1) / tile);
    size_t bytes = 0;
    auto add = [&](size_t b) {
        const size_t at = bytes;
        bytes += (b + 255) / 256 * 256;
        return at;
    };
    const size_t at_raw = add(4 * n * sizeof(double));
    const size_t at_key[2] = {add(n * 8), add(n * 8)}, at_index[2] = {add(n * 4), add(n * 4)}, at_track = add(n * 4);
    const size_t at_counts = add((size_t)kDigits * tiles * 4), at_totals = add(kDigits * 4);
    const size_t at_bt = add((size_t)nblocks * 4), at_sums = add((size_t)nblocks * sizeof(BlockSum));
    const size_t at_tds = add((size_t)n_tracks * sizeof(TrackDesc)), at_tests = add((size_t)n_tracks * sizeof(TrackTests));
    struct Scratch {
        char *p = nullptr;
        ~Scratch() { (void)dev_free(p); }
    } scratch;
    if (dev_malloc((void **)&scratch.p, std::max<size_t>(bytes, 256)) != hipSuccess) {
        (void)hipGetLastError();
        scratch.p = nullptr;
        return set_error(ST_ENOMEM, "device layout: %zu B of scratch", bytes);
    }
    char *const s = scratch.p;
    double *raw = (double *)(s + at_raw);
    const double *src[4] = {x, y, z, edep};
    TrackDesc *tds_dev = (TrackDesc *)(s + at_tds);
    TrackTests *tests = (TrackTests *)(s + at_tests);
    int32_t *bt = (int32_t *)(s + at_bt);
    auto column = [&](int k) { return UploadPart{raw + k * n, src[k], n * sizeof(double)}; };
    if (n_tracks == 0) return ST_OK;
    Geoms gs{};
    std::copy(geoms, geoms + n_geoms, gs.g);
    if (nblocks == 0) {
        const UploadPart only{tds_dev, tds, n_tracks * sizeof(TrackDesc)};
        ST_HIP_TRY(upload(&only, 1));
    } else {
        // z first: the sort runs while the other columns are uploaded (25.3 ->
        // 21 ms for 18.5e6 points when the upload took 20 ms; it takes 12 now)
        const UploadPart first[2] = {column(2), {tds_dev, tds, n_tracks * sizeof(TrackDesc)}};
        ST_HIP_TRY(upload(first, 2));
        const int bt_grid = (int)std::min<int64_t>((n_tracks + 3) / 4, 4096);
        ST_HIP_TRY(launch(block_track_kernel, bt_grid, kThreads, 0, stream, tds_dev, n_tracks, bbase, bt));
        SortArgs a{};
        a.key = (unsigned long long *)(s + at_key[0]);
        a.index = (uint32_t *)(s + at_index[0]);
        a.track = (uint32_t *)(s + at_track);
        a.key_out = (unsigned long long *)(s + at_key[1]);
        a.index_out = (uint32_t *)(s + at_index[1]);
        a.counts = (uint32_t *)(s + at_counts);
        a.totals = (uint32_t *)(s + at_totals);
        a.n = n_points;
        a.tiles = tiles;
        ST_HIP_TRY(launch(keys_kernel, (unsigned)nblocks, kThreads, 0, stream, tds_dev, bt, pbase, bbase, raw + 2 * n,
                          (unsigned long long *)a.key, (uint32_t *)a.index, (uint32_t *)a.track));
        auto count = few ? sort_count_kernel<kRowsFew> : sort_count_kernel<kRowsMany>;
        auto scatter = few ? sort_scatter_kernel<kRowsFew> : sort_scatter_kernel<kRowsMany>;
        auto pass = [&](int shift) -> int {
            a.shift = shift;
            ST_HIP_TRY(launch(count, tiles, kThreads, 0, stream, a));
            ST_HIP_TRY(launch(sort_scan_kernel, kDigits, kThreads, 0, stream, a.counts, a.totals, tiles));
            ST_HIP_TRY(launch(scatter, tiles, kThreads, 0, stream, a));
            const uint32_t *i = a.index;
            a.index = a.index_out;
            a.index_out = (uint32_t *)i;
            const unsigned long long *k = a.key;
            if (k) {
                a.key = a.key_out;
                a.key_out = (unsigned long long *)k;
            }
            return ST_OK;
        };
        int rc = ST_OK;
        for (int shift = 0; shift < 64 && !rc; shift += 8) rc = pass(shift);
        a.key = nullptr;   // then by track
        for (int shift = 0; shift < 32 && (n_tracks - 1) >> shift && !rc; shift += 8) rc = pass(shift);
        if (rc) return rc;
        const UploadPart rest[3] = {column(0), column(1), column(3)};
        ST_HIP_TRY(upload(rest, 3));
        BlockArgs ba{};
        ba.tds = tds_dev;
        ba.block_track = bt;
        ba.order = a.index;
        ba.x = raw;
        ba.y = raw + n;
        ba.z = raw + 2 * n;
        ba.e = raw + 3 * n;
        ba.dst = dst;
        ba.sums = (BlockSum *)(s + at_sums);
        ba.pbase = pbase;
        ba.bbase = bbase;
        ba.geoms = gs;
        ST_HIP_TRY(launch(block_kernel, (unsigned)nblocks, kThreads, 0, stream, ba));
    }
    ST_HIP_TRY(launch(track_kernel, (unsigned)n_tracks, 64, 0, stream, tds_dev, (const BlockSum *)(s + at_sums), dst.z,
                      pbase, bbase, precision, gs, tests));
    if (nblocks > 0)
        ST_HIP_TRY(launch(window_kernel, (unsigned)nblocks, kThreads, 0, stream, tds_dev, bt, dst, pbase, bbase, gs,
                          tests));
    ST_HIP_TRY(launch(flags_kernel, (unsigned)((n_tracks + kThreads - 1) / kThreads), kThreads, 0, stream, tds_dev,
                      tests, n_tracks));
    if (precision == ST_F64 && nblocks > 0)
        ST_HIP_TRY(launch(lineal_kernel, (unsigned)nblocks, kThreads, 0, stream, tds_dev, bt, dst.e, pbase, bbase, gs));
    ST_HIP_TRY(hipMemcpyAsync(tds, tds_dev, n_tracks * sizeof(TrackDesc), hipMemcpyDeviceToHost, stream));
    ST_HIP_TRY(hipStreamSynchronize(stream));
    return ST_OK;
}

}  // namespace st
