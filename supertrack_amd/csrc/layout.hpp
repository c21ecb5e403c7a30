// layout.hpp -- host-side layout of a batched track library: per-track
// records, each track's points sorted by z, per-block search keys and, for
// FP32 storage, block-relative FP32 points with per-block error bounds, and
// each track's eligibility for the fused kernel.  Plain C++ (no HIP): used by
// batch.hip to build the device library and by the CPU tests on its own.
#pragma once

#include <cmath>
#include <cstdint>
#include <vector>

#include "../../include/supertrack_amd.h"

namespace st {

constexpr int kBlk = 256;                              // points per library block
constexpr int64_t kMaxWindow = 768;                    // fast-path bound on spheres in a z-window two diameters wide
constexpr int64_t kMaxFastPoints = (int64_t)1 << 22;   // fast-path bound on points per track
constexpr uint32_t kFlagExact = 1u;                    // TrackDesc::flags: the exact per-segment path
constexpr uint32_t kFlagWave = 1u;                     // TrackDesc::wave: fits the one-wave kernel
constexpr uint32_t kFlagHot = 2u;                      // TrackDesc::wave: few spheres take most of a row of points
constexpr int kHotCopies = 4;                          // table entries per sphere of a kFlagHot track
constexpr int64_t kHotWindow = 24;                     // kFlagHot: bound on the spheres a flush keeps
constexpr int64_t kWaveWindow = 224;                   // one-wave kernel: bound on the spheres a flush keeps
constexpr int kWaveKeyBits = 31;                       // one-wave kernel: bits of its sphere keys
constexpr double kTwoM44 = 1.0 / 17592186044416.0;
// Per-point lineal energy limits of the fused kernel (its fixed-point
// conversions are exact only under 2^51): ST_F32 y * 2^32, ST_F64 y * 2^24.
constexpr double kMaxPointY32 = 262144.0;      // 2^18
constexpr double kMaxPointY64 = 67108864.0;    // 2^26

struct TrackDesc {
    int64_t offset;     // first point in the sorted arrays
    int64_t block0;     // first block in the block arrays
    int32_t n;
    int32_t nblocks;
    int32_t geom;
    uint32_t flags;
    uint32_t wave;      // one-wave kernel: kFlagWave, kFlagHot
    uint32_t pad;
    double xmin, xmax, ymin, ymax, zmax;
};

// ST_F32 block record (128 B, read through the scalar cache).  The fast path
// works in lattice units: q = (coordinate - gso) / D, so rint(q) is the
// sphere index and q - rint(q) the offset from the sphere centre; the voxel
// faces are the half-way planes q = -1/2 and q = N - 1/2, so a point that is
// not within dl of a half-way plane is inside the voxel iff every rint(q)
// lies in [0, N - 1].
//   oq*     (origin - gso) / D of the block's FP32 offsets (z with H' added);
//   dl      bound on |approximate - reference| of any shifted, offset
//           coordinate of the block in nm (FP32 rounding of the offsets plus,
//           with a wide margin, FP64 rounding of every step, any |shift| <= H');
//   fm      |q - rint(q)| >= fm: within dl of a half-way plane;
//   mrgq    |sum (rint(q) - q)^2 - r^2 / D^2| <= mrgq: within the error of
//           the squared distance;
//   sure,   squared distances (lattice units) below which a point is inside
//   maybe   its sphere and above which it is outside, whichever way a nearby
//           half-way plane is decided (sphere_thresholds);
//   k*, f*  oq* as its nearest integer and the rest, and
//   *32     the thresholds for a point brought to lattice units in FP32
//           (single_terms).
struct BlockF32 {
    double oqx, oqy, oqz, dl, fm, mrgq, sure, maybe;
    int32_t kx, ky, kz;
    float fx, fy, fz;
    float sure32, maybe32;
    float pad[8];
};

// Squared-distance thresholds of a geometry (r2q = r^2 / D^2) from fm and mrgq
// as above.  A coordinate within dl of a half-way plane has |q - rint(q)| >= fm,
// so its squared distance is at least fm^2: below min(r2q - mrgq, fm^2) no
// index is in doubt and the point is inside.  Rounding such a coordinate the
// other way changes the squared distance by at most 2 (1/2 - fm) per axis, so
// above r2q + mrgq + 8 (1/2 - fm) the point is outside.
#ifdef __HIPCC__
__host__ __device__
#endif
inline void sphere_thresholds(double r2q, double fm, double mrgq, double *sure, double *maybe)
{
    const double f2 = fm > 0.0 ? fm * fm : 0.0;
    *sure = r2q - mrgq < f2 ? r2q - mrgq : f2;
    *maybe = r2q + mrgq + 8.0 * (0.5 - fm);
}

// The FP32 terms of a block record whose other terms are set.  extent: the
// largest |FP32 offset| / D of the block.  A coordinate is then
// fma(offset, 1 / D, f + f') lattice units from sphere k + k' (f', k': the same
// of the segment's shift), off by at most dl / D, the rounding of 1 / D and of
// the fma (2^-24 of extent, and of extent + 1) and of f, f' and their sum
// (2^-24); the squared distance, at most 3/4, rounds three times.  Where the
// bounds mean nothing every point is in doubt.
#ifdef __HIPCC__
__host__ __device__
#endif
inline void single_terms(BlockF32 &bk, double extent, const st_geometry &g)
{
    const double ulp = 5.9604644775390625e-08;   // 2^-24
    const double k[3] = {rint(bk.oqx), rint(bk.oqy), rint(bk.oqz)};
    bk.kx = bk.ky = bk.kz = 0;
    bk.fx = bk.fy = bk.fz = 0.0f;
    bk.sure32 = -1.0f;
    bk.maybe32 = HUGE_VALF;
    for (float &v : bk.pad) v = 0.0f;
    if (!(extent < 65536.0 && fabs(k[0]) < 1073741824.0 && fabs(k[1]) < 1073741824.0 && fabs(k[2]) < 1073741824.0))
        return;
    bk.kx = (int32_t)k[0];
    bk.ky = (int32_t)k[1];
    bk.kz = (int32_t)k[2];
    bk.fx = (float)(bk.oqx - k[0]);
    bk.fy = (float)(bk.oqy - k[1]);
    bk.fz = (float)(bk.oqz - k[2]);
    const double e = bk.dl / g.diameter + ulp * (2.0 * extent + 2.0) * (1.0 + 1e-6);
    if (!(e < 0.25)) return;
    const double fm = 0.5 - (e + 8.0 * ulp);   // (8 ulp: the rounding of the squares compared with fm^2)
    double sure, maybe;
    sphere_thresholds((g.radius * g.radius) / (g.diameter * g.diameter), fm, 3.0 * e * (1.0 + 2.0 * e) + 4.0 * ulp,
                      &sure, &maybe);
    bk.sure32 = (float)(sure - ulp);
    bk.maybe32 = (float)(maybe + 2.0 * ulp);
}

// A deposit's lineal energy.  ST_F64 libraries hold it in place of the energy
// for their fast-path tracks.
#ifdef __HIPCC__
__host__ __device__
#endif
inline double lineal_energy(double edep, const st_geometry &g)
{
    return edep / ((2. / 3.) * g.diameter);
}

// One FP32 point: offsets from its block's origin (nm) and the energy (eV);
// the same 16-byte layout as HIP's float4, which the kernel loads.
struct PointF32 {
    float x, y, z, w;
};

// Host staging of one appended run of tracks, indexed from the run's first
// point and block.
struct ChunkLayout {
    std::vector<double> x, y, z, e;   // z-sorted FP64 points
    std::vector<double> zfirst;       // z of each block's first point
    std::vector<PointF32> p32;        // ST_F32 only
    std::vector<BlockF32> blocks;     // ST_F32 only
};

// Fills the records of n_tracks tracks (offsets[0..n_tracks] index the
// caller's arrays) placed from library point pbase and block bbase: offset,
// n, block range, geometry (geom_of_track may be NULL: 0).  Returns the
// number of blocks the tracks take.
int64_t plan_chunk(const int64_t *offsets, int64_t n_tracks, const int32_t *geom_of_track, int64_t pbase,
                   int64_t bbase, TrackDesc *tds);

// Sorts each planned track's points by z (stable; NaN last) into out, and
// completes its record: x/y bounds, last z, and the fast-path eligibility
// (finite data, at most kMaxFastPoints points, fixed-point headroom, indices
// below 2^30 for any shift, at most 2^32 - 2 spheres in one layer of the
// track's x/y extent, at most kMaxWindow spheres in any z-window two
// diameters wide), and whether the one-wave kernel takes it (kFlagWave: a
// fast-path track whose flushes keep at most kWaveWindow spheres and whose
// key box fits kWaveKeyBits).  ST_F32 also gets the FP32 points and block
// records.
void fill_chunk(const double *x, const double *y, const double *z, const double *edep, const int64_t *offsets,
                int64_t n_tracks, const st_geometry *geoms, int precision, int64_t pbase, int64_t bbase,
                int64_t nblocks, TrackDesc *tds, ChunkLayout &out);

// The flags of a fast-path track (z-sorted points) for the one-wave kernel: 0,
// kFlagWave, or kFlagWave | kFlagHot (at least 64 points per layer of spheres
// on average, and so few spheres in reach that each may take kHotCopies table
// entries, one per group of lanes).  window: window_bound of a window two
// diameters wide and three layers, if known (else -1).
uint32_t wave_flags(const double *x, const double *y, const double *z, int64_t n, const st_geometry &g, double xmin,
                    double xmax, double ymin, double ymax, int64_t window = -1);

// Largest number of distinct spheres that the points of any z-window of
// width w can touch, for any shift: min(points, x-cells * y-cells * layers).
int64_t window_bound(const double *x, const double *y, const double *z, int64_t n, double D, double w,
                     int64_t layers);

}  // namespace st
