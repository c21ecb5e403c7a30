// layout_gpu.hpp -- the library layout of layout.hpp computed on the device.
#pragma once

#include "layout.hpp"
#include "st_internal.hpp"

namespace st {

// Where a run of tracks goes: the library's device arrays (already offset to
// the run's first point and block); p32 and blocks null in ST_F64.
struct LayoutDst {
    double *x, *y, *z, *e;
    PointF32 *p32;
    double *zfirst;
    BlockF32 *blocks;
};

// plan_chunk's tracks (tds, host) laid out as fill_chunk does: uploads the
// run's points in their own order, sorts each track by z (stable; NaN last)
// and fills dst and the records' bounds and flags on the device.  Returns
// ST_ENOMEM if its scratch (64 B per point) cannot be allocated; the caller
// then lays the run out on the host.  At most 2^23 blocks and tracks (a
// workgroup for each).  Waits for the device.
int layout_chunk_device(const double *x, const double *y, const double *z, const double *edep, int64_t n_points,
                        int64_t n_tracks, const st_geometry *geoms, int n_geoms, int precision, int64_t pbase,
                        int64_t bbase, int64_t nblocks, TrackDesc *tds, const LayoutDst &dst);

}  // namespace st
