"""The library layout computed on the device against the host's (which runs
when the device's scratch cannot be allocated): the same tracks on each path,
the same points in the same order, so the same counts, point statistics
(which depend on the FP32 records' error bounds) and energy words."""
import ctypes as C

import numpy as np
import pytest

import supertrack_amd as st
from supertrack_amd import workloads as W

pytestmark = pytest.mark.gpu

HISTS = [("log", 1000, 1e-2, 1e3), ("lin", 3000, 0.01, 300.0)]


def _scan(points, geoms, gt, precision, host, n_os=3, shift_z=True):
    x, y, z, e, off = points
    if host:   # x, y, z, e, block starts, (points, blocks,) tables, then the scratch
        st.call("st_debug_fail_allocation", C.c_int64(9 if precision == st.ST_F32 else 7))
    try:
        lib = st.TrackLibrary(x, y, z, e, off, geoms, gt, precision)
    finally:
        st.call("st_debug_fail_allocation", C.c_int64(0))
    hs = [st.Histogram(nb, lo, hi, kind) for kind, nb, lo, hi in HISTS]
    out = []
    for kw in ({}, dict(table_slots=2048)):
        b = st.BatchRun(lib, hs, n_os, 3, True, shift_z, **kw)
        b.run()
        b.sync()
        out.append((b.stats(), b.balance()["energy_in"], [h.fetch() for h in hs]))
        b.free()
    info = lib.info()
    for h in hs:
        h.free()
    lib.free()
    return info, out


def _same(a, b):
    assert a[0] == b[0]
    for (s0, e0, c0), (s1, e1, c1) in zip(a[1], b[1]):
        assert s0 == s1 and e0 == e1
        for p, q in zip(c0, c1):
            np.testing.assert_array_equal(p, q)


@pytest.mark.parametrize("precision", [st.ST_F64, st.ST_F32])
@pytest.mark.parametrize("sizes", [[1], [255, 256, 257, 0, 1, 2047, 2048, 2049], [70000, 3, 0, 999], [40] * 300])
def test_device_layout_equals_host(precision, sizes):
    """Tracks with tied, negative, zero (both signs) and out-of-order z, runs
    beyond one sort tile, more than 256 tracks (two passes by track)."""
    rng = np.random.default_rng(len(sizes) + sizes[0])
    n = sum(sizes)
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    x, y = rng.normal(0, 60, n), rng.normal(50, 60, n)
    z = rng.uniform(-5000, 200, n)
    z[rng.random(n) < 0.2] = np.round(z[rng.random(n) < 0.2].mean())   # ties
    z[::7] = 0.0
    z[::14] = -0.0
    e = rng.uniform(1, 500, n)
    geoms = [st.SphericalGeometry(2.5e3, 10.0), st.SphericalGeometry(5e3, 100.0), st.SphericalGeometry(1e3, 1.0)]
    gt = (np.arange(len(sizes)) % 3).astype(np.int32)
    pts = (x, y, z, e, off)
    _same(_scan(pts, geoms, gt, precision, False), _scan(pts, geoms, gt, precision, True))


@pytest.mark.parametrize("precision", [st.ST_F64, st.ST_F32])
def test_device_layout_decides_every_path_like_host(precision):
    """Tracks on each side of the window bounds: synthetic tracks of rising
    density, sheets of each width, crowded columns, non-finite points and
    energies beyond the fixed-point headroom."""
    rng = np.random.default_rng(5)
    spec = dict(W.workload("cfg3")["synth"])
    parts = []
    for k, n in enumerate([2000, 20000, 120000, 300000]):
        parts.append(st.synth_library(dict(spec, n_min=n, n_max=n, stream_id=9), 1, k)[:4])
    for width in (20, 60, 95, 150, 400, 2400):   # sheets: spheres per layer rising through every limit
        m = 6000
        parts.append((rng.uniform(-width, width, m), rng.uniform(-width, width, m), rng.uniform(-2600, -2400, m),
                      rng.uniform(1, 100, m)))
    parts.append((np.full(9000, 3.0), np.full(9000, -7.0), rng.uniform(-2510, -2490, 9000), np.full(9000, 20.0)))
    for bad in (np.nan, np.inf):
        q = [v.copy() for v in parts[0]]
        q[2][17] = bad
        parts.append(q)
    q = [v.copy() for v in parts[0]]
    q[3][5] = 1e13
    parts.append(q)
    off = np.concatenate([[0], np.cumsum([len(p[0]) for p in parts])]).astype(np.int64)
    pts = (*(np.concatenate([p[a] for p in parts]) for a in range(4)), off)
    for hd in ((2.5e3, 10.0), (2.5e3, 2.0), (5e3, 100.0)):
        geoms = [st.SphericalGeometry(*hd)]
        a = _scan(pts, geoms, None, precision, False, 2)
        assert a[0]["exact_tracks"] >= 3
        _same(a, _scan(pts, geoms, None, precision, True, 2))
