"""The one-wave batched kernel (the default launch) at the sizes where it can
go wrong: rows of 64 and blocks of 256 points with remainders, segments cut
into parts, tracks whose points crowd into few spheres, oversample groups."""
import numpy as np
import pytest

import pyoracle as po
import supertrack_amd as st
from supertrack_amd import workloads as W
from test_gpu_batch import check_bins, compare_records, gpu_run, oracle_segments

pytestmark = pytest.mark.gpu

HIST = [("log", 1000, 1e-2, 1e3)]


def _tracks(sizes, half_length, seed, length=None):
    """Primaries with clusters, cut or repeated to the sizes asked for."""
    spec = dict(W.workload("cfg2")["synth"], voxel_half_length=half_length, entry_half_length=half_length)
    parts = []
    for k, n in enumerate(sizes):
        if n == 0:
            parts.append([np.zeros(0)] * 4)
            continue
        x, y, z, e, _ = st.synth_library(dict(spec, n_min=n, n_max=n, stream_id=seed), 1, k)
        if length:   # squeeze along z: many points per layer of spheres
            z = -2 * half_length + (z - z.min()) * length / max(z.max() - z.min(), 1.0)
        parts.append([x, y, z, e])
    off = np.concatenate([[0], np.cumsum([len(p[0]) for p in parts])]).astype(np.int64)
    return (*(np.concatenate([p[a] for p in parts]) for a in range(4)), off)


@pytest.mark.parametrize("precision,rtol", [(st.ST_F64, 1e-12), (st.ST_F32, 1e-6)])
@pytest.mark.parametrize("half_length,diameter,length", [(2.5e3, 10.0, None), (2.5e3, 2.0, None),
                                                         (5e3, 100.0, 600.0)])
def test_wave_rows_and_blocks(precision, rtol, half_length, diameter, length):
    sizes = [1, 63, 64, 65, 0, 127, 128, 129, 255, 256, 257, 511, 513, 1000, 4097]
    x, y, z, e, off = _tracks(sizes, half_length, 31, length)
    n_os = 7
    g = po.geometry(half_length, diameter)
    oracle = oracle_segments(x, y, z, e, off, [g], None, n_os, 5, True, True)
    counts, rec, info, edges = gpu_run(x, y, z, e, off, [(half_length, diameter)], None, n_os, 5, True, True, precision,
                                       HIST, record=200000)
    assert info["exact_tracks"] == 0
    compare_records(rec, oracle, rtol)
    check_bins(counts, edges, oracle, rtol)


@pytest.mark.parametrize("precision", [st.ST_F64, st.ST_F32])
@pytest.mark.parametrize("half_length,diameter,length,n_os", [(2.5e3, 10.0, None, 3), (1e3, 1.0, None, 2),
                                                              (5e3, 100.0, 900.0, 3), (5e3, 100.0, None, 40)])
def test_wave_parts_equal_the_block_kernel(precision, half_length, diameter, length, n_os):
    """One large track among small ones: its segments are cut into parts at
    layers.  Counts, point statistics and the energy word equal the block
    kernel's, which scores whole segments."""
    sizes = [150001, 3000, 700, 90, 20011, 5, 1300, 64, 2222]
    x, y, z, e, off = _tracks(sizes, half_length, 77, length)
    lib = st.TrackLibrary(x, y, z, e, off, [st.SphericalGeometry(half_length, diameter)], None, precision)
    results = []
    for kw in ({}, dict(table_slots=1536)):
        hs = [st.Histogram(nb, lo, hi, kind) for kind, nb, lo, hi in HIST + [("lin", 3000, 0.01, 300.0)]]
        b = st.BatchRun(lib, hs, n_os, 9, True, True, **kw)
        for _ in range(2):   # the second pass: queues and slabs are cleared
            b.run()
            b.sync()
        s = b.stats()
        results.append(([h.fetch() for h in hs], s["points_scored"], s["points_in_sphere"], b.balance()["energy_in"]))
        b.free()
        for h in hs:
            h.free()
    lib.free()
    (c0, *r0), (c1, *r1) = results
    assert r0 == r1
    for a, b in zip(c0, c1):
        np.testing.assert_array_equal(a, b)
    assert int(c0[0].sum()) > 0
