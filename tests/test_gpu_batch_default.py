"""The default launch (the one-wave kernel) where the older tests name a shape
of the block kernel: passes repeat bit for bit and equal the block kernel's, on
small libraries and on the full-size one, and beyond the number of entries at
which a wave moves the workgroup's counts to the device counters early."""
import numpy as np
import pytest

import supertrack_amd as st
from supertrack_amd import workloads as W

pytestmark = pytest.mark.gpu


def _pass(lib, hists, n_os, seed=W.SEED, **kw):
    hs = [st.Histogram(nb, lo, hi, kind) for kind, nb, lo, hi in hists]
    b = st.BatchRun(lib, hs, n_os, seed, True, True, **kw)
    shape = b.params()
    print(f"{n_os} oversamples, {shape}", flush=True)
    b.run()
    b.sync()
    bal = b.balance()
    assert bal["energy_in"] == bal["energy_out"] and bal["entries_created"] == bal["entries_retired"], bal
    out = [h.fetch() for h in hs], b.stats(), bal, shape
    b.free()
    for h in hs:
        h.free()
    return out


def _same(results):
    """(The points decided anew in FP64 are each kernel's own: their bounds differ.)"""
    c0, s0, k0, p0 = results[0]
    for c, s, k, p in results[1:]:
        for a, b in zip(c0, c):
            np.testing.assert_array_equal(a, b)
        if (p["table_slots"] == ONE_WAVE) != (p0["table_slots"] == ONE_WAVE):
            s = dict(s, fp64_rechecks=s0["fp64_rechecks"])
        assert s == s0
        assert k["energy_in"] == k0["energy_in"]
    assert sum(int(a.sum()) for a in c0) > 1000


ONE_WAVE = 416


@pytest.mark.parametrize("precision", [st.ST_F64, st.ST_F32])
@pytest.mark.parametrize("half_length,diameter", [(2.5e3, 10.0), (2.5e3, 2.0), (5e3, 100.0)])
def test_default_is_deterministic_and_equals_named_shapes(precision, half_length, diameter):
    x, y, z, e, off = st.synth_library(dict(W.workload("cfg3")["synth"], n_max=100000, voxel_half_length=half_length,
                                            entry_half_length=half_length), 24, 50)
    lib = st.TrackLibrary(x, y, z, e, off, [st.SphericalGeometry(half_length, diameter)], None, precision)
    hists = [("log", 1000, 1e-2, 1e3), ("lin", 3000, 0.01, 300.0)]
    default = [_pass(lib, hists, 8, use_graph=graph) for graph in (True, True, False, False)]
    assert default[0][3]["table_slots"] == ONE_WAVE
    named = [_pass(lib, hists, 8, table_slots=slots, blocks_per_cu=bpc, points_per_thread=ppt)
             for slots, bpc, ppt in ((1536, 5, 1), (2048, 2, 2))]
    _same(default + named + [_pass(lib, hists, 8, autotune=True)])
    lib.free()


def test_full_size_library_default():
    """4096 tracks, 5.98e8 points, 1000 oversamples, 2 nm spheres: the default
    twice, and the block kernel's own default shape."""
    w = W.workload("cfg4")
    x, y, z, e, off, _ = W.make_library(w)
    print(f"library of {int(off[-1])} points", flush=True)
    lib = st.TrackLibrary(x, y, z, e, off, W.geometries(w), None, st.ST_F32)
    del x, y, z, e
    n_os = w["n_oversamples"]
    results = [_pass(lib, w["hists"], n_os) for _ in range(2)]
    assert results[0][3]["table_slots"] == ONE_WAVE
    _same(results + [_pass(lib, w["hists"], n_os, table_slots=1280, blocks_per_cu=7, points_per_thread=1)])
    lib.free()
    counts, stats, bal, _ = results[0]
    total = sum(int(a.sum()) for a in counts)
    assert total <= bal["entries_retired"] <= stats["points_in_sphere"] <= stats["points_scored"] <= int(off[-1]) * n_os


def test_counts_moved_early():
    """More than 2^27 retired entries per wave (6144 waves): the waves move the
    workgroup's counts to the device counters in mid-pass."""
    spec = dict(W.workload("cfg4")["synth"], n_min=20000, n_max=20000)
    x, y, z, e, off = st.synth_library(spec, 256, 0)
    lib = st.TrackLibrary(x, y, z, e, off, [st.SphericalGeometry(2.5e3, 2.0)], None, st.ST_F32)
    hists = [("log", 1000, 1e-2, 1e3)]
    probe = _pass(lib, hists, 2000)
    waves = 256 * probe[3]["blocks_per_cu"] * (probe[3]["block_threads"] // 64)
    n_os = int(1.15 * (1 << 27) * waves / probe[2]["entries_retired"] * 2000)
    results = [_pass(lib, hists, n_os), _pass(lib, hists, n_os, table_slots=1280, blocks_per_cu=7, points_per_thread=1)]
    assert results[0][3]["table_slots"] == ONE_WAVE
    assert results[0][2]["entries_retired"] > waves << 27
    _same(results)
    lib.free()
