"""Libraries of which the one-wave kernel takes some tracks only: short passes
are left to the block kernel altogether, long ones are shared by the two, and
both give the same counts as either forced."""
import ctypes as C

import numpy as np
import pytest

import supertrack_amd as st
from supertrack_amd import _capi
from supertrack_amd import workloads as W

pytestmark = pytest.mark.gpu

ONE_WAVE = 416
HISTS = [("log", 1000, 1e-2, 1e3), ("lin", 3000, 0.01, 300.0)]


def _library(precision):
    spec = dict(W.workload("cfg4")["synth"])
    parts = [st.synth_library(dict(spec, n_min=n, n_max=n, p_cluster=0.6, p_cluster_max=0.6), 1, k)[:4]
             for k, n in enumerate([120000, 400000, 900, 4000, 60000, 300000, 15000, 2500])]
    off = np.concatenate([[0], np.cumsum([len(p[0]) for p in parts])]).astype(np.int64)
    return st.TrackLibrary(*(np.concatenate([p[a] for p in parts]) for a in range(4)), off,
                           [st.SphericalGeometry(2.5e3, 5.0)], None, precision)


def _pass(lib, n_os, **kw):
    hs = [st.Histogram(nb, lo, hi, kind) for kind, nb, lo, hi in HISTS]
    b = st.BatchRun(lib, hs, n_os, 5, True, True, **kw)
    for _ in range(2):
        b.run()
        b.sync()
    s, shape, energy = b.stats(), b.params(), b.balance()["energy_in"]
    counts = [h.fetch() for h in hs]
    b.free()
    for h in hs:
        h.free()
    return shape["table_slots"] == ONE_WAVE, (s["points_scored"], s["points_in_sphere"], energy), counts


def _static(lib, n_os):
    hs = [st.Histogram(nb, lo, hi, kind) for kind, nb, lo, hi in HISTS]
    o = _capi.BatchOpts()
    o.n_oversamples, o.shift_xy, o.shift_z, o.seed = n_os, 1, 1, 5
    for _ in range(2):
        st.call("st_batch_run_static", lib.h, C.byref(o), (C.c_void_p * 2)(*[h.h for h in hs]), 2, None, None)
    st.synchronize()
    counts = [h.fetch() for h in hs]
    for h in hs:
        h.free()
    return counts


@pytest.mark.parametrize("precision", [st.ST_F64, st.ST_F32])
def test_short_and_long_passes(precision):
    lib = _library(precision)
    assert lib.info()["exact_tracks"] == 0
    seen = []
    for n_os in (1, 20, 3000):
        wave, *default = _pass(lib, n_os)
        seen.append(wave)
        assert _pass(lib, n_os, table_slots=ONE_WAVE)[0]
        for other in (_pass(lib, n_os, table_slots=ONE_WAVE)[1:], _pass(lib, n_os, table_slots=1536)[1:]):
            assert other[0] == default[0]
            for a, b in zip(other[1], default[1]):
                np.testing.assert_array_equal(a, b)
        for a, b in zip(_static(lib, n_os), default[1]):
            np.testing.assert_array_equal(a, b)
        assert default[1][0].sum() > 0
    assert seen == [False, False, True]
    assert _pass(lib, 3, autotune=True)[2][0].sum() > 0
    lib.free()
