"""The launch shape that st_batch_params reports, of a tuned batch or of the
defaults, can be passed to another batch and to the allocation-free pass."""
import ctypes as C

import numpy as np
import pytest

import supertrack_amd as st
from supertrack_amd import _capi
from supertrack_amd import workloads as W

pytestmark = pytest.mark.gpu

ST_EINVAL = -1
HISTS = {"log": [("log", 1000, 1e-2, 1e3)], "wide": [("lin", 100000, 0.01, 300.0)]}


def _run(lib, hists, **kw):
    hs = [st.Histogram(nb, lo, hi, kind) for kind, nb, lo, hi in hists]
    b = st.BatchRun(lib, hs, 6, 77, True, True, **kw)
    b.run()
    b.sync()
    out = b.params(), b.stats(), [h.fetch() for h in hs]
    b.free()
    for h in hs:
        h.free()
    return out


def _static(lib, hists, shape):
    hs = [st.Histogram(nb, lo, hi, kind) for kind, nb, lo, hi in hists]
    o = _capi.BatchOpts()
    o.n_oversamples, o.shift_xy, o.shift_z, o.seed = 6, 1, 1, 77
    for k, v in shape.items():
        setattr(o, k, v)
    stats = np.zeros(7, np.int64)
    rc = st.lib().st_batch_run_static(lib.h, C.byref(o), (C.c_void_p * len(hs))(*[h.h for h in hs]), len(hs), None,
                                      stats.ctypes.data_as(_capi.c_int64_p))
    out = rc, int(stats[2]), [h.fetch() for h in hs]
    for h in hs:
        h.free()
    return out


@pytest.mark.parametrize("precision", [st.ST_F64, st.ST_F32])
@pytest.mark.parametrize("hists", ["log", "wide"])
@pytest.mark.parametrize("first", [dict(), dict(autotune=True), dict(table_slots=2048)])
def test_shape_handed_on(precision, hists, first):
    spec = dict(W.workload("cfg3")["synth"], n_max=60000)
    x, y, z, e, off = st.synth_library(spec, 12, 0)
    lib = st.TrackLibrary(x, y, z, e, off, [st.SphericalGeometry(2.5e3, 10.0)], None, precision)
    shape, stats, want = _run(lib, HISTS[hists], **first)
    again, stats2, got = _run(lib, HISTS[hists], **shape)
    assert again == shape and stats2 == stats
    rc, in_sphere, static = _static(lib, HISTS[hists], shape)
    assert rc == 0 and in_sphere == stats["points_in_sphere"]
    for a, b, c in zip(want, got, static):
        np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(a, c)
    assert want[0].sum() > 100
    if shape["table_slots"] < 1280:   # the one-wave kernel
        few, stats3, got = _run(lib, HISTS[hists], **dict(shape, blocks_per_cu=1))
        assert few["blocks_per_cu"] == 1 and stats3 == stats
        np.testing.assert_array_equal(got[0], want[0])
        for bad in (dict(points_per_thread=2), dict(hist_copies=2), dict(table_slots=shape["table_slots"] + 1)):
            with pytest.raises(st.SuperTrackError):
                _run(lib, HISTS[hists], **dict(shape, **bad))
            assert _static(lib, HISTS[hists], dict(shape, **bad))[0] == ST_EINVAL
    lib.free()
