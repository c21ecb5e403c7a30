"""A batch on a stream of its own: what its first pass needs is queued on the
stream the pass runs on, so it neither waits for other work on the default
stream nor runs before its work queues are built, and a batch moved while a
pass is under way ends that pass first."""
import ctypes as C

import numpy as np
import pytest

import supertrack_amd as st
from supertrack_amd import workloads as W

pytestmark = pytest.mark.gpu

HISTS = [("log", 1000, 1e-2, 1e3)]
NON_BLOCKING = 1


@pytest.fixture()
def streams():
    hip = C.CDLL("libamdhip64.so")
    made = []
    for _ in range(2):
        s = C.c_void_p()
        assert hip.hipStreamCreateWithFlags(C.byref(s), NON_BLOCKING) == 0
        made.append(s)
    yield made
    for s in made:
        assert hip.hipStreamSynchronize(s) == 0
        assert hip.hipStreamDestroy(s) == 0


def _library(n_tracks, precision, t0=0, broad=False, n_max=60000):
    x, y, z, e, off = st.synth_library(dict(W.workload("cfg3")["synth"], n_max=n_max), n_tracks, t0)
    if broad:   # the last track: a sheet across the voxel (exact path)
        n = int(off[-1] - off[-2])
        rng = np.random.default_rng(n)
        x[off[-2]:], y[off[-2]:] = rng.uniform(-2.5e3, 2.5e3, n), rng.uniform(-2.5e3, 2.5e3, n)
        z[off[-2]:] = rng.uniform(-2520.0, -2480.0, n)
    return st.TrackLibrary(x, y, z, e, off, [st.SphericalGeometry(2.5e3, 10.0)], None, precision)


def _hists():
    return [st.Histogram(nb, lo, hi, kind) for kind, nb, lo, hi in HISTS]


@pytest.mark.parametrize("use_graph", [False, True])
@pytest.mark.parametrize("kw", [{}, dict(table_slots=2048)])
def test_batch_made_while_the_default_stream_is_busy(streams, use_graph, kw):
    big = _library(64, st.ST_F32, n_max=600000)
    small = _library(9, st.ST_F32, 100, broad=True)
    assert small.info()["exact_tracks"] == 1
    href, hbig = _hists(), _hists()
    ref = st.BatchRun(small, href, 5, 11, True, True, **kw)
    ref.run()
    ref.sync()
    want, stats, energy = href[0].fetch(), ref.stats(), ref.balance()["energy_in"]
    ref.free()   # (its blocks, with what it wrote there, are taken again below)
    long = st.BatchRun(big, hbig, 2000, 3, True, True)
    for k in range(4):
        long.run()
        h = _hists()
        b = st.BatchRun(small, h, 5, 11, True, True, use_graph=use_graph, **kw)
        assert b.stats()["points_scored"] == 0 if k == 0 else True
        st.call("st_batch_set_stream", b.h, streams[k % 2])
        b.run()
        b.sync()
        np.testing.assert_array_equal(h[0].fetch(), want)
        assert b.stats() == stats and b.balance()["energy_in"] == energy
        b.free()
        h[0].free()
    long.sync()
    for o in (long, *href, *hbig, big, small):
        o.free()


@pytest.mark.parametrize("precision", [st.ST_F64, st.ST_F32])
@pytest.mark.parametrize("use_graph", [False, True])
def test_batch_moved_during_a_pass(streams, precision, use_graph):
    lib = _library(24, precision, broad=True, n_max=200000)
    hs = _hists()
    b = st.BatchRun(lib, hs, 20, 7, True, True, use_graph=use_graph)
    b.run()
    b.sync()
    want, stats = hs[0].fetch(), b.stats()
    assert want.sum() > 0
    for s in (streams[0], streams[1], None, streams[0]):
        b.run()
        st.call("st_batch_set_stream", b.h, s)
        b.run()
        b.sync()
        np.testing.assert_array_equal(hs[0].fetch(), 2 * want)
        assert b.stats() == stats
    # given back with a pass on the stream before
    b.run()
    st.call("st_batch_set_stream", b.h, streams[1])
    b.free()
    st.synchronize()
    np.testing.assert_array_equal(hs[0].fetch(), want)
    hs[0].free()
    lib.free()
