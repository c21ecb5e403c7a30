"""An error that a call has reported is over: calls that launch kernels do not
report it again, nor an error of the caller's own HIP calls on the thread."""
import ctypes as C

import numpy as np
import pytest

import supertrack_amd as st
from supertrack_amd import _capi
from supertrack_amd import workloads as W

pytestmark = pytest.mark.gpu


def _leave_out_of_memory():
    p = C.c_void_p()
    assert st.lib().st_malloc(C.byref(p), C.c_size_t(1 << 50)) == -2   # ST_ENOMEM


def _leave_callers_own():
    hip = C.CDLL("libamdhip64.so")
    assert hip.hipMemcpy(None, np.zeros(1).ctypes.data_as(C.c_void_p), C.c_size_t(8), 1) != 0


@pytest.mark.parametrize("leave", [_leave_out_of_memory, _leave_callers_own])
def test_calls_after_a_reported_error(leave):
    w = W.workload("cfg3")
    x, y, z, e, off = st.synth_library(dict(w["synth"], n_max=20000), 3, 0)
    geoms = [st.SphericalGeometry(2.5e3, 10.0)]
    n = int(off[1])
    points = [v[:n] for v in (x, y, z, e)]

    def on_each_step(steps):
        out = []
        for step in steps:
            leave()
            out.append(step())
        return out

    # one track, step by step: a scoring launch, the sort-free and the radix histogram
    got = []
    for capacity in (n, (1 << 18) + 1):
        for queued in (False, True):
            leave()
            trk = st.Track(*points)
            leave()
            pairs = st.VolumeEdepPair(capacity)
            leave()
            h = st.Histogram(3000, 0.01, 300.0, "lin")
            leave()
            m = st.VoxelConstrainedSphereMethod(geoms[0], True, True)
            m.set_queued(queued)
            on_each_step([lambda: m.allocate_track_process(trk, 5, 0, 2), lambda: h.allocate_track_process(pairs),
                          lambda: m.process_track(trk, pairs), lambda: h.sort_reduce_and_add_to_histogram(pairs),
                          lambda: m.process_track(trk, pairs), lambda: h.sort_reduce_and_add_to_histogram(pairs),
                          m.free_track_process, lambda: h.fetch(reset=False), h.free_track_process,
                          lambda: h.fetch(reset=True)])
            got.append(h.counts())
            for o in (m, h, pairs, trk):
                o.free()
    for c in got[1:]:
        np.testing.assert_array_equal(c, got[0])
    assert got[0].sum() > 0
    # a copy, a library, a batch and the allocation-free pass
    leave()
    d = st.DeviceArray.from_numpy(x)
    leave()
    assert np.array_equal(d.to_numpy(np.float64, len(x)), x)
    d.free()
    for precision in (st.ST_F64, st.ST_F32):
        leave()
        lib = st.TrackLibrary(x, y, z, e, off, geoms, None, precision)
        h = st.Histogram(1000, 1e-2, 1e3, "log")
        for kw in (dict(use_graph=False), dict(use_graph=True), dict(table_slots=2048)):
            leave()
            b = st.BatchRun(lib, [h], 3, 5, True, True, **kw)
            _, _, counts = on_each_step([b.run, b.sync, h.fetch])
            assert counts.sum() > 0
            b.free()
        o = _capi.BatchOpts()
        o.n_oversamples, o.shift_xy, o.shift_z, o.seed = 3, 1, 1, 5
        stats = np.zeros(7, np.int64)
        leave()
        st.call("st_batch_run_static", lib.h, C.byref(o), (C.c_void_p * 1)(h.h), 1, None,
                stats.ctypes.data_as(_capi.c_int64_p))
        leave()
        np.testing.assert_array_equal(h.fetch(), counts)
        h.free()
        lib.free()
