"""Scoring kernels of several methods at once, each on its own stream and
thread: their workgroups wait for lower tiles of their own track only, whichever
of them the device has room for, and each method's pairs equal those it leaves
alone on the device."""
import ctypes as C
import threading

import numpy as np
import pytest

import pyoracle as po
import supertrack_amd as st
from supertrack_amd import workloads as W

pytestmark = pytest.mark.gpu

N_OS = 12


def _score(points, track_index, stream):
    trk = st.Track(*points)
    pairs = st.VolumeEdepPair(len(points[0]))
    m = st.VoxelConstrainedSphereMethod(st.SphericalGeometry(2.5e3, 2.0), True, True)
    if stream is not None:
        m.set_stream(stream)
    out = []
    m.allocate_track_process(trk, W.SEED, track_index, N_OS)
    for k in range(N_OS):
        m.process_track(trk, pairs)
        if k % 4 == 3:   # (kernels follow one another without a wait in between)
            out.append(pairs.download())
    m.free_track_process()
    for o in (m, pairs, trk):
        o.free()
    return out


# 1024-point tiles: one, a few, the most that one pass over the CUs takes, more
@pytest.mark.parametrize("n", [700, 5000, 261000, 263000])
def test_methods_on_streams_at_once(n):
    spec = dict(W.workload("cfg2")["synth"], n_min=n, n_max=n)
    workers = 6
    tracks = [st.synth_library(dict(spec, stream_id=40 + k), 1, k)[:4] for k in range(workers)]
    want = [_score(tracks[k], k, None) for k in range(workers)]
    g = po.geometry(2.5e3, 2.0)
    oracle = po.track_segments(*tracks[0], g, W.SEED, 0, N_OS, True, True)
    for (keys, ys), (wk, wy, _, _) in zip(want[0], oracle[3::4]):
        np.testing.assert_array_equal(keys, wk)
        np.testing.assert_array_equal(ys, wy)
    hip = C.CDLL("libamdhip64.so")
    streams, got, errs = [], [None] * workers, []
    for _ in range(workers):
        s = C.c_void_p()
        assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0
        streams.append(s)

    def work(k):
        try:
            got[k] = _score(tracks[k], k, streams[k])
        except Exception as ex:   # reported by the main thread
            errs.append(ex)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(workers)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errs, errs
    for a, b in zip(got, want):
        for (ka, ya), (kb, yb) in zip(a, b):
            np.testing.assert_array_equal(ka, kb)
            np.testing.assert_array_equal(ya, yb)
    for s in streams:
        assert hip.hipStreamDestroy(s) == 0
