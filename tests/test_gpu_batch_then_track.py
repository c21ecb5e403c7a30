"""A histogram used by a batch and then by the per-track path: a track begins
with zeroed counters, whether the batch's pass before it was launched or
replayed from its graph."""
import numpy as np
import pytest

import supertrack_amd as st
from supertrack_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_graph", [False, True])
@pytest.mark.parametrize("passes", [1, 2, 3])
def test_track_after_batch(use_graph, passes):
    w = W.workload("cfg2")
    x, y, z, e, off, _ = W.make_library(w, n_tracks=2)
    geom = st.SphericalGeometry(2.5e3, 10.0)
    h = st.Histogram(3000, 0.01, 300.0, "lin")

    def track():
        n = int(off[1])
        t, p = st.Track(x[:n], y[:n], z[:n], e[:n]), st.VolumeEdepPair(n)
        m = st.VoxelConstrainedSphereMethod(geom, True, True)
        h.cpu[:] = 0.0
        m.allocate_track_process(t, 5, 0, 3)
        h.allocate_track_process(p)
        for _ in range(3):
            m.process_track(t, p)
            h.sort_reduce_and_add_to_histogram(p)
        m.free_track_process()
        h.free_track_process()
        for o in (m, p, t):
            o.free()
        return h.counts()

    want = track()
    lib = st.TrackLibrary(x, y, z, e, off, [geom], None, st.ST_F32)
    b = st.BatchRun(lib, [h], 10, 5, True, True, use_graph=use_graph)
    for _ in range(passes):
        h.fetch(reset=True)
        b.run()
    b.sync()
    np.testing.assert_array_equal(track(), want)
    assert want.sum() > 0
    for o in (b, lib, h):
        o.free()
