"""The batched form's exact per-segment tracks: those of up to 12288 points run
many oversamples per launch.  Counts equal the per-track loop's, on both sides
of that size, over more oversamples than one launch holds, with one and two
histograms."""
import numpy as np
import pytest

import supertrack_amd as st
from supertrack_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,n_os", [([3000], 1450), ([12288, 40, 12289], 6), ([1, 700, 20000], 9)])
@pytest.mark.parametrize("hists", [[("lin", 3000, 0.01, 300.0)], [("log", 1000, 1e-2, 1e3), ("lin", 500, 0.1, 50.0)]])
def test_exact_tracks_equal_the_per_track_loop(sizes, n_os, hists):
    spec = dict(W.workload("cfg2")["synth"])
    parts = [st.synth_library(dict(spec, n_min=n, n_max=n, stream_id=4), 1, k)[:4] for k, n in enumerate(sizes)]
    parts = [[v.copy() for v in p] for p in parts]
    for p in parts:
        p[0][len(p[0]) // 2] = np.nan   # a non-finite point: the exact path
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    x, y, z, e = (np.concatenate([p[a] for p in parts]) for a in range(4))
    g = st.SphericalGeometry(2.5e3, 10.0)
    lib = st.TrackLibrary(x, y, z, e, off, [g], None, st.ST_F64)
    assert lib.info()["exact_tracks"] == len(sizes)
    hs = [st.Histogram(nb, lo, hi, kind) for kind, nb, lo, hi in hists]
    b = st.BatchRun(lib, hs, n_os, 21, True, True)
    for _ in range(2):
        b.run()
        b.sync()
        got = [h.fetch() for h in hs]
    b.free()
    lib.free()
    for (kind, nb, lo, hi), c, h in zip(hists, got, hs):
        want = st.Histogram(nb, lo, hi, kind)
        st.run_plain(x, y, z, e, off, g, want, n_os, 21, True, True)
        np.testing.assert_array_equal(c.astype(np.float64), want.counts())
        want.free()
        h.free()
