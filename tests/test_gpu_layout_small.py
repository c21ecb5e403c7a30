"""Libraries of a few small tracks, laid out on the host, on both sides of the
sizes where the device takes over: counts equal the oracle's, and a library of
the same tracks appended to others is laid out as the whole is."""
import numpy as np
import pytest

import pyoracle as po
import supertrack_amd as st
from supertrack_amd import workloads as W

pytestmark = pytest.mark.gpu

KIND, NB, LO, HI = "log", 1000, 1e-2, 1e3


def _tracks(sizes):
    parts = []
    for k, n in enumerate(sizes):
        if n == 0:
            parts.append([np.zeros(0)] * 4)
            continue
        spec = dict(W.workload("cfg2")["synth"], n_min=n, n_max=n, stream_id=77)
        parts.append([np.asarray(v) for v in st.synth_library(spec, 1, k)[:4]])
    off = np.concatenate([[0], np.cumsum([len(p[0]) for p in parts])]).astype(np.int64)
    return (*(np.concatenate([np.zeros(0), *(p[a] for p in parts)]) for a in range(4)), off)


@pytest.mark.parametrize("precision", [st.ST_F64, st.ST_F32])
@pytest.mark.parametrize("sizes", [[], [0], [1], [0, 1, 0, 2], [1024], [1025], [256, 256, 256, 256], [256, 256, 256, 257],
                                   [200] * 4, [200] * 5, [64, 63, 300, 65]])
def test_few_small_tracks(precision, sizes):
    x, y, z, e, off = _tracks(sizes)
    g = po.geometry(2.5e3, 10.0)
    edges = po.edges(KIND, LO, HI, NB)
    n_os = 40
    want = np.zeros(NB, np.uint64)
    if len(x):
        want = po.run(x, y, z, e, off, [g], None, n_os, 5, True, True, [edges])[0][0]
    geoms = [st.SphericalGeometry(2.5e3, 10.0)]

    def counts(lib):
        h = st.Histogram(NB, LO, HI, KIND)
        b = st.BatchRun(lib, [h], n_os, 5, True, True)
        b.run()
        b.sync()
        out = h.fetch(), b.stats(), b.balance()["energy_in"]
        for o in (b, h, lib):
            o.free()
        return out

    whole, *rest = counts(st.TrackLibrary(x, y, z, e, off, geoms, None, precision))
    np.testing.assert_array_equal(whole, want)
    chunks = [(x, y, z, e, off[k:k + 2], None) for k in range(len(sizes))]   # one append a track
    parts, *rest2 = counts(st.TrackLibrary.streamed(len(sizes), len(x), chunks, geoms, precision))
    np.testing.assert_array_equal(parts, want)
    assert rest == rest2
