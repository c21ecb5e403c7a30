"""Wide histograms in the batched form: on both sides of the widths at which
the one-wave kernel's workgroups stop counting in bins of their own, counts
equal the block kernel's."""
import numpy as np
import pytest

import supertrack_amd as st
from supertrack_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,diameter,least", [(st.ST_F64, 10.0, 5), (st.ST_F32, 10.0, 6), (st.ST_F64, 2.0, 4),
                                                      (st.ST_F32, 2.0, 4)])
def test_wide_histograms(precision, diameter, least):
    x, y, z, e, off = st.synth_library(dict(W.workload("cfg3")["synth"], n_max=30000), 20, 3)
    lib = st.TrackLibrary(x, y, z, e, off, [st.SphericalGeometry(2.5e3, diameter)], None, precision)
    private, fewest = set(), 24
    for nbins in (1000, 20000, 26000, 27000, 28000, 29000, 30000, 31000, 32000, 33000, 34000, 36000, 50000):
        got = []
        for kw in ({}, dict(table_slots=2048)):
            h = st.Histogram(nbins, 0.01, 300.0, "log")
            b = st.BatchRun(lib, [h], 5, 9, True, True, **kw)
            p = b.params()
            b.run()
            b.sync()
            got.append(h.fetch())
            b.free()
            h.free()
            if not kw:
                waves = p["block_threads"] // 64 * p["blocks_per_cu"]
                private.add(p["hist_copies"])
                fewest = min(fewest, waves)
                assert waves >= (least if p["hist_copies"] else 16), (nbins, p)
        np.testing.assert_array_equal(got[0], got[1])
        assert got[0].sum() > 1000
    assert private == {0, 1} and fewest <= least + 1
    lib.free()
