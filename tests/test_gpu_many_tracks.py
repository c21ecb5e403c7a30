"""Libraries of very many tracks: more blocks of points and more tracks than one
grid of the device layout may have (2^24 workgroups of 256 threads, 2^26 of 64),
appended in one call."""
import numpy as np
import pytest

import supertrack_amd as st

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [st.ST_F64, st.ST_F32])
def test_more_tracks_than_a_grid_of_blocks(precision):
    """2^24 + 5 tracks of one point at a sphere's centre, some empty ones among
    them; without shifts every point is one sphere."""
    n = (1 << 24) + 5
    g = st.SphericalGeometry(2.5e3, 10.0)
    rng = np.random.default_rng(2)
    cell = rng.integers(0, g.n_linear, (3, n), dtype=np.int32)
    x, y, z = (g.gso + c * g.diameter for c in cell)
    z -= g.half_length                       # (the track's z is taken from the voxel's centre)
    values = np.array([20.0, 95.0, 400.0])
    pick = rng.integers(0, 3, n)
    off = np.arange(n + 1, dtype=np.int64)
    off = np.insert(off, [5, 1 << 22, n], [5, 1 << 22, n])   # empty tracks
    print(f"library of {len(off) - 1} tracks", flush=True)
    lib = st.TrackLibrary(x, y, z, values[pick], off, [g], None, precision)
    assert lib.info()["fast_tracks"] == n + 3
    h = st.Histogram(1000, 0.01, 300.0, "lin")
    b = st.BatchRun(lib, [h], 1, 1, False, False)
    print("pass", flush=True)
    b.run()
    b.sync()
    counts = h.fetch()
    want = np.zeros(1000, np.uint64)
    bins = np.searchsorted(h.edges, values / ((2.0 / 3.0) * g.diameter), side="right") - 1
    np.add.at(want, bins, np.bincount(pick, minlength=3).astype(np.uint64))
    np.testing.assert_array_equal(counts, want)
    assert b.stats()["points_in_sphere"] == n
    for o in (b, h, lib):
        o.free()
