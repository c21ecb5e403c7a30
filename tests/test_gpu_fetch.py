"""Counts fetched by the device itself (histograms of up to 8192 bins) and by
a copy (longer ones): the same counts as the host's search finds, kept or
cleared as asked, again after every add."""
import numpy as np
import pytest

import supertrack_amd as st

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbins", [1, 255, 257, 8191, 8192, 8193])
def test_fetch_and_clear_around_the_slot_size(nbins):
    n = 5000
    rng = np.random.default_rng(nbins)
    h = st.Histogram(nbins, 0.0, 100.0, "lin")
    edges = h.edges
    lineal = rng.uniform(0.0, 100.0, n)
    # (every pair has its own sphere: each lineal energy is one count)
    want = np.histogram(lineal[(lineal >= edges[0]) & (lineal < edges[-1])], bins=edges)[0].astype(np.uint64)
    pairs = st.VolumeEdepPair(n)
    pairs.upload(np.arange(1, n + 1, dtype=np.uint64), lineal)
    h.allocate_track_process(pairs)
    for times in (1, 2):
        h.sort_reduce_and_add_to_histogram(pairs)
        assert np.array_equal(h.fetch(reset=False), times * want)
    assert np.array_equal(h.fetch(reset=True), 2 * want)
    assert not h.fetch(reset=False).any()
    h.sort_reduce_and_add_to_histogram(pairs)
    h.free_track_process()   # added to the host's bins, cleared behind
    assert np.array_equal(h.counts(), want.astype(np.int64))
    assert not h.fetch(reset=False).any()
