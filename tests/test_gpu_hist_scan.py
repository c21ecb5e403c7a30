"""Histogram of pairs without a sort (capacities up to 2^18 pairs): bins equal
the oracle's at the edges of its paths -- pairs read before the count is known
(capacity 8192), keys held in registers (28672 pairs) or read twice, lists of
more than 1024 pairs per workgroup, spheres with thousands of pairs."""
import numpy as np
import pytest

import pyoracle as po
import supertrack_amd as st

pytestmark = pytest.mark.gpu


def _bins(nb, lo, hi, keys, ys, capacity, kind="lin"):
    h = st.Histogram(nb, lo, hi, kind)
    p = st.VolumeEdepPair(capacity)
    p.upload(keys, ys)
    h.allocate_track_process(p)
    h.sort_reduce_and_add_to_histogram(p)
    h.free_track_process()
    got = h.counts()
    p.free()
    h.free()
    return got


def _check(keys, ys, capacity, nb=3000, kind="lin"):
    _, sums = po.reduce_pairs(keys, ys)
    edges = po.edges(kind, 0.01, 300.0, nb)
    want = np.zeros(nb)
    b = np.searchsorted(edges, sums, side="right") - 1
    np.add.at(want, b[(sums >= edges[0]) & (sums < edges[-1])], 1.0)
    np.testing.assert_array_equal(_bins(nb, 0.01, 300.0, keys, ys, capacity, kind), want)


@pytest.mark.parametrize("m,capacity", [(1, 1), (63, 64), (1024, 1025), (4900, 8191), (8192, 8192), (5000, 8193),
                                        (28672, 30000), (28673, 30000), (16384, 40000), (90001, 1 << 18),
                                        (1 << 18, 1 << 18), (70000, (1 << 18) + 1)])
@pytest.mark.parametrize("spread", [1 << 40, 3000])
def test_scan_matches_oracle(m, capacity, spread):
    rng = np.random.default_rng(m + spread % 97)
    keys = rng.integers(0, spread, m).astype(np.uint64)
    ys = rng.lognormal(0.3, 0.8, m)
    _check(keys, ys, capacity, 3000 if m % 2 else 5000)
    _check(keys, ys, capacity, 1000, "log")


@pytest.mark.parametrize("m,capacity", [(8000, 8192), (20000, 30000), (60000, 100000)])
def test_scan_few_spheres_with_many_pairs(m, capacity):
    """All pairs in one sphere; in a handful, among many small ones; the
    largest key value among them."""
    rng = np.random.default_rng(m)
    ys = rng.uniform(1e-6, 1e-3, m)
    _check(np.full(m, 77, np.uint64), ys, capacity)
    keys = rng.integers(0, 1 << 30, m).astype(np.uint64)
    keys[rng.random(m) < 0.3] = 5
    keys[rng.random(m) < 0.3] = 123456789
    keys[::50] = np.uint64(0xFFFFFFFFFFFFFFFF)
    _check(keys, ys, capacity)


@pytest.mark.parametrize("m,capacity", [(8192, 8192), (14336, 30000), (14337, 30000), (90000, 1 << 18)])
@pytest.mark.parametrize("spheres", [3, 40, 500])
def test_scan_sums_carried_from_list_to_list(m, capacity, spheres):
    """Shares of many lists: spheres that come back in every list and ones that
    leave, of very uneven sizes."""
    rng = np.random.default_rng(m + spheres)
    which = (rng.random(m) ** 4 * spheres).astype(np.int64)
    which = (which + np.arange(m) * spheres // (2 * m)) % spheres
    names = rng.integers(0, 1 << 40, spheres).astype(np.uint64)
    names[0] = np.uint64(0xFFFFFFFFFFFFFFFF)
    ys = rng.lognormal(-6.0, 3.0, m)
    ys[::97] = -ys[::97]
    _check(names[which], ys, capacity)
