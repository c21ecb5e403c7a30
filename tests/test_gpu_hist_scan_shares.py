"""The sort-free histogram where one workgroup's share holds more spheres than
its table (2048): it is split over 16 more hash values, and a part that still
exceeds the list (960 pairs) is summed sphere by sphere in key order.  Keys are
made from chosen hash values, so that they all fall in one share."""
import numpy as np
import pytest

import supertrack_amd as st
from test_gpu_hist_scan import _check

pytestmark = pytest.mark.gpu

MULTIPLIER = 0x9E3779B97F4A7C15
INVERSE = pow(MULTIPLIER, -1, 1 << 64)


def _part_bits(capacity):
    b = 2
    while b < 8 and (capacity >> b) > 128:
        b += 1
    return b


def _keys(rng, n, capacity, part, sub=None):
    """n distinct keys of workgroup `part` (and of its 16th `sub`)."""
    bits = _part_bits(capacity)
    low = rng.choice(1 << 24, n, replace=False).astype(object) * (1 << 20) + 12345
    top = [part * 16 + (sub if sub is not None else k % 16) for k in range(n)]
    hashes = [(t << (60 - bits)) | int(v) for t, v in zip(top, low)]
    assert all(h >> (64 - bits) == part for h in hashes)
    keys = np.array([h * INVERSE % (1 << 64) for h in hashes], np.uint64)
    assert len(np.unique(keys)) == n
    return keys


# (capacities up to 8192 pairs are read ahead by another form of the kernel)
@pytest.mark.parametrize("capacity,spheres", [(8192, 2500), (12000, 2500), (1 << 18, 3000)])
@pytest.mark.parametrize("sub", [None, 5])
def test_more_spheres_than_the_table(capacity, spheres, sub):
    rng = np.random.default_rng(capacity + spheres)
    bits = _part_bits(capacity)
    names = _keys(rng, spheres, capacity, (1 << bits) - 2, sub)
    which = np.concatenate([rng.permutation(spheres), rng.integers(0, spheres, capacity // 2 - spheres)
                            if capacity // 2 > spheres and capacity < 20000 else rng.integers(0, spheres, 2000)])
    rng.shuffle(which)
    _check(names[which], rng.lognormal(0.3, 0.8, len(which)), capacity)


@pytest.mark.parametrize("capacity", [8192, 12000, 1 << 18])
@pytest.mark.parametrize("before,run", [(960, 960), (960, 961), (1024, 1024), (700, 4000)])
def test_one_sphere_fills_whole_steps(capacity, before, run):
    """Among more spheres than the table holds, one with a run of consecutive
    pairs as long as a step over the pairs (and begun with it), or longer."""
    rng = np.random.default_rng(run)
    bits = _part_bits(capacity)
    names = _keys(rng, 2200, capacity, 1, 3)
    other = _keys(rng, 300, capacity, 2 % (1 << bits))
    keys = np.concatenate([names[:before], np.full(run, names[1000]), names[before:], other, names[::3]])
    keys = keys[:capacity]
    ys = rng.lognormal(-4.0, 2.0, len(keys))
    ys[::31] = -ys[::31]
    _check(keys, ys, capacity)
    _check(keys[::-1].copy(), ys, capacity, 1000, "log")
