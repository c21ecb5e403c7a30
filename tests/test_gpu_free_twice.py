"""Device memory given back twice is refused, as hipFree refuses it, and is not
handed out to two takers afterwards; an address inside a block gives the block
back."""
import ctypes as C

import numpy as np
import pytest

import supertrack_amd as st
from supertrack_amd import _capi

pytestmark = pytest.mark.gpu

ST_EHIP = -3


def _malloc(nbytes):
    p = C.c_void_p()
    st.call("st_malloc", C.byref(p), C.c_size_t(nbytes))
    return p


def _holds(blocks, nbytes):
    """Every block keeps its own bytes: no two overlap."""
    for k, p in enumerate(blocks):
        st.call("st_memset", p, k + 1, C.c_size_t(nbytes))
    out = np.zeros(nbytes, np.uint8)
    for k, p in enumerate(blocks):
        st.call("st_memcpy_dtoh", out.ctypes.data_as(C.c_void_p), p, C.c_size_t(nbytes))
        assert (out == k + 1).all()


# (kept blocks, and one too large to be kept)
@pytest.mark.parametrize("nbytes", [1, 256, 5000, 300001, 16 << 20, (16 << 20) + 1])
@pytest.mark.parametrize("inner", [False, True])
def test_free_twice(nbytes, inner):
    p = _malloc(nbytes)
    at = C.c_void_p(p.value + (nbytes - 1 if inner else 0))
    st.call("st_free", at)
    for again in (p, at):
        assert st.lib().st_free(again) == ST_EHIP
    blocks = [_malloc(nbytes) for _ in range(3)]
    assert len({b.value for b in blocks}) == 3
    _holds(blocks, nbytes)
    for b in blocks:
        st.call("st_free", b)
        assert st.lib().st_free(b) == ST_EHIP


def test_copies_of_a_track_and_of_pairs():
    n = 4000
    a = np.arange(n, dtype=np.float64)
    first = st.Track(a, a, a, a)
    copy = _capi.Track.from_buffer_copy(first.c)
    first.free()
    st.lib().st_track_free(C.byref(copy))   # its arrays are gone: nothing happens
    tracks = [st.Track(a + k, a, a, a) for k in range(3)]
    for k, t in enumerate(tracks):
        np.testing.assert_array_equal(t.download()[0], a + k)
    assert len({p for t in tracks for p in (t.c.x, t.c.y, t.c.z, t.c.edep)}) == 12
    for t in tracks:
        t.free()
    first = st.VolumeEdepPair(n)
    copy = _capi.Pairs.from_buffer_copy(first.c)
    first.free()
    st.lib().st_pairs_free(C.byref(copy))
    pairs = [st.VolumeEdepPair(n) for _ in range(3)]
    for k, p in enumerate(pairs):
        p.upload(np.full(10 + k, k, np.uint64), np.full(10 + k, 1.0))
    for k, p in enumerate(pairs):
        keys, _ = p.download()
        assert len(keys) == 10 + k and (keys == k).all()
        p.free()
