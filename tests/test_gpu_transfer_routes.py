"""Copies at the sizes where the way they take changes: the kernel over a small
buffer, hipMemcpy, large buffers; one column or several, at each alignment of
the device's address; counts of wide histograms straight to the caller."""
import ctypes as C

import numpy as np
import pytest

import supertrack_amd as st
from supertrack_amd import _capi

pytestmark = pytest.mark.gpu

KIB, MIB = 1 << 10, 1 << 20


@pytest.mark.parametrize("nbytes", [7, 64 * KIB - 1, 64 * KIB, 64 * KIB + 1, 512 * KIB, 16 * MIB - 1, 16 * MIB,
                                    16 * MIB + 9, 33 * MIB])
@pytest.mark.parametrize("shift", [0, 4, 8, 16])
def test_one_column(nbytes, shift):
    a = np.random.default_rng(nbytes + shift).integers(0, 256, nbytes, np.uint8)
    d = st.DeviceArray(nbytes + 64)
    st.call("st_memset", d.ptr, 9, C.c_size_t(nbytes + 64))
    st.call("st_memcpy_htod", C.c_void_p(d.ptr.value + shift), a.ctypes.data_as(C.c_void_p), C.c_size_t(nbytes))
    out = np.zeros(nbytes, np.uint8)
    st.call("st_memcpy_dtoh", out.ctypes.data_as(C.c_void_p), C.c_void_p(d.ptr.value + shift), C.c_size_t(nbytes))
    assert np.array_equal(out, a)
    whole = d.to_numpy(np.uint8, nbytes + 64)
    assert (whole[:shift] == 9).all() and (whole[shift + nbytes:] == 9).all()
    d.free()


# four columns of up to 512 KiB with their paddings, and of 4 MiB, in all
@pytest.mark.parametrize("n", [1, 16383, 16384, 16385, 131071, 131072, 131073, 600001])
@pytest.mark.parametrize("shift", [0, 4, 8])
def test_four_columns(n, shift):
    cols = [np.random.default_rng(n + k).standard_normal(n) for k in range(4)]
    d = st.DeviceArray(4 * (8 * n + 32))
    t = _capi.Track()
    at = [d.ptr.value + shift + k * (8 * n + 32) for k in range(4)]
    t.x, t.y, t.z, t.edep = at
    t.capacity = n
    st.call("st_track_upload", C.byref(t), *[c.ctypes.data_as(_capi.c_double_p) for c in cols], C.c_int64(n))
    for p, c in zip(at, cols):
        out = np.zeros(n)
        st.call("st_memcpy_dtoh", out.ctypes.data_as(C.c_void_p), C.c_void_p(p), C.c_size_t(8 * n))
        np.testing.assert_array_equal(out, c)
    d.free()


@pytest.mark.parametrize("nbins", [8192, 8193, 100000])
def test_wide_counts(nbins):
    rng = np.random.default_rng(nbins)
    m = 5000
    keys, ys = np.arange(m, dtype=np.uint64), rng.uniform(0.0, 320.0, m)
    h = st.Histogram(nbins, 0.01, 300.0, "lin")
    p = st.VolumeEdepPair(m)
    p.upload(keys, ys)
    inside = (ys >= h.edges[0]) & (ys < h.edges[-1])
    want = np.bincount(np.searchsorted(h.edges, ys[inside], side="right") - 1, minlength=nbins)
    for k in range(3):
        h.allocate_track_process(p)
        h.sort_reduce_and_add_to_histogram(p)
        np.testing.assert_array_equal(h.fetch(reset=False), want)
        if k == 1:
            h.free_track_process()
            np.testing.assert_array_equal(h.counts(), want)
        else:
            np.testing.assert_array_equal(h.fetch(reset=True), want)
        assert h.fetch().sum() == 0
    p.free()
    h.free()
