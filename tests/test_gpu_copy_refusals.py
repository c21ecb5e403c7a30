"""Copies, fills and uploads of ranges that are not what the call names: what
hipMemcpy and hipMemset refuse is refused (with nothing written), what they
accept is copied, whichever way the bytes are staged."""
import ctypes as C

import numpy as np
import pytest

import supertrack_amd as st
from supertrack_amd import _capi

pytestmark = pytest.mark.gpu

ST_EHIP = -3
KIB, MIB = 1 << 10, 1 << 20
# one kernel for the buffer, queued copies of small and of large buffers, hipMemcpy
SIZES = [1000, 8000, 400 * KIB, 700 * KIB, 5 * MIB, 20 * MIB]


def _lib():
    return st.lib()


def _malloc(nbytes):
    p = C.c_void_p()
    st.call("st_malloc", C.byref(p), C.c_size_t(nbytes))
    return p


def _host(a):
    return a.ctypes.data_as(C.c_void_p)


def _bytes(nbytes, seed=0):
    return np.random.default_rng(nbytes + seed).integers(0, 256, nbytes, np.uint8)


def _read(p, nbytes):
    out = np.zeros(nbytes, np.uint8)
    st.call("st_memcpy_dtoh", _host(out), p, C.c_size_t(nbytes))
    return out


@pytest.mark.parametrize("nbytes", SIZES)
def test_ranges_past_an_allocation(nbytes):
    p, q = _malloc(nbytes), _malloc(nbytes)
    a = _bytes(nbytes + 64)
    st.call("st_memcpy_htod", p, _host(a), C.c_size_t(nbytes))
    for at, more in ((0, 1), (0, 16), (nbytes - 8, 9), (nbytes, 1), (8, nbytes)):
        if at == nbytes and nbytes > 16 * MIB:   # (what lies there may be another allocation)
            continue
        there, n = C.c_void_p(p.value + at), C.c_size_t(nbytes + more if at == 0 else more)
        assert _lib().st_memset(there, 0, n) == ST_EHIP, (at, more)
        assert _lib().st_memcpy_dtoh(_host(a.copy()), there, n) == ST_EHIP, (at, more)
        assert _lib().st_memcpy_dtod(there, q, n) == ST_EHIP, (at, more)
        assert _lib().st_memcpy_dtod(q, there, n) == ST_EHIP, (at, more)
        if nbytes <= 16 * MIB or at >= nbytes - 8:   # (larger ones: the part before the refused piece is written)
            assert _lib().st_memcpy_htod(there, _host(_bytes(nbytes + 64, 1)), n) == ST_EHIP, (at, more)
    assert np.array_equal(_read(p, nbytes), a[:nbytes])
    if nbytes <= 16 * MIB:
        assert _lib().st_free(C.c_void_p(p.value + nbytes)) == ST_EHIP
    st.call("st_free", p)
    st.call("st_free", q)


@pytest.mark.parametrize("nbytes", SIZES)
def test_null_and_host_addresses(nbytes):
    p = _malloc(nbytes)
    a, b, n = _bytes(nbytes), np.zeros(nbytes, np.uint8), C.c_size_t(nbytes)
    st.call("st_memcpy_htod", p, _host(a), n)
    assert _lib().st_memcpy_htod(None, _host(a), n) == ST_EHIP
    assert _lib().st_memcpy_htod(p, None, n) == ST_EHIP
    assert _lib().st_memcpy_dtoh(None, p, n) == ST_EHIP
    assert _lib().st_memcpy_dtoh(_host(b), None, n) == ST_EHIP
    # host memory in the device's place
    assert _lib().st_memcpy_htod(_host(b), _host(a), n) == ST_EHIP
    assert _lib().st_memcpy_dtoh(_host(b), _host(a), n) == ST_EHIP
    assert not b.any()
    assert np.array_equal(_read(p, nbytes), a)
    st.call("st_free", p)


@pytest.mark.parametrize("nbytes", SIZES)
@pytest.mark.parametrize("shift", [0, 1, 8])
def test_device_and_pinned_memory_in_the_hosts_place(nbytes, shift):
    hip = C.CDLL("libamdhip64.so")
    pin = C.c_void_p()
    assert hip.hipHostMalloc(C.byref(pin), C.c_size_t(nbytes + shift), 0) == 0
    p, q = _malloc(nbytes + shift), _malloc(nbytes)
    a, n = _bytes(nbytes), C.c_size_t(nbytes)
    inner, pinned = C.c_void_p(p.value + shift), C.c_void_p(pin.value + shift)
    st.call("st_memcpy_htod", inner, _host(a), n)
    st.call("st_memcpy_htod", q, inner, n)          # device to device, by its address
    assert np.array_equal(_read(q, nbytes), a)
    st.call("st_memset", q, 0, n)
    st.call("st_memcpy_dtoh", q, inner, n)
    assert np.array_equal(_read(q, nbytes), a)
    view = np.frombuffer((C.c_char * nbytes).from_address(pinned.value), np.uint8)
    st.call("st_memcpy_dtoh", pinned, q, n)         # pinned memory
    assert np.array_equal(view, a)
    st.call("st_memset", q, 0, n)
    st.call("st_memcpy_htod", q, pinned, n)
    assert np.array_equal(_read(q, nbytes), a)
    st.call("st_memcpy_htod", pinned, _host(a[::-1].copy()), n)   # (mapped: a device address too)
    assert np.array_equal(view, a[::-1])
    # past the pinned allocation
    big = _malloc(nbytes + 4096)
    assert _lib().st_memcpy_htod(big, pinned, C.c_size_t(nbytes + 8)) == ST_EHIP
    assert _lib().st_memcpy_dtoh(pinned, big, C.c_size_t(nbytes + 8)) == ST_EHIP
    for x in (p, q, big):
        st.call("st_free", x)
    assert hip.hipHostFree(pin) == 0


@pytest.mark.parametrize("n", [10, 5000, 100000])
def test_a_track_larger_than_its_arrays(n):
    """A track that the caller describes: its capacity is not to be trusted."""
    a = np.arange(n + 50, dtype=np.float64)
    t = _capi.Track()
    st.call("st_track_alloc", C.byref(t), C.c_int64(n))
    t.capacity = n + 50
    d = a.ctypes.data_as(_capi.c_double_p)
    assert _lib().st_track_upload(C.byref(t), d, d, d, d, C.c_int64(n + 50)) == ST_EHIP
    st.call("st_track_upload", C.byref(t), d, d, d, d, C.c_int64(n))
    assert np.array_equal(_read(C.c_void_p(t.z), 8 * n).view(np.float64), a[:n])
    t.capacity = n
    st.lib().st_track_free(C.byref(t))


@pytest.mark.parametrize("n", [100, 4000, 40000])
def test_a_track_in_the_callers_own_memory(n):
    """Arrays of another allocator, each at an odd place inside one block."""
    hip = C.CDLL("libamdhip64.so")
    base = C.c_void_p()
    assert hip.hipMalloc(C.byref(base), C.c_size_t(4 * (8 * n + 24) + 100)) == 0
    cols = [np.random.default_rng(k).standard_normal(n) for k in range(4)]
    t = _capi.Track()
    at = [base.value + 8 + k * (8 * n + 24) for k in range(4)]
    t.x, t.y, t.z, t.edep = at
    t.capacity = n
    st.call("st_track_upload", C.byref(t), *[c.ctypes.data_as(_capi.c_double_p) for c in cols], C.c_int64(n))
    for p, c in zip(at, cols):
        assert np.array_equal(_read(C.c_void_p(p), 8 * n).view(np.float64), c)
    # its last column passes the end of the block
    t.edep = base.value + 4 * (8 * n + 24) + 100 - 8 * n + 8
    assert _lib().st_track_upload(C.byref(t), *[c.ctypes.data_as(_capi.c_double_p) for c in cols],
                                  C.c_int64(n)) == ST_EHIP
    assert hip.hipFree(base) == 0
