"""Staged copies between host and device and kept device blocks: the bytes
arrive whole at the sizes where the buffers, their number and the number of
copying threads change, from several threads at once; blocks taken again hold
no one else's data."""
import ctypes as C
import threading

import numpy as np
import pytest

import supertrack_amd as st

pytestmark = pytest.mark.gpu

KIB, MIB = 1 << 10, 1 << 20


def _round_trip(a):
    dev = C.c_void_p()
    st.call("st_malloc", C.byref(dev), C.c_size_t(a.nbytes))
    st.call("st_memcpy_htod", dev, a.ctypes.data_as(C.c_void_p), C.c_size_t(a.nbytes))
    b = np.zeros_like(a)
    st.call("st_memcpy_dtoh", b.ctypes.data_as(C.c_void_p), dev, C.c_size_t(a.nbytes))
    st.call("st_free", dev)
    return b


@pytest.mark.parametrize("nbytes", [1, 255, 512 * KIB - 1, 512 * KIB, 512 * KIB + 1, 2 * MIB - 1, 2 * MIB, 4 * MIB + 1,
                                    8 * MIB, 24 * MIB + 13, 41 * MIB])
def test_bytes_arrive_whole(nbytes):
    a = np.random.default_rng(nbytes).integers(0, 256, nbytes, np.uint8)
    assert np.array_equal(_round_trip(a), a)


@pytest.mark.parametrize("shift", [1, 8, 16])
def test_any_device_address(shift):
    a = np.random.default_rng(shift).integers(0, 256, 70001, np.uint8)
    dev = C.c_void_p()
    st.call("st_malloc", C.byref(dev), C.c_size_t(a.nbytes + 64))
    st.call("st_memset", dev, 7, C.c_size_t(a.nbytes + 64))
    st.call("st_memcpy_htod", C.c_void_p(dev.value + shift), a.ctypes.data_as(C.c_void_p), C.c_size_t(a.nbytes))
    b = np.zeros(a.nbytes + 64, np.uint8)
    st.call("st_memcpy_dtoh", b.ctypes.data_as(C.c_void_p), dev, C.c_size_t(b.nbytes))
    st.call("st_free", dev)
    assert np.array_equal(b[shift:shift + a.nbytes], a)
    assert (b[:shift] == 7).all() and (b[shift + a.nbytes:] == 7).all()


@pytest.mark.parametrize("n", [1, 31, 16384, 16385, 65536, 300001, 1100000])
def test_track_columns(n):
    rng = np.random.default_rng(n)
    cols = [rng.standard_normal(n) for _ in range(4)]
    t = st.Track(*cols)
    for p, a in zip((t.c.x, t.c.y, t.c.z, t.c.edep), cols):
        b = np.zeros(n)
        st.call("st_memcpy_dtoh", b.ctypes.data_as(C.c_void_p), p, C.c_size_t(b.nbytes))
        assert np.array_equal(a, b)
    t.free()


def test_several_threads():
    bad = []

    def work(k):
        rng = np.random.default_rng(k)
        for _ in range(6):
            a = rng.integers(0, 256, int(rng.integers(1, 9 * MIB)), np.uint8)
            if not np.array_equal(_round_trip(a), a):
                bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_blocks_taken_again():
    n = 5000
    for _ in range(3):
        pairs = st.VolumeEdepPair(n)
        assert pairs.count() == n
        keys, lineal = pairs.download()
        assert not keys.any() and not lineal.any()
        pairs.upload(np.arange(1, n + 1, dtype=np.uint64), np.full(n, 2.5))
        h = st.Histogram(50, 0.0, 10.0, "lin")
        assert not h.fetch(reset=False).any()
        h.allocate_track_process(pairs)
        h.sort_reduce_and_add_to_histogram(pairs)
        got = h.fetch(reset=False)
        assert got.sum() == n and got.max() == n
        h.free()
        pairs.free()
