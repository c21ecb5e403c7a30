"""Allocations while a stream is captured: those that a relaxed capture of the
same thread, or a capture of another thread, allowed still work and leave the
capture whole, also when they take blocks given back before."""
import ctypes as C
import threading

import numpy as np
import pytest

import supertrack_amd as st

pytestmark = pytest.mark.gpu

RELAXED, THREAD_LOCAL, GLOBAL = 2, 1, 0


def _malloc():
    p = C.c_void_p()
    st.call("st_malloc", C.byref(p), C.c_size_t(70000))
    return lambda: st.call("st_free", p)


@pytest.fixture()
def captured():
    """Captures a copy; the graph runs at the end and must have done it."""
    hip = C.CDLL("libamdhip64.so")
    s = C.c_void_p()
    assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0
    src = st.DeviceArray.from_numpy(np.arange(100.0))
    dst = st.DeviceArray.from_numpy(np.zeros(100))
    state = {}

    def begin(mode):
        assert hip.hipStreamBeginCapture(s, mode) == 0
        assert hip.hipMemcpyAsync(dst.ptr, src.ptr, C.c_size_t(800), 3, s) == 0

    def end():
        g, x = C.c_void_p(), C.c_void_p()
        assert hip.hipStreamEndCapture(s, C.byref(g)) == 0
        assert hip.hipGraphInstantiate(C.byref(x), g, None, None, C.c_size_t(0)) == 0
        assert hip.hipGraphLaunch(x, s) == 0 and hip.hipStreamSynchronize(s) == 0
        assert hip.hipGraphExecDestroy(x) == 0 and hip.hipGraphDestroy(g) == 0
        np.testing.assert_array_equal(dst.to_numpy(np.float64, 100), np.arange(100.0))

    state.update(begin=begin, end=end, hip=hip, stream=s)
    yield state
    assert hip.hipStreamDestroy(s) == 0
    src.free()
    dst.free()


@pytest.mark.parametrize("make", [_malloc, lambda: st.Track(capacity=1000).free,
                                  lambda: st.VolumeEdepPair(1000).free])
@pytest.mark.parametrize("mode", [RELAXED, THREAD_LOCAL])
def test_allocations_leave_a_capture_whole(captured, make, mode):
    h = st.Histogram(10, 0.0, 1.0, "lin")
    make()()   # kept blocks
    made = []
    captured["begin"](mode)
    if mode == RELAXED:
        made.append(make())
    else:
        t = threading.Thread(target=lambda: made.append(make()))
        t.start()
        t.join()
    captured["end"]()
    assert len(made) == 1
    made[0]()
    assert h.fetch().sum() == 0
    h.free()


def test_a_refused_allocation_keeps_the_block(captured):
    """A capture that forbids allocations: the call reports it, and the block
    is there for the next one."""
    _malloc()()
    hip, s = captured["hip"], captured["stream"]
    assert hip.hipStreamBeginCapture(s, GLOBAL) == 0
    with pytest.raises(st.SuperTrackError):
        _malloc()
    g = C.c_void_p()
    assert hip.hipStreamEndCapture(s, C.byref(g)) != 0   # (ended by the refused call, as ever)
    hip.hipGetLastError()
    frees = [_malloc() for _ in range(3)]
    for f in frees:
        f()
    captured["begin"](RELAXED)
    captured["end"]()
