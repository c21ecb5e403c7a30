"""The host layout, which st_library_append falls back to, really runs when the
device's scratch cannot be had: the one allocation that fails here is used up
by a library that is made all the same."""
import ctypes as C

import numpy as np
import pytest

import supertrack_amd as st
from supertrack_amd import workloads as W
from test_gpu_layout import HISTS, _same, _scan

pytestmark = pytest.mark.gpu


def _allocations_left():
    """Allocations made before one fails (None: none fails)."""
    for k in range(40):
        p = C.c_void_p()
        if st.lib().st_malloc(C.byref(p), C.c_size_t(64)) != 0:
            return k
        st.call("st_free", p)
    return None


@pytest.mark.parametrize("precision", [st.ST_F64, st.ST_F32])
def test_one_failed_allocation_is_the_layouts_scratch(precision):
    """Every allocation of st_library_create fails once: only one of them, the
    layout's, does not fail the call, and it is the one that the comparison of
    the two layouts lets fail."""
    x, y, z, e, off = st.synth_library(dict(W.workload("cfg3")["synth"], n_max=20000), 3, 0)
    geoms = [st.SphericalGeometry(2.5e3, 10.0)]
    made = []
    for k in range(1, 40):
        st.call("st_debug_fail_allocation", C.c_int64(k))
        try:
            lib = st.TrackLibrary(x, y, z, e, off, geoms, None, precision)
            left = _allocations_left()
            made.append((k, left))
            lib.free()
            if left is not None:   # not reached: the library makes fewer allocations
                break
        except st.SuperTrackError as ex:
            assert ex.code == -2
        finally:
            st.call("st_debug_fail_allocation", C.c_int64(0))
    assert [left for _, left in made] == [None, 0], made
    assert made[0][0] == (9 if precision == st.ST_F32 else 7)   # (the number that test_gpu_layout uses)
    _same(_scan((x, y, z, e, off), geoms, None, precision, False), _scan((x, y, z, e, off), geoms, None, precision, True))
    assert len(HISTS) == 2 and _allocations_left() is None
