"""The largest grid a context takes: kernels address an FP64 vector by 32-bit byte
offsets, so storage past 2^29 - 2 points is refused with its reason before any
device call.  cv_ctx_bytes still says what such a grid would need."""
import ctypes as C
import os

import pytest

from curvib_old_amd import _lib

pytestmark = pytest.mark.skipif(not os.path.exists(_lib.SO_PATH), reason="the library is not built")


def desc(storage):
    d = _lib.GridDesc()
    d.IM, d.JM, d.KM = (v - 1 for v in storage)
    for q, b in enumerate((7, 7, 1, 1, 7, 7)):
        d.bctype[q] = b
    d.mglevels, d.ren, d.dt, d.st = 1, 100.0, 1e-3, 1.0
    return d


# 2^29 - 1, 2^29, thin grids past them, about the largest the description itself takes
@pytest.mark.parametrize("storage", [(233, 1103, 2089), (1024, 1024, 512), (5, 5, 21474837), (1290, 1290, 1290)])
def test_storage_past_the_offsets_is_refused(storage):
    n = storage[0] * storage[1] * storage[2]
    assert 2 ** 29 - 2 < n < 2 ** 31
    d, h = desc(storage), C.c_void_p()
    assert _lib.load().cv_ctx_create(C.byref(d), 0, C.byref(h)) == _lib.CV_ERR_ARG and not h
    assert str(n) in _lib.last_error() and str(2 ** 29 - 2) in _lib.last_error(), _lib.last_error()
    assert _lib.load().cv_ctx_bytes(C.byref(d), 1) >= 800 * n


@pytest.mark.parametrize("storage", [(870, 4859, 127), (5, 5, 21474836), (1024, 1024, 511)])
def test_storage_up_to_the_offsets_is_not(storage):
    """Device 1000 ends the call before anything is allocated."""
    assert storage[0] * storage[1] * storage[2] <= 2 ** 29 - 2
    d, h = desc(storage), C.c_void_p()
    assert _lib.load().cv_ctx_create(C.byref(d), 1000, C.byref(h)) == _lib.CV_ERR_HIP and not h
