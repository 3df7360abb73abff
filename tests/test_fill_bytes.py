"""lsjk_memset_zero and lsjk_enqueue_zero clear the bytes asked for, to the last one, and no others."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 3, 4, 7, 255, 1024 * 1024 + 2])
def test_fill(product_backend, n):
    import capi_ctypes as C
    print("fill", n, flush=True)
    lib = C.Lib(0)
    L = lib.L
    L.lsjk_enqueue_zero.argtypes = [C.vp, C.csz]
    size = n + 64
    d = C.vp()
    lib.check(L.lsjk_malloc(ctypes.byref(d), size))
    try:
        for clear in (L.lsjk_memset_zero, L.lsjk_enqueue_zero):
            for offset in (0, 16):
                a = np.full(size, 0xa5, np.uint8)
                lib.check(L.lsjk_memcpy_htod(d, a.ctypes.data, size))
                lib.check(clear(C.vp(d.value + offset), n))
                lib.check(L.lsjk_memcpy_dtoh(a.ctypes.data, d, size))
                assert not a[offset:offset + n].any()
                assert (a[:offset] == 0xa5).all() and (a[offset + n:] == 0xa5).all()
    finally:
        lib.free(d)
