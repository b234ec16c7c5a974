"""A large download into pinned host memory takes the plain copy, also once the
sliced one is available, and returns the same bytes as one into ordinary memory."""
import ctypes as C

import numpy as np
import pytest

import dgk

pytestmark = pytest.mark.gpu


def test_download_into_pinned_memory():
    hip = C.CDLL("libamdhip64.so.7")
    with dgk.Solver.structured("HIP", 49, 48, 50, 3) as s:
        n = s.Ne * s.Np
        q = (np.arange(n, dtype=np.float64) * 1.25 - 7.0).reshape(s.Ne, s.Np)
        s.set_field(dgk.FIELD_Q, q)
        p = C.c_void_p()
        assert hip.hipHostMalloc(C.byref(p), C.c_size_t(8 * n), C.c_uint(0)) == 0
        try:
            out = np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_double)), (s.Ne, s.Np))
            for _ in range(2):
                out[:] = 0
                assert dgk.lib().dgk_get_field(s._h, dgk.FIELD_Q, p, n) == 0
                assert np.array_equal(out, q)
                assert np.array_equal(s.get_field(dgk.FIELD_Q), q)
        finally:
            del out
            assert hip.hipHostFree(p) == 0
