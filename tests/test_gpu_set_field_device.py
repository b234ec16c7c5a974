"""dgk_set_field from an array in device memory: the runtime's copy takes it, so
nothing may read it on the host.  Fields set that way, constant and varying, give
the steps that the same fields give from host memory."""
import ctypes as C

import numpy as np
import pytest

import dgk
from dgk import inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["HIP", "HIP_MP"])
@pytest.mark.parametrize("wind", ["constant", "last node differs", "varying"])
def test_device_array_equals_host_array(form, wind):
    dgk.lib()
    hip = C.CDLL("libamdhip64.so.7")
    ne, p = (3, 2, 5), 4
    q, u, v, w = inputs.random_fields(*ne, p, seed=41, vel_scale=0.6)
    if wind != "varying":
        u, v, w = (np.full_like(q, c) for c in (0.4, -0.3, 0.55))
    if wind == "last node differs":
        w[-1, -1] *= 1.5
    n = q.size
    dev = C.c_void_p()
    assert hip.hipMalloc(C.byref(dev), C.c_size_t(8 * n)) == 0
    got = []
    try:
        for from_device in (False, True):
            with dgk.Solver.structured(form, *ne, p) as s:
                for which, f in enumerate((q, u, v, w)):
                    if from_device:
                        f = np.ascontiguousarray(f)
                        assert hip.hipMemcpy(dev, C.c_void_p(f.ctypes.data), C.c_size_t(8 * n), 1) == 0
                        rc = dgk.lib().dgk_set_field(s._h, which, dev, n)
                        assert rc == 0, dgk.lib().dgk_last_error()
                    else:
                        s.set_field(which, f)
                s.step(1e-3, 3)
                got.append([s.get_field(k) for k in range(4)])
    finally:
        assert hip.hipFree(dev) == 0
    for a, b in zip(*got):
        assert np.array_equal(a, b)
