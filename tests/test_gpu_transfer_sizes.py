"""f between host memory and float storage on either side of the sizes at which
the conversion moves from the host to the device, for pinned and for pageable
memory: set_f rounds each double to the nearest float and get_f returns the
stored floats exactly, by every route and with every remainder of the four
values that a lane converts; denormal floats, infinities and NaN among them.
"""
import ctypes
import math

import numpy as np
import pytest

from conftest import sld_box

pytestmark = pytest.mark.gpu

# products just below and above 2^18 and 3 2^20 values, of 4 k + 0, 1, 2, 3
SIZES = [(22, 22, 22, 24), (23, 23, 23, 23), (25, 23, 22, 23), (23, 27, 21, 23), (24, 24, 24, 24), (40, 40, 40, 36),
         (41, 43, 45, 38), (44, 45, 40, 39), (45, 45, 40, 39)]


def pinned(n):
    """n doubles of pinned memory from the HIP runtime the library uses."""
    from hip_buffers import hip
    lib = hip()
    p = ctypes.c_void_p()
    lib.hipHostMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t, ctypes.c_uint]
    lib.hipHostFree.argtypes = [ctypes.c_void_p]
    assert lib.hipHostMalloc(ctypes.byref(p), 8 * n, 0) == 0
    return np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_double)), (n,)), lambda: lib.hipHostFree(p)


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("memory", ["pinned", "pageable"])
def test_float_f_by_either_route(vlp, n, memory):
    m = math.prod(n)
    rng = np.random.default_rng(m)
    with vlp.Vlp4d(vlp.VlpConfig.make(*sld_box(n)), precision=32) as sim:
        a, free = pinned(m) if memory == "pinned" else (np.empty(m), lambda: None)
        try:
            a[:] = rng.standard_normal(m) * np.exp(rng.uniform(-20, 20, m))
            a[:6] = [1.0e-39, -1.5e-45, 1.0e-46, 3.5e38, -math.inf, math.nan]
            a[-3:] = [1.0 + 2.0 ** -24, 1.0 + 3 * 2.0 ** -24, -1.2e-38]
            with np.errstate(over="ignore"):
                want = a.astype(np.float32).astype(np.float64)
            sim._check(sim.lib.vlp_set_f(sim.h, vlp._dptr(a), m))
            a[:] = 0
            sim._check(sim.lib.vlp_get_f(sim.h, vlp._dptr(a), m))
            assert np.array_equal(a, want, equal_nan=True)
        finally:
            free()
