"""vlj_fixed_sum_device at the sizes where its split can go wrong: none to a few
values, both workgroup sizes and the line between them, one pass and several,
odd counts, and arrays that start between two 16-byte boundaries."""
import ctypes as C

import numpy as np
import pytest

from test_zz_no_alloc import D2H, H2D, hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 2, 3, 2047, 2048, 2049, 65535, 65536, 65537, 8192 * 256 - 1, 8192 * 256 + 3])
def test_sum_over_the_splits(lj, n):
    from virial_particles import _lib

    h = hip()
    rng = np.random.default_rng(n + 1)
    scale = 2.0 ** 32
    values = rng.standard_normal(n + 1) * 2.0 ** rng.integers(-20, 11, n + 1)
    d, o = C.c_void_p(), C.c_void_p()
    assert h.hipMalloc(C.byref(d), (n + 1) * 8) == 0 and h.hipMalloc(C.byref(o), 8) == 0
    try:
        assert h.hipMemcpy(d, values.ctypes.data, (n + 1) * 8, H2D) == 0
        for first in (0, 1):
            for _ in range(2):  # the ticket is back at zero
                assert _lib.lib().vlj_fixed_sum_device(C.c_void_p(d.value + 8 * first), n, scale, o, None) == 0
            assert h.hipDeviceSynchronize() == 0
            out = np.zeros(1, dtype=np.int64)
            assert h.hipMemcpy(out.ctypes.data, o, 8, D2H) == 0
            assert int(out[0]) == int(np.rint(values[first:first + n] * scale).astype(np.int64).sum())
    finally:
        h.hipFree(d)
        h.hipFree(o)
