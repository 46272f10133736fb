"""argmax of rows of any length: the turns and groups of the kernel, ties across them, the last id, values that are not numbers."""
import ctypes as C

import numpy as np
import pytest

from puppygrad_amd import _lib

pytestmark = pytest.mark.gpu


def argmax_dev(x):
    x, out, lib = np.ascontiguousarray(x, np.float32), C.c_uint32(7), _lib.load()
    assert lib.pg_op_argmax(0, x.ctypes.data_as(C.POINTER(C.c_float)), C.c_uint64(x.size), C.byref(out)) == 0
    return out.value


@pytest.mark.parametrize("n", [1, 2, 63, 64, 1023, 1024, 1025, 8191, 8192, 8193, 16384, 16385, 50257, 51200, 51201, 65535, 65536, 65537, 73729, 120000])
def test_the_first_maximum(n):
    rng = np.random.default_rng(n)
    x = rng.standard_normal(n).astype(np.float32)
    assert argmax_dev(x) == np.argmax(x)
    for at in {0, n - 1, n // 2, 1023 % n, 1024 % n, 8191 % n, 8192 % n, 65535 % n, 65536 % n}:
        y = x.copy()
        y[at] = 9.0
        assert argmax_dev(y) == at
        y[rng.integers(at, n, 5)] = 9.0  # equal ones behind it, in later turns, groups, lanes
        assert argmax_dev(y) == at
        y[rng.integers(0, n, 3)] = np.nan
        y[at] = 9.0
        assert argmax_dev(y) == at
    assert argmax_dev(np.zeros(n)) == 0
    assert argmax_dev(np.full(n, -np.inf)) == 0 and argmax_dev(np.full(n, np.nan)) == 0
    y = np.full(n, -np.inf)
    y[-1] = -3e38
    assert argmax_dev(y) == n - 1
