"""From how many rows of a prompt on a stack model's last layer goes on with the wanted ones alone."""
import ctypes as C

import pytest

from puppygrad_amd import _lib


@pytest.mark.parametrize("wanted,post_norm,parallel", [(0, 0, 0), (1, 4, 4), (2, 8, 2048), (3, 12, 2048), (31, 124, 2048), (32, 128, 2048)])
def test_lines(wanted, post_norm, parallel):
    f = _lib.load().pg_testing_few_rows_from
    f.argtypes, f.restype = [C.c_int32, C.c_uint64], C.c_uint64
    assert (f(1, wanted), f(0, wanted)) == (post_norm, parallel)
