"""Sums over the lanes of a wavefront (pg_wave.h): additions in the order of a butterfly over 32, 16, 8, 4, 2, 1, bit for bit."""
import ctypes as C

import numpy as np
import pytest

from helpers import DeviceArray
from puppygrad_amd import _lib

pytestmark = pytest.mark.gpu


def lane_sums_dev(x, y):
    lib = _lib.load()
    f = lib.pg_testing_lane_sums_dev
    f.argtypes, f.restype = [C.c_int32, C.c_void_p, C.c_void_p, C.c_void_p, C.c_uint64, C.c_void_p], C.c_int
    held = [DeviceArray(x), DeviceArray(y), DeviceArray(np.full((5, *x.shape), np.nan))]
    status = f(0, None, held[0].ptr, held[1].ptr, len(x), held[2].ptr)
    got = held[2].download()
    for d in held:
        d.free()
    assert status == 0, lib.pg_last_error_message().decode()
    return got


def butterfly(v, distances):
    lanes = np.arange(64)
    for d in distances:
        v = v + v[:, lanes ^ d]
    return v


def test_sums_are_those_of_a_butterfly():
    rng = np.random.default_rng(3)
    x = (rng.standard_normal((200, 64)) * 10.0 ** rng.uniform(-3, 3, (200, 64))).astype(np.float32)
    # (products of numbers of 14 bits: exact in f64, as is their sum with an f32 number of their size)
    y = (rng.integers(1 << 13, 1 << 14, (200, 64)) * 2.0 ** -13).astype(np.float32)
    x[100:] = y[:100]
    got = lane_sums_dev(x, y)
    np.testing.assert_array_equal(got[0], butterfly(x, (32, 16, 8, 4, 2, 1)))
    np.testing.assert_array_equal(got[2], butterfly(x, (4, 2, 1)))
    np.testing.assert_array_equal(got[3], butterfly(x, (8, 4, 2, 1)))
    np.testing.assert_array_equal(got[4], butterfly(x, (1, 2, 4, 8)))
    a, b = x[100:], y[100:]
    other = (a * b)[:, np.arange(64) ^ 32]
    first = (a.astype(np.float64) * b + other).astype(np.float32)
    want = butterfly(first, (16, 8, 4, 2, 1))
    np.testing.assert_array_equal(got[1][100:], want)
    assert (want != butterfly(a * b, (32, 16, 8, 4, 2, 1))).any()
