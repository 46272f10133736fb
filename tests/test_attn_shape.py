"""Which block shape a prompt's attention takes (attn_cut_shape): the lines on 256 CUs, and a part of the chip."""
import ctypes as C

import pytest

from puppygrad_amd import _lib


def shape(rows, heads, n, cus=256):
    f = _lib.load().pg_testing_attn_shape
    f.argtypes, f.restype = [C.c_int32] * 4, C.c_int32
    return f(rows, heads, n, cus)


@pytest.mark.parametrize("rows,heads,n,want", [
    (32, 25, 32, 0), (33, 12, 16, 22), (33, 12, 15, 0), (64, 12, 16, 22), (65, 12, 7, 0), (65, 12, 8, 24), (128, 12, 16, 42), (128, 20, 16, 41),
    (256, 16, 11, 41), (257, 12, 11, 22), (400, 12, 5, 42), (401, 12, 4, 24), (401, 12, 5, 24), (512, 25, 14, 22), (512, 25, 15, 41),
    (1000, 25, 1, 24), (1024, 12, 1, 0), (577, 25, 1, 24), (576, 25, 1, 0)])
def test_lines(rows, heads, n, want):
    assert shape(rows, heads, n) == want


def test_half_of_the_chip_takes_half_of_the_blocks():
    for rows in (33, 64, 100, 257, 600, 1000):
        for n in (2, 5, 16, 60):
            assert shape(rows, 12, n, 128) == shape(rows, 24, n, 256)
