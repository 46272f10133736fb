"""Which rows of activations a model keeps in cut form (gemm_takes_cut): both sides of every limit."""
import ctypes as C

import pytest

from puppygrad_amd import _lib

F32, BF16, INT8 = _lib.PG_STORE_F32, _lib.PG_STORE_BF16, _lib.PG_STORE_INT8
NEVER = 0x7fffffff


def takes(rows, width, storage, inner=None, bound=33, cus=256):
    f = _lib.load().pg_testing_takes_cut
    f.argtypes, f.restype = [C.c_int32] * 6, C.c_int32
    return bool(f(rows, width, inner or 4 * width, storage, bound, cus))


# the last row count of a width on 256 CUs
LAST = {F32: {256: 1024, 512: 1024, 768: 1024, 1024: 320, 1280: 256, 1600: 192},
        BF16: {256: 1472, 512: 704, 768: 512, 1024: 320, 1280: 256, 1600: 192},
        INT8: {256: 3072, 512: 1536, 768: 1024, 1024: 768, 1280: 576, 1600: 448}}


@pytest.mark.parametrize("storage", LAST)
def test_both_sides_of_the_limits(storage):
    for width, last in LAST[storage].items():
        want = set(range(33, last + 1))
        if storage == F32:  # (65 to 128 rows: on the f32 cores at every setting of the bound)
            want -= set(range(65, 129))
        if storage == INT8:  # (few rows: where the product is small)
            want |= set(range(17, {1280: 25, 1600: 16}.get(width, 32) + 1))
        assert {m for m in range(1, 4000) if takes(m, width, storage)} == want, width


def test_the_bound_is_for_f32_rows():
    for bound in (33, 40, 65, 200):
        took = [m for m in range(1, 1100) if takes(m, 768, F32, bound=bound)]
        assert took == [m for m in range(bound, 1025) if not 65 <= m <= 128]
    assert not any(takes(m, 768, F32, bound=NEVER) for m in range(1, 1100))
    assert takes(40, 768, BF16, bound=NEVER) and takes(40, 768, INT8, bound=NEVER)


def test_other_widths_and_parts_of_the_chip():
    assert not takes(64, 224, BF16) and not takes(64, 784, BF16) and not takes(64, 768, BF16, inner=3088)
    assert takes(64, 768, BF16, inner=768)  # c_attn is the widest then: two rounds of 48 columns of it
    assert takes(640, 768, BF16, inner=768) and not takes(704, 768, BF16, inner=768)
    for storage in (F32, BF16, INT8):  # half of the CUs: half of the rounds
        last = LAST[storage][768] // 2
        assert takes(last, 768, storage, cus=128) and not takes(last + 1, 768, storage, cus=128)
