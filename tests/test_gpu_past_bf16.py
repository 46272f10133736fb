"""Small batches and grouped rows against bf16 and int8 matrices where an input is infinite, NaN, finite but infinite
as bf16, or gives a product that only its rounded first part overflows: the kernels repeat such sums in f32."""
import numpy as np
import pytest

from helpers import DeviceArray, as_bf16, grouped_dev, product_dev

pytestmark = pytest.mark.gpu
# 1.5045 2^121 times 85, and (1 + 2^-8 + 2^-20) 2^126 times 4 (1 - 2^-8), stay below 2^128; with the first factor
# rounded up to bf16 they do not
EDGE = {"int8": (np.float32(1.5045 * 2.0 ** 121), 85.0), "bf16": (np.float32((1 + 2.0 ** -8 + 2.0 ** -20) * 2.0 ** 126), 4 - 2.0 ** -6)}
VALUES = ["inf", "-inf", "nan", "3.4e38", "edge"]


def operands(rows, k, n, storage, value, at):
    """x with the value in row `at`, the matrix as it is stored, its scales, and what it stands for"""
    r = np.random.default_rng([rows, k, n])
    x = np.clip(r.standard_normal((rows, k)), -4, 4).astype(np.float32)
    w = np.where(r.random((n, k)) < 0.5, -1.0, 1.0)
    scale = np.full(n, 2.0 ** -10 if value == "edge" else 0.25, np.float32)
    factor = EDGE[storage][1] if value == "edge" else 1.0
    column = 5 * k // 7
    w[:, column] *= factor
    x[at, column] = EDGE[storage][0] if value == "edge" else np.float32(value)
    if storage == "int8":
        return x, w.astype(np.int8), scale, w * scale[:, None].astype(np.float64)
    if value != "edge":
        w *= 0.25
    return x, as_bf16(w), None, w


def check(got, x, values, at):
    others = np.arange(len(x)) != at
    want = x[others].astype(np.float64) @ values.T
    bound = (x.shape[1] + 8) * 2.0 ** -24 * (np.abs(x[others]).astype(np.float64) @ np.abs(values).T)  # f32 sums of K products
    assert (np.abs(got[others] - want) <= bound).all()
    with np.errstate(invalid="ignore"):
        want = x[at].astype(np.float64) @ values.T
    np.testing.assert_array_equal(np.isnan(got[at]), np.isnan(want))
    finite = np.isfinite(want)
    np.testing.assert_array_equal(got[at][~finite], want[~finite].astype(np.float32))
    np.testing.assert_allclose(got[at][finite], want[finite], rtol=1e-6)


# 16-row forms with 16 and 32 rows of W, 32 rows, 64 rows; few rows of W and a deep K: cut over blocks
@pytest.mark.parametrize("value", VALUES)
@pytest.mark.parametrize("rows", [2, 16, 20, 32, 50])
@pytest.mark.parametrize("storage", ["bf16", "int8"])
def test_small_batches(storage, rows, value):
    for k, n, ws in ((1024, 260, 0), (192, 9000, 0), (4096, 100, 8 * rows * 100)):
        x, w, scale, values = operands(rows, k, n, storage, value, rows - 1)
        check(product_dev(x, w, None, scale, ws_floats=ws), x, values, rows - 1)


@pytest.mark.parametrize("value", VALUES)
@pytest.mark.parametrize("rows", [3, 16, 31])
def test_packed_rows(rows, value):
    for k, n, ws in ((1024, 260, 0), (192, 9000, 0), (4096, 100, 8 * rows * 100)):
        x, w, _, values = operands(rows, k, n, "bf16", value, 1)
        check(product_dev(x, w, ws_floats=ws, packed=True), x, values, 1)


@pytest.mark.parametrize("value", VALUES)
@pytest.mark.parametrize("tile_rows", [32, 64, 128])
def test_grouped_rows(tile_rows, value):
    k, n, at = 288, 132, 7
    x, w, _, values = operands(50, k, 2 * n, "bf16", value, at)
    rows = np.random.default_rng(1).integers(0, 50, 3 * tile_rows)
    rows[tile_rows + 3] = at
    dx = DeviceArray(x)
    got = grouped_dev(dx.ptr, 3 * tile_rows, w.reshape(2, n, k), [1, 0, 1], rows, tile_rows)
    for tile, group in enumerate((1, 0, 1)):
        mine, part = rows[tile * tile_rows:][:tile_rows], got[tile * tile_rows:][:tile_rows]
        for i in np.flatnonzero(mine == at)[:2]:
            keep = (mine != at) | (np.arange(tile_rows) == i)
            check(part[keep], x[mine[keep]], values[group * n:][:n], int(np.flatnonzero(np.flatnonzero(keep) == i)[0]))
    dx.free()


@pytest.mark.parametrize("tile_rows", [32, 64, 128])
def test_grouped_pairs(tile_rows):
    """gate and up of column pairs: the value meets small weights, so that both and their product are finite."""
    k, n, at = 288, 132, 7
    x, _, _, values = operands(50, k, 2 * n, "bf16", "3.4e38", at)
    values[:, 5 * k // 7] = np.ldexp(values[:, 5 * k // 7], -120)
    rows = np.random.default_rng(2).integers(0, 50, 2 * tile_rows)
    rows[tile_rows + 5] = at
    dx = DeviceArray(x)
    got = grouped_dev(dx.ptr, 2 * tile_rows, as_bf16(values).reshape(2, n, k), [1, 0], rows, tile_rows, silu_pair=True)
    for tile, group in enumerate((1, 0)):
        c = x[rows[tile * tile_rows:][:tile_rows]].astype(np.float64) @ values[group * n:][:n].T
        gate, up = c[:, 0::2], c[:, 1::2]
        want = gate / (1 + np.exp(-gate)) * up
        # f32 sums of K products: (K + 8) 2^-24 of the sum of their sizes, in both factors (the slope of c / (1 + e^-c) is
        # at most 1.1)
        size = np.abs(x[rows[tile * tile_rows:][:tile_rows]]).astype(np.float64) @ np.abs(values[group * n:][:n]).T
        err = (k + 8) * 2.0 ** -24 * size
        bound = 1.2 * err[:, 0::2] * np.abs(up) + err[:, 1::2] * np.abs(gate) + err[:, 0::2] * err[:, 1::2] + 1e-6 * np.abs(want)
        assert (np.abs(got[tile * tile_rows:][:tile_rows] - want) <= bound).all()
    dx.free()
