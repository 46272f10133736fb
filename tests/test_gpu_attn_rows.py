"""Causal attention of prompts on the bf16 matrix cores (pg_attn_cut.hip): every block shape at the edges of its tiles, large
scores, values that are not finite or infinite as bf16, and the sizes at which the planner changes shape."""
import ctypes as C

import numpy as np
import pytest

import attn_parts
from helpers import DeviceArray
from puppygrad_amd import _lib

pytestmark = pytest.mark.gpu

SHAPES = [41, 22, 42, 24]


def attention_rows_dev(qkv, heads, shape):
    lib = _lib.load()
    f = lib.pg_testing_attention_rows_dev
    u, v, i = C.c_uint64, C.c_void_p, C.c_int32
    f.argtypes, f.restype = [i, v, v, u, u, u, i, v, v, v], C.c_int
    n, rows, _ = qkv.shape
    panel = np.full((n, heads, rows, 64), np.nan)
    held = [DeviceArray(qkv), DeviceArray(panel), DeviceArray(panel), DeviceArray(np.full((n, rows, 64 * heads), np.nan))]
    status = f(0, None, held[0].ptr, rows, heads, n, shape, held[1].ptr, held[2].ptr, held[3].ptr)
    keys, values, out = (d.download() for d in held[1:])
    for d in held:
        d.free()
    assert status == 0, lib.pg_last_error_message().decode()
    return keys, values, out


def split(qkv, heads):
    n, rows, _ = qkv.shape
    return qkv.reshape(n, rows, 3, heads, 64).transpose(2, 0, 3, 1, 4)  # q, k, v: [n][heads][rows][64]


def exact(qkv, heads):
    q, k, v = split(qkv.astype(np.float64), heads)
    s = q @ k.transpose(0, 1, 3, 2) / 8.0
    rows = s.shape[-1]
    s = np.where(np.tril(np.ones((rows, rows), bool)), s, -np.inf)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    return (p @ v).transpose(0, 2, 1, 3).reshape(len(qkv), rows, -1), p, v, q, k


def check(qkv, heads, shape):
    keys, values, out = attention_rows_dev(qkv, heads, shape)
    _, k, v = split(qkv, heads)
    np.testing.assert_array_equal(keys, k)
    np.testing.assert_array_equal(values, v)
    want, p, v, q, k = exact(qkv, heads)
    # A score is a sum of 64 products, right to 70 2^-24 sum |q k| / 8 (an eighth of the squares' root in each); the weights carry
    # that relative error, twice in the quotient, and the sums of weights and products at most rows + 8 roundings.
    size = np.abs(q) @ np.abs(k).transpose(0, 1, 3, 2) / 8.0
    size = np.where(np.tril(np.ones(size.shape[-2:], bool)), size, 0.0).max(-1, keepdims=True)
    rel = 2.0 ** -24 * (2 * 72 * size + qkv.shape[1] + 16)
    bound = (rel * (p @ np.abs(v))).transpose(0, 2, 1, 3).reshape(want.shape)
    assert (np.abs(out - want) <= bound).all(), f"{(np.abs(out - want) / bound).max():.2f} of the bound"


# one token, one tile and one more, a block of 64 and 128 and one more, ragged; more tiles than key groups
@pytest.mark.parametrize("rows,heads,n", [(1, 1, 1), (31, 2, 2), (32, 1, 3), (33, 3, 1), (64, 1, 2), (65, 2, 1), (127, 1, 1), (129, 2, 2),
                                          (160, 1, 1), (300, 3, 2), (517, 1, 1)])
@pytest.mark.parametrize("shape", SHAPES)
def test_shapes_at_their_edges(shape, rows, heads, n):
    rng = np.random.default_rng([rows, heads, n])
    check(rng.standard_normal((n, rows, 192 * heads)).astype(np.float32), heads, shape)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("which", ["scores", "weights"])
def test_every_product_of_the_parts_counts(shape, which):
    """A product of the parts left out is twice the bound and more (test_attn_parts.py)."""
    qkv = attn_parts.operands(which)
    got, size = attention_rows_dev(qkv, 1, shape)[2][0, attn_parts.FIRST:], attn_parts.attention(qkv)[1]
    err = np.abs(got - attn_parts.exact(qkv)) / (attn_parts.BOUND[which] * size)
    assert (err <= 1.0).all(), f"{err.max():.2f} of the bound"


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("scale", [0.01, 5.0, 12.0])
def test_flat_and_steep_weights(shape, scale):
    """Scores from next to equal to hundreds apart, growing along the keys (the running maximum moves in every tile) and
    falling (it never moves after the first)."""
    rng = np.random.default_rng(7)
    qkv = rng.standard_normal((2, 200, 192)).astype(np.float32)
    qkv[:, :, :128] *= np.float32(scale)
    qkv[0, :, 64:128] += np.linspace(0, 3, 200, dtype=np.float32)[:, None] * qkv[0, 150, :64]
    qkv[1, :, 64:128] += np.linspace(3, 0, 200, dtype=np.float32)[:, None] * qkv[1, 150, :64]
    check(qkv, 1, shape)


@pytest.mark.parametrize("shape", SHAPES)
def test_values_past_bf16(shape):
    """3.39e38 and more is infinite as bf16 and a finite value in f32."""
    rng = np.random.default_rng(8)
    qkv = rng.standard_normal((1, 100, 192)).astype(np.float32)
    qkv[0, 40, 130] = 3.4e38
    out = attention_rows_dev(qkv, 1, shape)[2]
    want = exact(qkv, 1)[0]
    np.testing.assert_allclose(out, want, rtol=2e-5, atol=2e-5)
    assert np.isfinite(out).all()


@pytest.mark.parametrize("shape", SHAPES)
def test_not_finite(shape):
    rng = np.random.default_rng(9)
    qkv = np.abs(rng.standard_normal((1, 100, 192))).astype(np.float32)
    qkv[0, 50, 70] = -np.inf  # a key: no weight for any query behind it
    qkv[0, 60, 180] = np.inf  # a value
    qkv[0, 70, 140] = np.nan
    out = attention_rows_dev(qkv, 1, shape)[2][0]
    with np.errstate(invalid="ignore"):
        want = exact(qkv[:, :50], 1)[0][0]
    np.testing.assert_allclose(out[:50], want, rtol=2e-5, atol=2e-6)
    clean = np.delete(qkv, 50, 1)
    clean[0, 59, 180] = clean[0, 69, 140] = 0.0
    after = np.insert(exact(clean, 1)[0][0], 50, np.nan, 0)
    dims = np.setdiff1d(np.arange(64), [140 - 128, 180 - 128])
    np.testing.assert_allclose(out[51:, dims], after[51:, dims], rtol=2e-5, atol=2e-6)
    assert np.isposinf(out[60:, 180 - 128]).all() and np.isnan(out[70:, 140 - 128]).all()
    assert np.isfinite(out[51:70, 140 - 128]).all() and np.isfinite(out[51:60, 180 - 128]).all()


# sequences of 20 to 600 tokens in ones, a few and many: the planner's shapes, each on both sides of where it changes
@pytest.mark.parametrize("rows,heads,n", [(32, 12, 16), (33, 12, 16), (64, 12, 15), (65, 12, 7), (100, 12, 8), (100, 12, 16), (128, 20, 16),
                                          (200, 16, 3), (256, 16, 11), (257, 12, 11), (400, 25, 1), (600, 25, 1), (640, 25, 1)])
def test_planned_shapes(rows, heads, n):
    rng = np.random.default_rng([rows, heads, n, 1])
    check(rng.standard_normal((n, rows, 192 * heads)).astype(np.float32), heads, 0)
