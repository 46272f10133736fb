"""Attention of prompts in half form (pg_attn_half.hip): every block shape at its edges."""
import ctypes as C

import numpy as np
import pytest

from helpers import DeviceArray
from puppygrad_amd import _lib

pytestmark = pytest.mark.gpu


def attention_half_dev(qkv, heads, shape, sq, sk, sv, cut=False):
    f = _lib.load().pg_testing_attention_half_dev
    u, v, i, s = C.c_uint64, C.c_void_p, C.c_int32, C.c_float
    f.argtypes, f.restype = [i, v, v, u, u, u, i, s, s, s, i, v, v, v], C.c_int
    n, t, _ = qkv.shape
    m, k = n * t, 64 * heads
    mp = (m + 15) // 16 * 16
    held = [DeviceArray(qkv)] + [DeviceArray(np.full(size, np.nan, np.float32)) for size in (m * k, m * k, mp * k * 3 // 2)]
    status = f(0, None, held[0].ptr, t, heads, n, shape, sq, sk, sv, cut, held[1].ptr, held[2].ptr, held[3].ptr)
    keys, values, out = (d.download() for d in held[1:])
    for d in held:
        d.free()
    assert status == 0, _lib.load().pg_last_error_message().decode()
    if cut:
        parts = (out.view(np.uint16).astype(np.uint32) << 16).view(np.float32).reshape(k // 8, 3, mp, 8)
    else:
        parts = out.view(np.float16)[:2 * mp * k].reshape(k // 8, 2, mp, 8) / np.float32(sv)
    out = parts[:, :, :m].astype(np.float64).sum(1).transpose(1, 0, 2).reshape(n, t, k)
    return out, keys.reshape(n, heads, t, 64), values.reshape(n, heads, t, 64)


# one tile, its edges, tiles that some key groups or query groups have none of
@pytest.mark.parametrize("t", [1, 31, 32, 33, 64, 65, 127, 130, 200, 290])
@pytest.mark.parametrize("shape", [41, 22, 24, 18, 14, 0])
@pytest.mark.parametrize("cut", [False, True])
def test_shapes_at_their_edges(shape, t, cut):
    rng = np.random.default_rng([t, shape])
    heads, n = 2, 2
    qkv = rng.standard_normal((n, t, 3, heads, 64)).astype(np.float32)
    qkv[:, :, 0] *= 3.0
    qkv[1, :, 1:] *= 10.0 ** rng.uniform(-2, 1, (t, 1, 1, 1))  # keys and values of unequal size
    out, keys, values = attention_half_dev(qkv.reshape(n, t, -1), heads, shape, 512.0, 256.0, 64.0, cut)
    np.testing.assert_array_equal(keys, qkv[:, :, 1].transpose(0, 2, 1, 3))
    np.testing.assert_array_equal(values, qkv[:, :, 2].transpose(0, 2, 1, 3))
    q, k, v = (qkv[:, :, j].transpose(0, 2, 1, 3).astype(np.float64) for j in range(3))
    s = np.where(np.tril(np.ones((t, t), bool)), q @ k.transpose(0, 1, 3, 2) / 8.0, -np.inf)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    want = (p @ v).transpose(0, 2, 1, 3).reshape(n, t, -1)
    # a score is off by (64 + 12) 2^-24 of the sum of its products' sizes, and a weight by that much of itself; a sum of weights or
    # of weighted values by (keys + 12) 2^-24, and half form's unit, here of a key, of a value and of a weight
    size = np.abs(q) @ np.abs(k).transpose(0, 1, 3, 2) / 8.0 * 76 * 2.0 ** -24 + np.abs(q).sum(-1)[..., None] / 8.0 * 2.0 ** -25 / 256.0
    rel = np.where(p > 0, size, 0.0).max(-1)[..., None] * 2 + (2 * t + 24) * 2.0 ** -24
    bound = (rel * (p @ np.abs(v)) + 2.0 ** -25 / 64.0 + t * 2.0 ** -32 * np.abs(v).max(2)[:, :, None]).transpose(0, 2, 1, 3).reshape(n, t, -1)
    assert (np.abs(out - want) <= bound).all(), f"{(np.abs(out - want) / bound).max():.2f} of the bound"


def test_every_product_of_the_parts_counts():
    """Scores of 8 and 0 whose second parts are large and of one sign, values that weigh both alike with opposite signs."""
    rng = np.random.default_rng(4)
    rich = lambda *shape: 1.0 + 2.0 ** -12 + rng.integers(0, 4, shape) * 2.0 ** -22
    t = 160
    for which in ("scores", "weights"):
        q, k, v = np.zeros((t, 64)), np.zeros((t, 64)), np.zeros((t, 64))
        if which == "scores":
            strong = np.arange(t) % 2 == 0
            q[:], k[strong] = rich(t, 64), rich(strong.sum(), 64)
            v[strong], v[~strong] = 1.0, -2980.0
        else:
            q[:, 0] = 8.0
            k[np.arange(t) % 32 != 0, 0] = np.log(0.5 + 2.0 ** -13)
            v[:] = rich(t, 64)
        qkv = np.concatenate([q, k, v], 1).astype(np.float32)
        s = qkv[:, :64].astype(np.float64) @ qkv[:, 64:128].T.astype(np.float64) / 8.0
        s = np.where(np.tril(np.ones((t, t), bool)), s, -np.inf)
        p = np.exp(s - s.max(-1, keepdims=True))
        p /= p.sum(-1, keepdims=True)
        w = qkv[:, 128:].astype(np.float64)
        for shape in (41, 22, 24, 18, 14):
            got, _, _ = attention_half_dev(qkv[None], 1, shape, 1.0, 1.0, 1.0)
            # (a score of 8 is off by 2^-21 at most, a part left out makes it 2^-12 of 8)
            bound = (96 if which == "scores" else 48) * 2.0 ** -24 * (p @ np.abs(w))
            assert (np.abs(got[0] - p @ w) <= bound)[40:].all(), (which, shape, (np.abs(got[0] - p @ w) / bound)[40:].max())
