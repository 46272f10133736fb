"""Attention operands whose second and third bf16 parts are large and of one sign, and attention over a choice of the parts'
products in f64: which product counts how much."""
import numpy as np

from puppygrad_amd import synth

PRODUCTS = [(0, 0), (0, 1), (1, 0), (1, 1), (0, 2), (2, 0)]  # (part of one operand, part of the other)
ROWS, FIRST = 160, 40  # queries from FIRST on see both kinds of key in number
# of the sum of the weights' and values' sizes: f32 sums of these sizes stay within it, a product left out does not
BOUND = {"scores": 64 * 2.0 ** -24, "weights": 24 * 2.0 ** -24}


def parts(x):
    """f32 as three bf16 numbers whose sum it is."""
    out, rest = [], np.asarray(x, np.float32)
    for _ in range(3):
        p = synth.round_bf16(rest.reshape(-1)).reshape(rest.shape)
        out.append(p)
        rest = rest - p
    return [p.astype(np.float64) for p in out]


def operands(which, seed=4):
    """qkv [1][ROWS][192] for one head."""
    rng = np.random.default_rng(seed)
    rich = lambda *shape: 1.0 + 2.0 ** -9 + 2.0 ** -18 + rng.integers(0, 4, shape) * 2.0 ** -22
    q, k, v = np.zeros((ROWS, 64)), np.zeros((ROWS, 64)), np.zeros((ROWS, 64))
    if which == "scores":
        # scores of 8 and 0, values that weigh both alike with opposite signs: an error of a score is one of the result
        strong = np.arange(ROWS) % 2 == 0
        q[:], k[strong] = rich(ROWS, 64), rich(strong.sum(), 64)
        v[strong], v[~strong] = 1.0, -np.exp(8.0)
    else:
        # a key of weight 1 in every tile of 32, the others of 1/2 + 2^-10 + 2^-19
        q[:, 0] = 8.0
        k[np.arange(ROWS) % 32 != 0, 0] = np.log(0.5 + 2.0 ** -10 + 2.0 ** -19)
        v[:] = rich(ROWS, 64)
    return np.concatenate([q, k, v], 1).astype(np.float32)[None]


def attention(qkv, scores=PRODUCTS, weights=PRODUCTS):
    """Output and, for the bound, sum of weight and value sizes, rows FIRST and on."""
    q, k, v = (qkv[0, :, 64 * i:64 * i + 64] for i in range(3))
    qp, kp, vp = parts(q), parts(k), parts(v)
    s = sum(kp[a] @ qp[b].T for a, b in scores).T / 8.0
    s = np.where(np.tril(np.ones(s.shape, bool)), s, -np.inf)
    p = np.exp(s - s.max(-1, keepdims=True))
    pp = parts(p)
    total = p.sum(-1, keepdims=True)
    out = sum(pp[b] @ vp[a] for a, b in weights) / total
    return out[FIRST:], ((p / total) @ np.abs(v.astype(np.float64)))[FIRST:]


def exact(qkv):
    q, k, v = (qkv[0, :, 64 * i:64 * i + 64].astype(np.float64) for i in range(3))
    s = q @ k.T / 8.0
    s = np.where(np.tril(np.ones(s.shape, bool)), s, -np.inf)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    return (p @ v)[FIRST:]
