"""Shared test helpers: an independent float64 GPT-2 in matrix form, fixtures, tolerances."""
from pathlib import Path

import numpy as np

from puppygrad_amd import Gpt2Config, synth

GOLDEN = Path(__file__).resolve().parent / "golden"

# north-star logit tolerance for the fp32 path
ABS_TOL, REL_TOL = 1e-4, 1e-3


def assert_logits_close(got, want, abs_tol=ABS_TOL, rel_tol=REL_TOL, what="logits"):
    got, want = np.asarray(got, np.float64), np.asarray(want, np.float64)
    assert got.shape == want.shape, (got.shape, want.shape)
    err = np.abs(got - want)
    bound = abs_tol + rel_tol * np.abs(want)
    bad = err > bound
    assert not bad.any(), (f"{what}: {bad.sum()} of {bad.size} outside {abs_tol} abs + {rel_tol} "
                           f"rel; max err {err.max():.3e} at {np.unravel_index(err.argmax(), err.shape)}")


def numpy_gpt2_forward(cfg: Gpt2Config, w, ids, lm_head=None) -> np.ndarray:
    """GPT-2 in float64 with whole-matrix numpy ops on the HF [in,out] weights.
    Written from the architecture, not from the oracle's loops: a transposed
    weight, a wrong head slice or a dropped residual fails against it.
    lm_head ([vocab, n_embd]) replaces the tied wte in the final projection only."""
    f = lambda a, *s: np.asarray(a, np.float64).reshape(*s)
    C, H, I, V = cfg.n_embd, cfg.n_head, cfg.n_inner, cfg.vocab_size
    hd = C // H
    T = len(ids)
    wte, wpe = f(w.wte, V, C), f(w.wpe, cfg.n_positions, C)
    x = wte[np.asarray(ids)] + wpe[:T]

    def ln(v, g, b):
        mu = v.mean(-1, keepdims=True)
        var = ((v - mu) ** 2).mean(-1, keepdims=True)
        return (v - mu) / np.sqrt(var + cfg.layer_norm_epsilon) * f(g, C) + f(b, C)

    mask = np.tril(np.ones((T, T), bool))
    for b in w.blocks:
        qkv = ln(x, b.ln_1_g, b.ln_1_b) @ f(b.c_attn_w, C, 3 * C) + f(b.c_attn_b, 3 * C)
        q, k, v = [qkv[:, i * C:(i + 1) * C].reshape(T, H, hd).transpose(1, 0, 2) for i in range(3)]
        s = q @ k.transpose(0, 2, 1) / np.sqrt(hd)
        s = np.where(mask, s, -np.inf)
        p = np.exp(s - s.max(-1, keepdims=True))
        p /= p.sum(-1, keepdims=True)
        a = (p @ v).transpose(1, 0, 2).reshape(T, C)
        x = x + a @ f(b.c_proj_w, C, C) + f(b.c_proj_b, C)
        h = ln(x, b.ln_2_g, b.ln_2_b) @ f(b.c_fc_w, C, I) + f(b.c_fc_b, I)
        h = 0.5 * h * (1.0 + np.tanh(np.sqrt(2.0 / np.pi) * (h + 0.044715 * h ** 3)))
        x = x + h @ f(b.c_proj_mlp_w, I, C) + f(b.c_proj_mlp_b, C)
    head = wte if lm_head is None else f(lm_head, V, C)
    return ln(x, w.ln_f_g, w.ln_f_b) @ head.T


def load_golden(name: str):
    z = np.load(GOLDEN / f"{name}.npz")
    c = [int(v) for v in z["config"]]
    cfg = Gpt2Config(vocab_size=c[0], n_positions=c[1], n_embd=c[2], n_layer=c[3], n_head=c[4],
                     n_inner=c[5], layer_norm_epsilon=float(z["eps"]))
    w = synth.random_weights(cfg, int(z["weight_seed"]), perturb=bool(z["perturb"]))
    return cfg, w, z


def small_cases():
    """(name, config, weights, ids) for models small enough for any test."""
    out = []
    cfg = synth.tiny_config()
    out.append(("tiny", cfg, synth.tiny_weights(cfg), [1, 2, 3]))
    cfg = Gpt2Config(vocab_size=131, n_positions=40, n_embd=128, n_layer=2, n_head=2)
    out.append(("c128", cfg, synth.random_weights(cfg, 0x5EED0201, perturb=True),
                list(synth.token_ids(17, 0x70C00201, 131))))
    cfg = Gpt2Config(vocab_size=300, n_positions=64, n_embd=36, n_layer=2, n_head=3, n_inner=100)
    out.append(("odd", cfg, synth.random_weights(cfg, 0x5EED0202, std=0.08, perturb=True),
                list(synth.token_ids(23, 0x70C00202, 300))))
    return out


class DeviceArray:
    """A host array mirrored in a device buffer of the library (pg_device_*)."""

    def __init__(self, host, dtype=np.float32):
        import ctypes as C
        from puppygrad_amd import _lib
        self._C, self.lib = C, _lib.load()
        self.host = np.ascontiguousarray(host, dtype=dtype)
        self.ptr = C.c_void_p()
        assert self.lib.pg_device_alloc(0, self.host.nbytes, C.byref(self.ptr)) == 0
        assert self.lib.pg_device_upload(0, self.ptr, self.host.ctypes.data_as(C.c_void_p),
                                         self.host.nbytes) == 0

    def download(self) -> np.ndarray:
        out = np.empty_like(self.host)
        assert self.lib.pg_device_download(0, out.ctypes.data_as(self._C.c_void_p), self.ptr,
                                           out.nbytes) == 0
        return out

    def free(self):
        assert self.lib.pg_device_free(0, self.ptr) == 0


def product_dev(x, w, bias=None, scales=None, tile=None, parts=1, ws_floats=0, packed=False):
    """x [rows][k] times w [n][k] (f32, bf16 as uint16 or int8 with scales) through the library's testing entry:
    a given tile (rows, columns and 1 for the other form of that size) and number of parts of the bf16
    matrix-core kernels, or (tile None) the planner's choice."""
    import ctypes as C
    from puppygrad_amd import _lib
    lib = _lib.load()
    f = lib.pg_testing_product_dev
    u, v, i = C.c_uint64, C.c_void_p, C.c_int32
    f.argtypes, f.restype = [i, v, v, u, u, u, v, i, v, v, v, i, i, i, i, i, v, u], C.c_int
    (rows, k), n = x.shape, w.shape[0]
    storage = {np.dtype(np.float32): _lib.PG_STORE_F32, np.dtype(np.uint16): _lib.PG_STORE_BF16,
               np.dtype(np.int8): _lib.PG_STORE_INT8}[w.dtype]
    stored = x
    if packed:  # float4 of four columns of all 32 rows side by side
        stored = np.zeros((k // 4, 32, 4), np.float32)
        stored[:, :rows] = x.reshape(rows, k // 4, 4).transpose(1, 0, 2)
    held = [DeviceArray(stored), DeviceArray(w, dtype=w.dtype), DeviceArray(np.full((rows, n), np.nan))]
    scale = DeviceArray(scales) if scales is not None else None
    b = DeviceArray(bias) if bias is not None else None
    ws = DeviceArray(np.full(ws_floats, np.nan)) if ws_floats else None
    held += [d for d in (scale, b, ws) if d is not None]
    ptr = lambda d: d.ptr if d is not None else None
    status = f(0, None, held[0].ptr, rows, k, n, held[1].ptr, storage, ptr(scale), ptr(b), held[2].ptr, int(packed),
               *(tuple(tile or ()) + (0, 0, 0))[:3], parts, ptr(ws), ws_floats)
    got = held[2].download()
    for d in held:
        d.free()
    assert status == 0, lib.pg_last_error_message().decode()
    return got


def as_bf16(a):
    """uint16 of a value that is a bf16 number already."""
    return (np.ascontiguousarray(a, np.float32).view(np.uint32) >> 16).astype(np.uint16)


def grouped_dev(x, rows, w, group_tile, group_rows, tile_rows, silu_pair=False):
    """launch_gemm_grouped through the library's testing entry: x a device pointer to rows of w.shape[2] values, w
    [groups][n][k] (f32 or bf16 as uint16), `rows` slots with their padding."""
    import ctypes as C
    from puppygrad_amd import _lib
    lib = _lib.load()
    f = lib.pg_testing_grouped_dev
    u, v, i = C.c_uint64, C.c_void_p, C.c_int32
    f.argtypes, f.restype = [i, v, v, u, u, u, v, i, i, v, i, v, v], C.c_int
    _, n, k = w.shape
    dw, tiles = DeviceArray(w, dtype=w.dtype), DeviceArray(group_tile, dtype=np.int32)
    slots = DeviceArray(group_rows, dtype=np.int32) if group_rows is not None else None
    out = DeviceArray(np.full((rows, n // 2 if silu_pair else n), np.nan))
    status = f(0, None, x, rows, k, n, dw.ptr, _lib.PG_STORE_BF16 if w.dtype == np.uint16 else _lib.PG_STORE_F32,
               int(silu_pair), out.ptr, tile_rows, tiles.ptr, slots.ptr if slots else None)
    got = out.download()
    for d in (dw, tiles, out) + ((slots,) if slots else ()):
        d.free()
    assert status == 0, lib.pg_last_error_message().decode()
    return got
