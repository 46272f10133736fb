"""Products in half form (pg_gemm_half.hip): every tile and block shape by name at its edges, inputs over the range that half form
holds, weights that it refuses, and the models that take it."""
import ctypes as C

import numpy as np
import pytest

from helpers import DeviceArray, as_bf16
from puppygrad_amd import Gpt2Config, Gpt2HipConfig, Gpt2Model, _lib, synth

pytestmark = pytest.mark.gpu

STORE = {"f32": _lib.PG_STORE_F32, "bf16": _lib.PG_STORE_BF16, "int8": _lib.PG_STORE_INT8}
TILE_64x128, TILE_128x128, TILE_128x128_8, TILE_128x256, ROWS, TILE_128x256_8 = range(6)
FORMS = [(s, t, 0, 0) for s in STORE for t in (TILE_64x128, TILE_128x128, TILE_128x128_8, TILE_128x256) if s != "f32" or t != TILE_128x256]
FORMS += [(s, TILE_128x256_8, 0, 0) for s in ("bf16", "int8")]
FORMS += [("cut", t, 0, 0) for t in (TILE_64x128, TILE_128x128_8)]  # f32 rows, both operands in cut form
FORMS += [("cut", ROWS, mt, rows) for mt in (1, 2, 3, 4) for rows in (8, 16, 24, 32, 40, 48) if mt > 2 or rows <= 32]
FORMS += [(s, ROWS, mt, rows) for s in STORE for mt in (1, 2, 3, 4) for rows in (8, 16, 24, 32, 40, 48, 56, 64) if mt > 2 or rows <= 32]


def up(n):
    return (n + 255) // 256 * 256


def half_product_dev(x, w, bias, scales, scale, tile, parts, mt, rows, gelu=False):
    """The product, and whether its weights were refused."""
    f = _lib.load().pg_testing_half_product_dev
    u, v, i = C.c_uint64, C.c_void_p, C.c_int32
    f.argtypes, f.restype = [i, v, v, u, u, u, v, i, v, v, v, C.c_float, i, i, i, i, i, v], C.c_int
    (m, k), n = x.shape, w.shape[0]
    storage = {np.dtype(np.float32): "f32", np.dtype(np.uint16): "bf16", np.dtype(np.int8): "int8"}[w.dtype]
    mp = (m + 15) // 16 * 16
    cut = scale == 0
    size = up((6 if cut else 4) * k * mp) + up(k * n * (6 if cut else 4 if storage == "f32" else 2)) + up(4 * n) + 256
    # (room for padded rows: NaN, which no result may show)
    held = [DeviceArray(x), DeviceArray(w, dtype=w.dtype), DeviceArray(np.full(parts * max(m, mp) * n * (3 if cut and gelu else 2) // 2, np.nan, np.float32)), DeviceArray(bias),
            DeviceArray(np.full(size // 4, np.nan, np.float32))]
    if scales is not None:
        held.append(DeviceArray(scales))
    status = f(0, None, held[0].ptr, m, k, n, held[1].ptr, STORE[storage], held[5].ptr if scales is not None else None, held[3].ptr,
               held[2].ptr, scale, tile, parts, mt, rows, gelu, held[4].ptr)
    got, work = held[2].download(), held[4].download()
    for d in held:
        d.free()
    assert status == 0, _lib.load().pg_last_error_message().decode()
    refused = work.view(np.uint32)[(size - 256) // 4] != 0
    if gelu and cut:  # back from cut form
        bf16 = got.view(np.uint16).reshape(-1)[:3 * n * mp].reshape(n // 8, 3, mp, 8)[:, :, :m].astype(np.uint32) << 16
        return bf16.view(np.float32).astype(np.float64).sum(1).transpose(1, 0, 2).reshape(m, n), refused
    if gelu:  # back from half form
        parts_of = got.view(np.float16).reshape(-1)[:2 * n * mp].reshape(n // 8, 2, mp, 8)[:, :, :m].astype(np.float64)
        return parts_of.sum(1).transpose(1, 0, 2).reshape(m, n), refused
    got = got[:parts * m * n].reshape(parts, m, n)
    return (got[0] if parts == 1 else got.sum(0, dtype=np.float64) + bias), refused


def operands(m, k, n, storage):
    rng = np.random.default_rng([m, k, n])
    x = (rng.standard_normal((m, k)) * 10.0 ** rng.uniform(-3, 1, (m, k))).astype(np.float32)
    w = (rng.standard_normal((n, k)) * 10.0 ** rng.uniform(-3, 1, (n, 1))).astype(np.float32)
    b = rng.standard_normal(n).astype(np.float32)
    if storage in ("f32", "cut"):
        return x, w, None, w.astype(np.float64), b
    if storage == "bf16":
        w = synth.round_bf16(w.reshape(-1)).reshape(w.shape)
        return x, as_bf16(w), None, w.astype(np.float64), b
    q, scales = rng.integers(-127, 128, (n, k)).astype(np.int8), np.abs(w[:, 0]) + np.float32(1e-3)
    return x, q, scales, q * scales[:, None].astype(np.float64), b


def bound_of(x, w, b, scale):
    """f32 sums of K products in any order, their operands off by 2^-23 (of x besides 2^-25 of the scaled unit) and lo lo left
    out, 2^-22; the bias and an int8 row's scale each rounded once.  Cut form (scale 0): the operands are whole, three of nine
    products are left out, 2^-24 and less together."""
    want = x @ w.T + b
    unit = 2.0 ** -25 / scale if scale else 0.0
    return want, (x.shape[1] + 20) * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T) + unit * np.abs(w).sum(1) + 2.0 ** -23 * np.abs(want)


# a row, an octet of columns more than a tile, two stages of K; a tile's rows and one more or less on both sides; chains of uneven
# length, and parts of one stage
@pytest.mark.parametrize("m,k,n,parts", [(1, 64, 64, 1), (63, 96, 136, 1), (65, 288, 128, 1), (128, 256, 264, 2), (129, 1056, 72, 1),
                                         (200, 416, 256, 5), (257, 544, 384, 1), (37, 2080, 520, 8)])
@pytest.mark.parametrize("storage,tile,mt,rows", FORMS)
def test_forms_at_their_edges(storage, tile, mt, rows, m, k, n, parts):
    x, w, scales, values, b = operands(m, k, n, storage)
    scale = 0.0 if storage == "cut" else 256.0
    got, refused = half_product_dev(x, w, b, scales, scale, tile, parts, mt, rows)
    want, bound = bound_of(x.astype(np.float64), values, b, scale)
    assert not refused and (np.abs(got - want) <= bound).all(), f"{(np.abs(got - want) / bound).max():.2f} of the bound"


@pytest.mark.parametrize("storage,tile,mt,rows", [(s, t, 3, 24) for s in STORE for t in range(6) if s != "f32" or t not in (TILE_128x256, TILE_128x256_8)])
def test_every_product_of_the_parts_counts(storage, tile, mt, rows):
    """Operands of one sign whose second parts are large: left out, one product of them is 2^-12 of the sum."""
    rng = np.random.default_rng(5)
    x = (1.0 + 2.0 ** -12 + rng.integers(0, 4, (70, 256)) * 2.0 ** -22).astype(np.float32)
    w = (1.0 + 2.0 ** -12 + rng.integers(0, 4, (136, 256)) * 2.0 ** -22).astype(np.float32)
    scales = None
    if storage == "bf16":
        w = synth.round_bf16(w.reshape(-1)).reshape(w.shape)
    stored, values = (as_bf16(w) if storage == "bf16" else w), w.astype(np.float64)
    if storage == "int8":
        stored, scales = rng.integers(100, 128, w.shape).astype(np.int8), np.full(len(w), 0.5, np.float32)
        values = stored * 0.5
    want = x.astype(np.float64) @ values.T
    got, _ = half_product_dev(x, stored, np.zeros(len(w), np.float32), scales, 1.0, tile, 1, mt, rows)
    # (chains of at most 512 products, 2^-24 each; lo lo, 2^-24 here)
    assert (np.abs(got - want) <= 64 * 2.0 ** -24 * want).all(), (np.abs(got - want) / want).max() * 2.0 ** 24


@pytest.mark.parametrize("storage,tile", [(s, t) for s in STORE for t in (TILE_64x128, TILE_128x128, TILE_128x128_8, TILE_128x256_8) if s != "f32" or t != TILE_128x256_8])
def test_sums_err_to_both_sides(storage, tile):
    """The instructions cut what they add downward; chains of their own for the small products, or of turned sign, leave no side to it."""
    rng = np.random.default_rng(8)
    x, w = rng.standard_normal((1024, 1024)).astype(np.float32), synth.round_bf16(rng.standard_normal(128 * 1024).astype(np.float32)).reshape(128, 1024)
    scales, stored, values = None, w if storage == "f32" else as_bf16(w), w.astype(np.float64)
    if storage == "int8":
        stored, scales = rng.integers(-127, 128, w.shape).astype(np.int8), np.full(len(w), 2.0 ** -7, np.float32)
        values = stored * 2.0 ** -7
    want = x.astype(np.float64) @ values.T
    got, _ = half_product_dev(x, stored, np.zeros(len(w), np.float32), scales, 1024.0, tile, 1, 0, 0)
    # (in units of 2^-23 of the outputs' size.  Each output is off by one such unit at random, the mean of 2^17 of them by 0.003; chains of
    # 64 columns and one sign were off by 0.16 and 0.19)
    off = (got - want).mean() / np.sqrt((want ** 2).mean()) * 2.0 ** 23
    assert abs(off) <= 0.04, off


@pytest.mark.parametrize("tile,mt,rows", [(TILE_64x128, 0, 0), (TILE_128x128_8, 0, 0), (ROWS, 1, 16), (ROWS, 3, 24), (ROWS, 4, 48)])
def test_every_product_of_the_cut_parts_counts(tile, mt, rows):
    """Operands 1 + 2^-9 + 2^-18 and a little: left out, one of the six products is 2^-18 of the sum at least."""
    rng = np.random.default_rng(6)
    x, w = ((1.0 + 2.0 ** -9 + 2.0 ** -18 + rng.integers(0, 4, (n, 64)) * 2.0 ** -22).astype(np.float32) for n in (70, 136))
    want = x.astype(np.float64) @ w.astype(np.float64).T
    got, _ = half_product_dev(x, w, np.zeros(len(w), np.float32), None, 0.0, tile, 1, mt, rows)
    # (the first parts' products are 1, their sums whole numbers; the small ones' sum, 2^-8 of them, is off by 2^-18 of itself at most;
    # the last additions round three times; three products of 2^-27 are left out)
    assert (np.abs(got - want) <= 5 * 2.0 ** -24 * want).all(), (np.abs(got - want) / want).max() * 2.0 ** 24


@pytest.mark.parametrize("storage,tile,mt,rows", [("bf16", TILE_64x128, 0, 0), ("bf16", TILE_128x256, 0, 0), ("bf16", TILE_128x256_8, 0, 0), ("bf16", ROWS, 4, 40),
                                                  ("cut", TILE_64x128, 0, 0), ("cut", TILE_128x128_8, 0, 0), ("cut", ROWS, 4, 48)])
def test_gelu_in_half_and_cut_form(storage, tile, mt, rows):
    x, w, scales, values, b = operands(77, 96, 136, storage)
    scale = 0.0 if storage == "cut" else 64.0
    got, _ = half_product_dev(x, w, b, scales, scale, tile, 1, mt, rows, gelu=True)
    want, bound = bound_of(x.astype(np.float64), values, b, scale)
    gelu = 0.5 * want * (1.0 + np.tanh(np.sqrt(2.0 / np.pi) * (want + 0.044715 * want ** 3)))
    # (its slope is at most 1.13; f32 arithmetic of a few steps; 2^-25 of half form's unit)
    assert (np.abs(got - gelu) <= 1.13 * bound + 2.0 ** -20 * np.abs(want) + 2.0 ** -24).all()


@pytest.mark.parametrize("storage", ["f32", "bf16"])
def test_weights_that_half_form_refuses(storage):
    """Values that are not finite; a row too small or too large to be scaled.  Not: a row that spans more than f16 numbers do, whose
    small weights are right to 2^-40 of its largest."""
    x, _, _, _, b = operands(40, 64, 64, "f32")
    rng = np.random.default_rng(3)
    for value, least, refused in ((1.0, 2.0 ** -20, False), (np.inf, 1.0, True), (np.nan, 1.0, True), (2.0 ** 80, 1.0, True),
                                  (2.0 ** -80, None, True), (1.0, 2.0 ** -45, False), (1.0, 2.0 ** -36, False), (0.0, 0.0, False)):
        w = synth.round_bf16(rng.standard_normal(64 * 64).astype(np.float32)).reshape(64, 64)
        if least is None or value == 0.0:
            w[5] = 0.0
        else:
            w[5, 9] = np.float32(1.0078125 * least)
        w[5, 7] = value
        product, got = half_product_dev(x, as_bf16(w) if storage == "bf16" else w, b, None, 256.0, TILE_64x128, 1, 0, 0)
        assert got == refused, (value, least)
        if not refused:
            want, bound = bound_of(x.astype(np.float64), w.astype(np.float64), b, 256.0)
            assert (np.abs(product - want) <= bound + 2.0 ** -40 * np.abs(w).max(1) * np.abs(x).sum(1, keepdims=True)).all(), (value, least)


def norm_half_dev(x, g, b, scale, parts=None, bias=None):
    """LayerNorm of x, or of x + bias + parts [p][rows][cols], back from half form (times scale) or cut form (scale 0), and the row itself."""
    f = _lib.load().pg_testing_norm_half_dev
    u, v, i, s = C.c_uint64, C.c_void_p, C.c_int32, C.c_float
    f.argtypes, f.restype = [i, v, v, u, u, v, v, s, s, i, v, v, v, v], C.c_int
    (m, k), n = x.shape, 0 if parts is None else len(parts)
    mp, planes = (m + 15) // 16 * 16, 2 if scale else 3
    held = [DeviceArray(x if n == 0 else np.full_like(x, np.nan)), DeviceArray(g), DeviceArray(b), DeviceArray(np.full(planes * mp * k // 2, np.nan))]
    held += [DeviceArray(a) for a in (parts, bias, x)] if n else []
    status = f(0, None, held[0].ptr, m, k, held[1].ptr, held[2].ptr, 1e-5, scale, n, *((d.ptr for d in held[4:]) if n else (None,) * 3), held[3].ptr)
    row, out = held[0].download(), held[3].download()
    for d in held:
        d.free()
    assert status == 0, _lib.load().pg_last_error_message().decode()
    if scale:
        values = out.view(np.float16).reshape(k // 8, 2, mp, 8)[:, :, :m].astype(np.float64) / scale
    else:
        values = (out.view(np.uint16).reshape(k // 8, 3, mp, 8)[:, :, :m].astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    return values.sum(1).transpose(1, 0, 2).reshape(m, k), row


# a block a row and a wavefront a row, at every number of values a lane holds: the last width of each, an odd octet, the widest
@pytest.mark.parametrize("cols", [8, 768, 776, 1280, 1792, 1800, 2048, 2560, 2736, 3648, 4096])
@pytest.mark.parametrize("rows", [1, 67, 300])
@pytest.mark.parametrize("parts", [0, 3])
@pytest.mark.parametrize("scale", [256.0, 0.0])
def test_norms_of_every_width(cols, rows, parts, scale):
    rng = np.random.default_rng([cols, rows, parts])
    x, (g, b, bias) = rng.standard_normal((rows, cols)).astype(np.float32) + np.float32(0.5), rng.standard_normal((3, cols)).astype(np.float32)
    ws = rng.standard_normal((parts, rows, cols)).astype(np.float32) if parts else None
    got, row = norm_half_dev(x, g, b, scale, ws, bias)
    want = x if not parts else x.astype(np.float64) + bias + ws.sum(0, dtype=np.float64)
    # (four roundings of values under 32)
    np.testing.assert_allclose(row, want, rtol=0, atol=4 * 2.0 ** -20 if parts else 0)
    r = row.astype(np.float64)
    d = r - r.mean(1, keepdims=True)
    inv = 1.0 / np.sqrt((d * d).mean(1, keepdims=True) + 1e-5)
    # (f32 sums over a lane's values and 64 lanes: of the mean, 72 + cols / 64 roundings of the values' mean size; of the squares as
    # many of themselves, half of which the root passes on; the cut: half form's 2^-23 and 2^-25 of its unit)
    n = (72 + cols / 64) * 2.0 ** -24
    bound = np.abs(g) * inv * n * np.abs(r).mean(1, keepdims=True) + (n + 2.0 ** -23) * np.abs(d * inv * g) + 2.0 ** -23 * np.abs(d * inv * g + b)
    bound += 2.0 ** -25 / scale if scale else 0.0
    off = np.abs(got - (d * inv * g + b))
    assert (off <= bound).all(), f"{(off / bound).max():.2f} of the bound"


def logits(model, ids):
    return model.prefill(ids, model.new_kv_cache()).to_host()


# the first rows that take the form, tiles that end in the middle, one prompt and several
@pytest.mark.parametrize("storage,width,batch,n", [("f32", 768, 1, 5), ("f32", 1280, 1, 32), ("bf16", 1600, 1, 17), ("int8", 1024, 2, 33), ("bf16", 768, 1, 270),
                                                   ("int8", 1280, 1, 190), ("f32", 768, 1, 1026), ("f32", 768, 1, 129), ("f32", 512, 3, 300), ("f32", 768, 4, 256), ("f32", 1280, 1, 257), ("bf16", 1024, 1, 330), ("int8", 1600, 1, 460),
                                                   ("f32", 1600, 3, 131), ("bf16", 768, 5, 207), ("int8", 768, 2, 700), ("f32", 512, 9, 130)])
def test_prompts(storage, width, batch, n):
    cfg = Gpt2Config(vocab_size=300, n_positions=1100, n_embd=width, n_layer=2, n_head=width // 64)
    w = synth.random_weights(cfg, 0x5EED0B00, perturb=True)
    model = Gpt2Model.new(cfg, w, Gpt2HipConfig(weight_storage=STORE[storage]))
    ids = synth.token_ids(batch * n, 0x70C00B00 + n, 300).reshape(batch, n)
    cache = model.new_kv_cache(batch)
    got = (model.prefill_batch(ids, cache) if batch > 1 else model.prefill(ids[0], cache)).to_host().reshape(batch, -1)
    for b in (0, batch - 1):  # the one-sequence kernels form the last token behind a prompt of other products' rows
        other = model.new_kv_cache()
        at = min(n - 1, 32)
        model.prefill([int(t) for t in ids[b, :at]], other)
        for t in ids[b, at:n - 1]:
            model.forward_one(int(t), other)
        want = model.forward_one(int(ids[b, n - 1]), other).to_host()
        # (the same values, sums of at most 6400 terms in other orders)
        assert np.linalg.norm(got[b] - want) <= 1e-5 * np.linalg.norm(want)


# steps whose rows take the form: the smallest, one more than a block's rows, K cut and not, several blocks of rows; and on the other
# side of the line (f32 up to 16 sequences, bf16 up to 32: packed rows)
@pytest.mark.parametrize("storage,width,batch", [("f32", 768, 17), ("f32", 1600, 17), ("bf16", 1024, 33), ("int8", 768, 17), ("int8", 1280, 33), ("bf16", 768, 70),
                                                 ("int8", 512, 130), ("f32", 768, 2), ("f32", 1600, 16), ("bf16", 1024, 32)])
@pytest.mark.parametrize("n", [3, 40, 300])
def test_batched_steps(storage, width, batch, n):
    cfg = Gpt2Config(vocab_size=300, n_positions=310, n_embd=width, n_layer=2, n_head=width // 64)
    model = Gpt2Model.new(cfg, synth.random_weights(cfg, 0x5EED0B01, perturb=True), Gpt2HipConfig(weight_storage=STORE[storage]))
    ids = synth.token_ids(batch * (n + 2), 0x70C00B01 + n, 300).reshape(batch, n + 2)
    cache = model.new_kv_cache(batch)
    model.prefill_batch(np.ascontiguousarray(ids[:, :n]), cache)
    model.forward_one_batch(ids[:, n], cache)
    got = model.forward_one_batch(ids[:, n + 1], cache).to_host()
    for b in (0, batch - 1):
        single = model.new_kv_cache()
        model.prefill([int(t) for t in ids[b, :n]], single)
        model.forward_one(int(ids[b, n]), single)
        want = model.forward_one(int(ids[b, n + 1]), single).to_host()
        # (the same values, sums of at most 6400 terms in other orders)
        assert np.linalg.norm(got[b] - want) <= 1e-5 * np.linalg.norm(want)


def test_copies_of_the_weights_can_be_declined():
    """A model without them takes their memory less and serves the same calls; none are made where no rows could take them."""
    cfg = Gpt2Config(vocab_size=97, n_positions=512, n_embd=1280, n_layer=2, n_head=20)
    w = synth.random_weights(cfg, 0x5EED0B0B, perturb=True)
    ids = [int(t) for t in synth.token_ids(300, 0x70C00B0B, 97)]
    weights = cfg.n_layer * 12 * cfg.n_embd ** 2

    def free():
        at = (C.c_size_t * 2)()
        assert _lib.load().hipMemGetInfo(C.byref(at, 0), C.byref(at, C.sizeof(C.c_size_t))) == 0
        return at[0]

    def taken(**kw):
        before = free()
        model = Gpt2Model.new(cfg, w, Gpt2HipConfig(**kw))
        return model, before - free()

    logits(Gpt2Model.new(cfg, w), ids)  # (what the process allocates once)
    for storage, bytes_each in (("f32", 6), ("bf16", 2), ("int8", 2)):
        with_them, more = taken(weight_storage=STORE[storage])
        without, less = taken(weight_storage=STORE[storage], weight_copies=1)
        # (allocations in pages of 2 MB)
        assert abs(more - less - bytes_each * weights) <= 8 << 20, (more, less)
        got, want = logits(without, ids), logits(with_them, ids)
        assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)
    _, never = taken(gemm_b9_min_rows=0xffffffff)
    assert never <= 4 * (weights + 700 * cfg.n_embd) + (8 << 20)
    with pytest.raises(Exception, match="weight_copies must be 0 or 1"):
        Gpt2Model.new(cfg, w, Gpt2HipConfig(weight_copies=2))


def test_a_set_bound_holds_for_few_rows():
    cfg = Gpt2Config(vocab_size=97, n_positions=64, n_embd=768, n_layer=1, n_head=12)
    w = synth.random_weights(cfg, 0x5EED0B04, perturb=True)
    ids = [int(t) for t in synth.token_ids(20, 0x70C00B04, 97)]
    never, at, past, alone = (logits(Gpt2Model.new(cfg, w, Gpt2HipConfig(gemm_b9_min_rows=b)), ids) for b in (0xffffffff, 20, 21, 0))
    np.testing.assert_array_equal(past, never)
    np.testing.assert_array_equal(at, alone)
    assert (at != never).any()


def test_a_bf16_weight_far_below_its_row_does_not_cost_a_model_its_form():
    cfg = Gpt2Config(vocab_size=97, n_positions=64, n_embd=768, n_layer=1, n_head=12)
    w = synth.random_weights(cfg, 0x5EED0B06, perturb=True)
    ids = [int(t) for t in synth.token_ids(40, 0x70C00B06, 97)]
    bf16 = Gpt2HipConfig(weight_storage=STORE["bf16"])
    w.blocks[0].c_fc_w.reshape(-1)[5] = 0.0
    want = logits(Gpt2Model.new(cfg, w, bf16), ids)
    w.blocks[0].c_fc_w.reshape(-1)[5] = 1.0078125 * 2.0 ** -60
    np.testing.assert_array_equal(logits(Gpt2Model.new(cfg, w, bf16), ids), want)  # (0 in that form; elsewhere other kernels' sums)


def test_scales_hold_for_models_of_any_size_of_values():
    """Gains, weights and shifts far from the usual: the bounds move with them."""
    cfg = Gpt2Config(vocab_size=97, n_positions=400, n_embd=512, n_layer=1, n_head=8)
    ids = [int(t) for t in synth.token_ids(400, 0x70C00B02, 97)]
    for gain, weight in ((1e3, 1.0), (1e-4, 1.0), (1.0, 1e-4), (3.0, 30.0)):
        w = synth.random_weights(cfg, 0x5EED0B02, perturb=True)
        for blk in w.blocks:
            blk.ln_1_g, blk.ln_2_g = blk.ln_1_g * np.float32(gain), blk.ln_2_g * np.float32(gain)
            blk.c_fc_w, blk.c_attn_w = blk.c_fc_w * np.float32(weight), blk.c_attn_w * np.float32(weight / gain)
        here = Gpt2Model.new(cfg, w, Gpt2HipConfig(weight_storage=STORE["bf16"]))
        # (the f32 cores' products of the same bf16 values)
        for blk in w.blocks:
            for name in ("c_attn_w", "c_proj_w", "c_fc_w", "c_proj_mlp_w"):
                a = getattr(blk, name)
                setattr(blk, name, synth.round_bf16(a.reshape(-1)).reshape(a.shape))
        w.wte = synth.round_bf16(w.wte.reshape(-1)).reshape(w.wte.shape)
        there = Gpt2Model.new(cfg, w, Gpt2HipConfig(gemm_b9_min_rows=0xffffffff))
        got, want = logits(here, ids), logits(there, ids)
        assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want), (gain, weight)
        # Of a prompt's rows all but the last leave the last layer behind its keys and values; here all of them go through it.  Queries and keys
        # are right to 3 2^-24, a score of size s to 6 2^-24 of it, and a weight to twice that where two keys share it; a score's standard
        # deviation is a query's times a key's, and the largest about four of them.
        size = 4 * (weight * 0.02) ** 2 * 512
        got, want = here.forward(ids).logits, there.forward(ids).logits
        off = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
        assert (off <= 1e-5 + size * 12 * 2.0 ** -24).all() and np.median(off) <= 1e-5, (gain, weight, off.max())


def uneven_weights(cfg, seed):
    """Norms, values, hidden units and dims of queries and keys whose columns are of sizes up to 10^8 apart, and what reads them of the inverse."""
    w = synth.random_weights(cfg, seed, perturb=True)
    rng, c, n = np.random.default_rng(seed), cfg.n_embd, cfg.n_inner

    def times(blk, name, by, rows, cols, at=slice(None)):  # by a column, or by a row (of the [in, out] matrix)
        a = np.array(getattr(blk, name), np.float32).reshape(rows, cols)
        a[:, at] *= by.astype(np.float32)
        setattr(blk, name, a.reshape(np.shape(getattr(blk, name))))

    for blk in w.blocks:
        for norm, matrix, out in (("ln_1", "c_attn_w", 3 * c), ("ln_2", "c_fc_w", n)):
            by = 10.0 ** rng.uniform(-4, 4, c)
            times(blk, norm + "_g", by, 1, c)
            times(blk, norm + "_b", by, 1, c)
            times(blk, matrix, 1.0 / by[:, None], c, out)
        score, value, inner = 10.0 ** rng.uniform(-4, 4, c), 10.0 ** rng.uniform(-4, 4, c), 10.0 ** rng.uniform(-3, 3, n)
        for at, by in ((slice(0, c), score), (slice(c, 2 * c), 1.0 / score), (slice(2 * c, None), value)):
            times(blk, "c_attn_w", by, c, 3 * c, at)
            times(blk, "c_attn_b", by, 1, 3 * c, at)
        times(blk, "c_proj_w", 1.0 / value[:, None], c, c)
        times(blk, "c_fc_w", inner, c, n)
        times(blk, "c_fc_b", inner, 1, n)
        times(blk, "c_proj_mlp_w", 1.0 / inner[:, None], n, c)
    return w


# (f32, 300 rows: cut form, with attention in half form)
@pytest.mark.parametrize("storage,batch,n", [("f32", 1, 20), ("f32", 1, 300), ("f32", 4, 300), ("bf16", 1, 40), ("bf16", 1, 300), ("int8", 1, 40), ("int8", 2, 170)])
def test_columns_of_unequal_size(storage, batch, n):
    """Every column counts as it does in f32, however far below the largest it is."""
    cfg = Gpt2Config(vocab_size=97, n_positions=320, n_embd=512, n_layer=2, n_head=8)
    model = Gpt2Model.new(cfg, uneven_weights(cfg, 0x5EED0B07), Gpt2HipConfig(weight_storage=STORE[storage]))
    ids = synth.token_ids(batch * (n + 1), 0x70C00B07, 97).reshape(batch, n + 1)
    cache = model.new_kv_cache(batch)
    got = [model.prefill_batch(np.ascontiguousarray(ids[:, :n]), cache).to_host().reshape(batch, -1)]
    if batch > 1:
        got.append(model.forward_one_batch(ids[:, n], cache).to_host())
    for b in (0, batch - 1):  # the one-sequence kernels
        single = model.new_kv_cache()
        want = [model.prefill([int(ids[b, 0])], single)]
        for t in ids[b, 1:]:
            want.append(model.forward_one(int(t), single))
            want[-1] = want[-1].to_host()
        for logit, ref in zip(got, want[n - 1:]):
            # (the same values, sums of at most 2048 terms in other orders)
            assert np.linalg.norm(logit[b] - ref) <= 1e-5 * np.linalg.norm(ref)


@pytest.mark.parametrize("storage,batch", [("f32", 8), ("bf16", 40), ("int8", 24)])
def test_steps_of_columns_of_unequal_size(storage, batch):
    cfg = Gpt2Config(vocab_size=97, n_positions=32, n_embd=512, n_layer=2, n_head=8)
    model = Gpt2Model.new(cfg, uneven_weights(cfg, 0x5EED0B08), Gpt2HipConfig(weight_storage=STORE[storage]))
    ids = synth.token_ids(batch * 3, 0x70C00B08, 97).reshape(batch, 3)
    cache = model.new_kv_cache(batch)
    model.prefill_batch(np.ascontiguousarray(ids[:, :2]), cache)
    got = model.forward_one_batch(ids[:, 2], cache).to_host()
    for b in (0, batch - 1):
        single = model.new_kv_cache()
        model.prefill([int(t) for t in ids[b, :2]], single)
        want = model.forward_one(int(ids[b, 2]), single).to_host()
        assert np.linalg.norm(got[b] - want) <= 1e-5 * np.linalg.norm(want)


def test_weights_of_24_bits_do_not_shift_the_keys():
    """Two f16 numbers drop a bit of a f32 weight in four.  Norms that are mostly their shifts make that the same error at every position;
    over the positions it is gone."""
    cfg = Gpt2Config(vocab_size=97, n_positions=512, n_embd=1280, n_layer=1, n_head=20)
    w = synth.random_weights(cfg, 0x5EED0B0A, perturb=True)
    blk, rng = w.blocks[0], np.random.default_rng(10)
    blk.ln_1_g = np.full(1280, 0.05, np.float32)
    blk.ln_1_b = rng.uniform(0.5, 1.0, 1280).astype(np.float32)
    ids = synth.token_ids(512, 0x70C00B0A, 97)
    model = Gpt2Model.new(cfg, w)
    cache = model.new_kv_cache()
    model.prefill([int(t) for t in ids], cache)
    got = cache.read_layer(0, 0).astype(np.float64).reshape(20, 512, 64)
    x = (np.float32(w.wte).reshape(97, 1280)[ids] + np.float32(w.wpe).reshape(-1, 1280)[:512]).astype(np.float64)
    d = x - x.mean(1, keepdims=True)
    y = d / np.sqrt((d * d).mean(1, keepdims=True) + cfg.layer_norm_epsilon) * 0.05 + blk.ln_1_b.astype(np.float64)
    at = slice(1280, 2560)
    want = y @ np.asarray(blk.c_attn_w, np.float64).reshape(1280, 3840)[:, at] + np.asarray(blk.c_attn_b, np.float64)[at]
    off = got.transpose(1, 0, 2).reshape(512, 1280) - want
    # (a quarter of the weights off by 2^-23 to 2^-24 of themselves is 0.7 of 2^-24 of the keys at every position; the sums' own roundings,
    # which are much the same at every position here, leave 0.36)
    assert np.sqrt((off.mean(0) ** 2).mean() / (want ** 2).mean()) <= 0.5 * 2.0 ** -24


@pytest.mark.parametrize("storage,batch", [("f32", 8), ("bf16", 40), ("int8", 24)])
@pytest.mark.parametrize("behind", [5, 60])  # (one share of the keys and several)
def test_a_step_behind_another_models_values(storage, batch, behind):
    """The cache holds values 10^4 times the largest that the stepping model can have itself."""
    cfg = Gpt2Config(vocab_size=97, n_positions=80, n_embd=512, n_layer=2, n_head=8)
    small, large = (synth.random_weights(cfg, 0x5EED0B09, perturb=True) for _ in range(2))
    for blk in large.blocks:
        blk.c_attn_b = np.array(blk.c_attn_b, np.float32)
        blk.c_attn_b[1024:] += np.float32(1e5)
    maker, model = (Gpt2Model.new(cfg, w, Gpt2HipConfig(weight_storage=STORE[storage])) for w in (large, small))
    ids = synth.token_ids(batch * (behind + 1), 0x70C00B09, 97).reshape(batch, behind + 1)
    cache = model.new_kv_cache(batch)
    maker.prefill_batch(np.ascontiguousarray(ids[:, :behind]), cache)
    got = model.forward_one_batch(ids[:, behind], cache).to_host()
    for b in (0, batch - 1):
        single = model.new_kv_cache()
        maker.prefill([int(t) for t in ids[b, :behind]], single)
        want = model.forward_one(int(ids[b, behind]), single).to_host()
        # (the same values, sums of at most 2048 terms in other orders)
        assert np.isfinite(want).all() and np.linalg.norm(got[b] - want) <= 1e-5 * np.linalg.norm(want)


@pytest.mark.parametrize("n", [20, 300])  # a block a row, a wavefront a row
def test_rows_whose_squares_are_past_f32(n):
    """Their norm is its shift, in half form as in f32 rows."""
    cfg = Gpt2Config(vocab_size=97, n_positions=400, n_embd=1600, n_layer=2, n_head=25)
    w = synth.random_weights(cfg, 0x5EED0B05, perturb=True)
    w.wte = w.wte * np.float32(1e22)
    w.wpe = w.wpe * np.float32(1e22)
    ids = [int(t) for t in synth.token_ids(n, 0x70C00B05, 97)]
    here, there = (Gpt2Model.new(cfg, w, Gpt2HipConfig(gemm_b9_min_rows=b)) for b in (0, 0xffffffff))
    got, want = logits(here, ids) / np.float32(1e22), logits(there, ids) / np.float32(1e22)
    assert np.isfinite(want).all() and np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)


@pytest.mark.parametrize("storage", STORE)
@pytest.mark.parametrize("how", ["small row", "large row", "infinite bound"])
def test_weights_without_half_form_are_served_as_before(storage, how):
    """A row that cannot be scaled, of a hidden unit whose share is kept; a bound that is not finite, of one that no token reaches."""
    cfg = Gpt2Config(vocab_size=97, n_positions=400, n_embd=512, n_layer=1, n_head=8)
    ids = [int(t) for t in synth.token_ids(400, 0x70C00B03, 97)]
    w = synth.random_weights(cfg, 0x5EED0B03, perturb=True)
    blk = w.blocks[0]
    if how == "infinite bound":
        blk.c_fc_b[3] = -np.inf
    else:
        by = np.float32(2.0 ** -80 if how == "small row" else 2.0 ** 80)
        blk.c_fc_w = np.array(blk.c_fc_w, np.float32).reshape(512, 2048)
        blk.c_fc_w[:, 3] *= by
        blk.c_fc_w = blk.c_fc_w.reshape(-1)
        blk.c_proj_mlp_w = np.array(blk.c_proj_mlp_w, np.float32).reshape(2048, 512)
        blk.c_proj_mlp_w[3] *= 1.0 / by if how == "large row" else 1.0
        blk.c_proj_mlp_w = blk.c_proj_mlp_w.reshape(-1)
    refused, without = (Gpt2Model.new(cfg, w, Gpt2HipConfig(weight_storage=STORE[storage], weight_copies=c)) for c in (0, 1))
    for n in (20, 50, 100, 400):
        got = logits(refused, ids[:n])
        np.testing.assert_array_equal(got, logits(without, ids[:n]))
        single = without.new_kv_cache()
        without.prefill(ids[:3], single)
        for t in ids[3:n - 1]:
            without.forward_one(t, single)
        want = without.forward_one(ids[n - 1], single).to_host()
        if np.isfinite(want).all():
            # (the same values, sums of at most 2048 terms in other orders)
            assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)
        else:
            assert how == "infinite bound" and not np.isfinite(got).any()
        # (the last layer's products of all rows: a prompt of 128 goes on with its last one there)
        every = refused.forward(ids[:n]).logits
        np.testing.assert_array_equal(every, without.forward(ids[:n]).logits)
        if np.isfinite(want).all():
            assert np.linalg.norm(every[-1] - want) <= 1e-5 * np.linalg.norm(want)
