"""Products with the input in cut form (pg_gemm_rows.hip): every block shape by name at its edges, values that are
infinite as bf16, and the models' own way through them, prompts and batched steps."""
import ctypes as C

import numpy as np
import pytest

from helpers import DeviceArray, as_bf16
from test_cut_form import LAST, takes
from puppygrad_amd import Gpt2Config, Gpt2HipConfig, Gpt2Model, _lib, synth

pytestmark = pytest.mark.gpu

# (16 rows, 16 rows of W) a block; two only for int8 rows, four only for narrower ones than f32
SHAPES = [(s, m, g) for s in ("f32", "bf16", "int8") for m, g in ((2, 1), (3, 1), (4, 1), (2, 2), (3, 2), (4, 2), (3, 3), (4, 3), (3, 4), (4, 4))
          if (m > 2 or s == "int8") and (g < 4 or s != "f32")]


def cut_product_dev(x, w, bias, scales, mt, ng, block_rows, parts=1):
    lib = _lib.load()
    f = lib.pg_testing_cut_product_dev
    u, v, i = C.c_uint64, C.c_void_p, C.c_int32
    f.argtypes, f.restype = [i, v, v, u, u, u, v, i, v, v, v, i, i, i, i, v], C.c_int
    (rows, k), n = x.shape, w.shape[0]
    storage = {np.dtype(np.float32): _lib.PG_STORE_F32, np.dtype(np.uint16): _lib.PG_STORE_BF16,
               np.dtype(np.int8): _lib.PG_STORE_INT8}[w.dtype]
    # (room for padded rows: NaN, which no result may show)
    held = [DeviceArray(x), DeviceArray(w, dtype=w.dtype), DeviceArray(np.full((parts, rows, n), np.nan)), DeviceArray(bias),
            DeviceArray(np.full(6 * k * ((rows + 15) // 16 * 16) // 4, np.nan))]
    if scales is not None:
        held.append(DeviceArray(scales))
    status = f(0, None, held[0].ptr, rows, k, n, held[1].ptr, storage, held[5].ptr if scales is not None else None,
               held[3].ptr, held[2].ptr, mt, ng, block_rows, parts, held[4].ptr)
    got = held[2].download()
    for d in held:
        d.free()
    assert status == 0, lib.pg_last_error_message().decode()
    return got[0] if parts == 1 else got.sum(0, dtype=np.float64) + bias


def operands(rows, k, n, storage):
    """x, the matrix as it is handed over, its scales, the values it stands for, bias"""
    rng = np.random.default_rng([rows, k, n])
    x = (rng.standard_normal((rows, k)) * 10.0 ** rng.uniform(-3, 3, (rows, k))).astype(np.float32)
    w = (rng.standard_normal((n, k)) * 10.0 ** rng.uniform(-3, 1, (n, k))).astype(np.float32)
    b = rng.standard_normal(n).astype(np.float32)
    if storage == "f32":
        return x, w, None, w.astype(np.float64), b
    if storage == "bf16":
        w = synth.round_bf16(w.reshape(-1)).reshape(w.shape)
        return x, as_bf16(w), None, w.astype(np.float64), b
    q, scales = rng.integers(-127, 128, (n, k)).astype(np.int8), np.abs(w[:, 0]) + np.float32(1e-3)
    return x, q, scales, q * scales[:, None].astype(np.float64), b


def within_f32_sums(got, x, w, b):
    """|error| <= (K + 8) 2^-24 sum |x w| + 2^-23 |result|: f32 sums of K products in any order, products right to
    2^-24, the bias and (int8) the row scale each rounded once."""
    x = x.astype(np.float64)
    want = x @ w.T + b
    bound = (x.shape[1] + 8) * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T) + 2.0 ** -23 * np.abs(want)
    assert (np.abs(got - want) <= bound).all(), f"{(np.abs(got - want) / bound).max():.2f} of the bound"


# one row, one octet of columns, one step of K; a block's rows and one more on both sides; idle wavefronts and an
# uneven number of steps; K cut into as many parts as there are steps for each wavefront, and unevenly
@pytest.mark.parametrize("rows,k,n,parts", [(1, 32, 8, 1), (16, 256, 40, 1), (33, 288, 136, 1), (49, 96, 72, 1), (65, 544, 264, 1),
                                            (37, 256, 24, 1), (40, 1056, 80, 4), (70, 2080, 56, 8), (64, 768, 2304, 3)])
@pytest.mark.parametrize("storage,mt,ng", SHAPES)
def test_blocks_at_their_edges(storage, mt, ng, rows, k, n, parts):
    x, w, scales, values, b = operands(rows, k, n, storage)
    for block_rows in sorted({8, 16 * ng - 8, 16 * ng} - {0}):
        within_f32_sums(cut_product_dev(x, w, b, scales, mt, ng, block_rows, parts), x, values, b)


@pytest.mark.parametrize("storage", ["f32", "bf16", "int8"])
def test_every_product_of_the_parts_counts(storage):
    """Operands of one sign whose second and third parts are large: left out, one product of the lowest that are formed
    is 2^-18 of the sum and more."""
    rng = np.random.default_rng(5)
    x = (1.0 + 2.0 ** -9 + 2.0 ** -18 + rng.integers(0, 4, (40, 256)) * 2.0 ** -22).astype(np.float32)
    w = (1.0 + 2.0 ** -9 + 2.0 ** -18 + rng.integers(0, 4, (64, 256)) * 2.0 ** -22).astype(np.float32)
    scales = None
    if storage == "bf16":
        w = synth.round_bf16(w.reshape(-1)).reshape(w.shape)
    stored, values = (as_bf16(w) if storage == "bf16" else w), w.astype(np.float64)
    if storage == "int8":
        stored, scales = rng.integers(100, 128, w.shape).astype(np.int8), np.full(64, 0.5, np.float32)
        values = stored * 0.5
    b = np.zeros(64, np.float32)
    want = x.astype(np.float64) @ values.T
    got = cut_product_dev(x, stored, b, scales, 3, 2, 32)
    # (sums of 256 terms, half of them over eight wavefronts; three products left out, 2^-24 together)
    assert (np.abs(got - want) <= 48 * 2.0 ** -24 * want).all(), (np.abs(got - want) / want).max() * 2.0 ** 24


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, np.float32(3.4e38), np.float32(-3.4028235e38)])
@pytest.mark.parametrize("storage", ["f32", "bf16", "int8"])
def test_values_past_bf16_meet_the_weights_as_in_f32(storage, value):
    x, w, scales, values, b = operands(40, 96, 64, storage)
    x = np.clip(x, -10, 10)
    x[17, 3] = value
    values = np.sign(values) * 0.25  # (an int8 row's scale multiplies its sum, which has to be finite without it)
    w = values.astype(np.float32)
    if storage == "bf16":
        w = as_bf16(w)
    if storage == "int8":
        w, scales = np.sign(w).astype(np.int8), np.full(64, 0.25, np.float32)
    got = cut_product_dev(x, w, b, scales, 3, 2, 32)
    others = np.arange(40) != 17
    within_f32_sums(got[others], x[others], values, b)
    with np.errstate(invalid="ignore"):
        want = x[17].astype(np.float64) @ values.T + b
    np.testing.assert_array_equal(np.isnan(got[17]), np.isnan(want))
    if np.isfinite(value):
        np.testing.assert_allclose(got[17], want, rtol=1e-6)
    else:
        np.testing.assert_array_equal(got[17][np.isinf(want)], want[np.isinf(want)])


def test_infinite_weights_and_weights_past_bf16():
    x, w, _, _, b = operands(40, 96, 64, "f32")
    x, w = np.clip(x, -10, 10), np.clip(w, -1, 1)
    x[:, 7] = np.where(np.abs(x[:, 7]) < 0.1, 0.1, x[:, 7])
    w[5, 7], w[9, 7] = np.inf, np.float32(3.4e37)
    w[11, 7] = np.float32(3.4028235e38)  # infinite as bf16
    x[:, 7] *= np.float32(0.05)
    got = cut_product_dev(x, w, b, None, 3, 2, 32)
    rest = np.setdiff1d(np.arange(64), [5, 9, 11])
    within_f32_sums(got[:, rest], x, w[rest].astype(np.float64), b[rest])
    np.testing.assert_array_equal(got[:, 5], np.where(x[:, 7] > 0, np.inf, -np.inf))
    np.testing.assert_allclose(got[:, [9, 11]], x.astype(np.float64) @ w[[9, 11]].astype(np.float64).T, rtol=1e-5)


# sizes that take the form: the first and the last of a width, ragged blocks between them; and the first past them (test_cut_form.py
# has all of them).  Logits of a prompt against those of its last token alone behind the others, which the one-sequence
# kernels form
@pytest.mark.parametrize("storage,width,n", [("f32", 768, 33), ("f32", 768, 64), ("f32", 1024, 130), ("f32", 1600, 166), ("bf16", 768, 49),
                                             ("bf16", 1600, 131), ("int8", 768, 17), ("int8", 768, 97), ("int8", 1600, 420),
                                             ("int8", 1280, 300), ("f32", 768, 455), ("f32", 768, 456), ("f32", 768, 1024), ("f32", 768, 1025),
                                             ("f32", 1280, 256), ("f32", 1600, 192), ("bf16", 768, 512), ("bf16", 768, 513), ("bf16", 1600, 192),
                                             ("int8", 768, 1024), ("int8", 768, 1025), ("int8", 1600, 448)])
@pytest.mark.parametrize("copies", [False, True])  # (with the weights kept a second time most of these rows are kept in other forms)
def test_prompts(storage, width, n, copies):
    cfg = Gpt2Config(vocab_size=300, n_positions=1100 if n > 512 else 512, n_embd=width, n_layer=2, n_head=width // 64)
    store = {"f32": _lib.PG_STORE_F32, "bf16": _lib.PG_STORE_BF16, "int8": _lib.PG_STORE_INT8}[storage]
    assert takes(n, width, store) == (n <= LAST[store][width])
    model = Gpt2Model.new(cfg, synth.random_weights(cfg, 0x5EED0A00, perturb=True), Gpt2HipConfig(weight_storage=store, weight_copies=0 if copies else 1))
    ids = [int(t) for t in synth.token_ids(n, 0x70C00A00 + n, cfg.vocab_size)]
    cache, other = model.new_kv_cache(), model.new_kv_cache()
    got = model.prefill(ids, cache).to_host()
    # token by token: the GEMM path needs four tokens
    for at in range(0, n - 1, 3):
        part = ids[at:min(at + 3, n - 1)]
        if at == 0:
            model.prefill(part, other)
        else:
            for t in part:
                model.forward_one(t, other)
    want = model.forward_one(ids[-1], other).to_host()
    # (the same values, sums of at most 6400 terms in other orders)
    assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)


def test_a_set_bound_of_the_bf16_cores_holds_for_the_cut_form():
    """Left alone, prompts of 33 to 64 rows are kept cut; a set bound, the default's own number too, keeps fewer rows on the
    f32 cores."""
    cfg = Gpt2Config(vocab_size=97, n_positions=64, n_embd=768, n_layer=1, n_head=12)
    w = synth.random_weights(cfg, 0x5EED0A02, perturb=True)
    ids = [int(t) for t in synth.token_ids(64, 0x70C00A02, cfg.vocab_size)]

    def logits(rows, bound):
        model = Gpt2Model.new(cfg, w, Gpt2HipConfig(gemm_b9_min_rows=bound))
        return model.prefill(ids[:rows], model.new_kv_cache()).to_host()

    for rows in (33, 64):
        on_f32_cores = logits(rows, 0xffffffff)
        assert (logits(rows, 0) != on_f32_cores).any() and (logits(rows, rows) != on_f32_cores).any()
        for bound in (rows + 1, 65, 128):
            np.testing.assert_array_equal(logits(rows, bound), on_f32_cores)


@pytest.mark.parametrize("storage,batch,n", [("f32", 33, 3), ("f32", 48, 20), ("bf16", 40, 7), ("int8", 17, 5), ("int8", 31, 9), ("int8", 65, 4),
                                             ("f32", 128, 3), ("f32", 129, 3), ("f32", 130, 2)])
@pytest.mark.parametrize("copies", [False, True])
def test_batched_steps(storage, batch, n, copies):
    cfg = Gpt2Config(vocab_size=300, n_positions=600, n_embd=768, n_layer=2, n_head=12)
    store = {"f32": _lib.PG_STORE_F32, "bf16": _lib.PG_STORE_BF16, "int8": _lib.PG_STORE_INT8}[storage]
    model = Gpt2Model.new(cfg, synth.random_weights(cfg, 0x5EED0A01, perturb=True), Gpt2HipConfig(weight_storage=store, weight_copies=0 if copies else 1))
    ids = synth.token_ids(batch * (n + 2), 0x70C00A01 + n, cfg.vocab_size).reshape(batch, n + 2)
    cache = model.new_kv_cache(batch)
    model.prefill_batch(np.ascontiguousarray(ids[:, :n]), cache)
    model.forward_one_batch(ids[:, n], cache)
    got = model.forward_one_batch(ids[:, n + 1], cache).to_host()
    for b in (0, 15, 16, batch - 1):
        single = model.new_kv_cache()
        model.prefill([int(t) for t in ids[b, :n]], single)
        model.forward_one(int(ids[b, n]), single)
        want = model.forward_one(int(ids[b, n + 1]), single).to_host()
        assert np.linalg.norm(got[b] - want) <= 1e-5 * np.linalg.norm(want)


@pytest.mark.parametrize("maker,user,batch", [("f32", "f32 never", 40), ("int8", "f32", 17), ("int8", "bf16", 31)])
def test_a_cache_of_another_model_leaves_the_step_to_its_own(maker, user, batch):
    """The form of a batched step's activations is the stepping model's, whichever model of these sizes made the cache."""
    cfg = Gpt2Config(vocab_size=300, n_positions=32, n_embd=768, n_layer=2, n_head=12)
    w = synth.random_weights(cfg, 0x5EED0A03, perturb=True)
    store = {"f32": _lib.PG_STORE_F32, "bf16": _lib.PG_STORE_BF16, "int8": _lib.PG_STORE_INT8}

    def model(name):
        bound = 0xffffffff if name.endswith("never") else 0
        return Gpt2Model.new(cfg, w, Gpt2HipConfig(weight_storage=store[name.split()[0]], gemm_b9_min_rows=bound))

    ids = synth.token_ids(batch * 6, 0x70C00A03, cfg.vocab_size).reshape(batch, 6)
    m, other = model(user), model(maker)
    steps = []
    for cache in (m.new_kv_cache(batch), other.new_kv_cache(batch)):
        m.prefill_batch(np.ascontiguousarray(ids[:, :5]), cache)
        steps.append(m.forward_one_batch(ids[:, 5], cache).to_host())
    if batch > 32:
        np.testing.assert_array_equal(steps[1], steps[0])
    else:  # (a cache of the model's own is packed: the same kernel, sums of at most 3072 terms in other orders)
        assert np.linalg.norm(steps[1] - steps[0]) <= 1e-5 * np.linalg.norm(steps[0])


@pytest.mark.parametrize("storage,rows", [("f32", 40), ("bf16", 64), ("int8", 100)])
def test_models_wider_than_the_norms_that_keep_a_row_in_registers(storage, rows):
    """n_embd past 4096 has no half form and takes cut form: a prompt of so many rows, and a step of so many sequences."""
    cfg = Gpt2Config(vocab_size=97, n_positions=128, n_embd=4160, n_layer=1, n_head=65, n_inner=512)
    store = {"f32": _lib.PG_STORE_F32, "bf16": _lib.PG_STORE_BF16, "int8": _lib.PG_STORE_INT8}[storage]
    assert takes(rows, 4160, store, 512)
    model = Gpt2Model.new(cfg, synth.random_weights(cfg, 0x5EED0A03, perturb=True), Gpt2HipConfig(weight_storage=store))
    ids = synth.token_ids(rows + 1, 0x70C00A03, cfg.vocab_size)
    cache = model.new_kv_cache()
    got = model.prefill([int(t) for t in ids[:rows]], cache).to_host()
    single = model.new_kv_cache()
    for at, t in enumerate(ids[:rows]):
        last = model.prefill([int(t)], single) if at == 0 else model.forward_one(int(t), single)
    want = last.to_host()
    # (the same values, sums of at most 4160 terms in other orders)
    assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)
    batch = model.new_kv_cache(rows)
    model.prefill_batch(np.ascontiguousarray(ids[:rows, None]), batch)
    step = model.forward_one_batch(np.full(rows, ids[rows], ids.dtype), batch).to_host()
    for b in (0, rows - 1):
        single = model.new_kv_cache()
        model.prefill([int(ids[b])], single)
        want = model.forward_one(int(ids[rows]), single).to_host()
        assert np.linalg.norm(step[b] - want) <= 1e-5 * np.linalg.norm(want)


@pytest.mark.parametrize("batch", [1, 3, 40])
@pytest.mark.parametrize("width,inner,vocab", [(768, 3072, 1031), (256, 1024, 300), (768, 256, 97)])
def test_a_cache_follows_the_sizes_of_the_model_that_uses_it(batch, width, inner, vocab):
    """n_inner and vocab_size are no sizes of a cache: one made by a model of others, smaller or larger, serves as the model's own does."""
    sizes = dict(n_positions=300, n_embd=width, n_layer=2, n_head=width // 64)
    cfg, other = Gpt2Config(vocab_size=vocab, n_inner=inner, **sizes), Gpt2Config(vocab_size=260, n_inner=512, **sizes)
    model = Gpt2Model.new(cfg, synth.random_weights(cfg, 0x5EED0A05, perturb=True))
    maker = Gpt2Model.new(other, synth.random_weights(other, 0x5EED0A06, perturb=True), Gpt2HipConfig(attn_item_keys=256))
    ids = synth.token_ids(batch * 10, 0x70C00A05, 90).reshape(batch, 10)
    got = []
    for cache in (model.new_kv_cache(batch), maker.new_kv_cache(batch)):
        if got:
            maker.prefill_batch(np.ascontiguousarray(ids), cache)
        steps = [model.prefill_batch(np.ascontiguousarray(ids[:, :9]), cache).to_host(), model.forward_one_batch(ids[:, 9], cache).to_host()]
        steps.append(model.decode_greedy_batch(cache, 5)[0])
        got.append(steps)
    for a, b in zip(*got):
        assert a.shape == b.shape
        # (steps in other forms: sums of at most 3072 terms in other orders)
        assert np.linalg.norm(a.astype(np.float64) - b) <= 1e-5 * np.linalg.norm(a)
