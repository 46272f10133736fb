"""Products of more than 64 rows, most of them on the bf16 matrix cores with f32 operands cut into three bf16
parts: the planner's choice through the public entry points, and every tile of those kernels by name at its edges,
with one to a few stages of K, whole and cut, against each storage of the weights."""
import ctypes

import numpy as np
import pytest

from helpers import DeviceArray, as_bf16, grouped_dev, product_dev
from puppygrad_amd import Gpt2Config, Gpt2HipConfig, Gpt2Model, _lib, synth

pytestmark = pytest.mark.gpu


def ok(status):
    assert status == 0, _lib.load().pg_last_error_message().decode()


def within_f32_sums(got, x, w, b):
    """|error| <= (K + 8) 2^-24 sum |x w| + 2^-23 |result|: f32 sums of K products in any order, products
    right to 2^-24, the bias and (int8) the row scale each rounded once."""
    x, w = x.astype(np.float64), w.astype(np.float64)
    want = x @ w.T + b
    bound = (x.shape[1] + 8) * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T) + 2.0 ** -23 * np.abs(want)
    assert (np.abs(got - want) <= bound).all(), f"{(np.abs(got - want) / bound).max():.2f} of the bound"


def operands(rows, k, n):
    rng = np.random.default_rng([rows, k, n])
    x = (rng.standard_normal((rows, k)) * 10.0 ** rng.uniform(-3, 3, (rows, k))).astype(np.float32)
    w = (rng.standard_normal((n, k)) * 10.0 ** rng.uniform(-3, 1, (n, k))).astype(np.float32)
    return x, w, rng.standard_normal(n).astype(np.float32)


# one to five stages of 16 columns with ragged rows and columns; deep K on few tiles (cut); 256-row tiles
@pytest.mark.parametrize("rows,k,n", [(65, 16, 2560), (127, 32, 1281), (129, 48, 1300), (65, 64, 1412), (200, 80, 777),
                                      (70, 2048, 1284), (257, 4096, 640), (513, 144, 2562), (600, 1600, 1600), (1025, 96, 1024)])
def test_f32_rows(rows, k, n):
    x, w, b = operands(rows, k, n)
    got = np.empty((rows, n), np.float32)
    ok(_lib.load().pg_op_dense(0, _lib.f32p(x.reshape(-1)), rows, k, n, _lib.f32p(w.reshape(-1)), _lib.f32p(b),
                               _lib.f32p(got.reshape(-1))))
    within_f32_sums(got, x, w, b)


# 33 to 64 rows: the small-batch kernel with two tiles of rows, one step of 64 columns for eight wavefronts and
# more, K cut over blocks; then one to three stages of 32 columns upward; the last shape has 512 tiles of 128 x 256
@pytest.mark.parametrize("rows,k,n", [(33, 64, 100), (37, 1280, 3840), (64, 576, 5120), (50, 5120, 1280), (65, 64, 1600), (129, 128, 1537), (191, 192, 800), (600, 320, 1031), (2000, 64, 8000)])
def test_int8_rows(rows, k, n):
    x, w, b = operands(rows, k, n)
    q = np.random.default_rng(n).integers(-127, 128, (n, k)).astype(np.int8)
    scales = np.abs(w[:, 0]) + np.float32(1e-3)
    dx, dq, ds, db, dy = DeviceArray(x), DeviceArray(q, dtype=np.int8), DeviceArray(scales), DeviceArray(b), DeviceArray(np.zeros((rows, n)))
    ok(_lib.load().pg_op_quantized_dense_dev(0, None, dx.ptr, rows, k, n, dq.ptr, ds.ptr, db.ptr, dy.ptr))
    got = dy.download()
    within_f32_sums(got, x, q.astype(np.float64) * scales[:, None].astype(np.float64), b)
    for d in (dx, dq, ds, db, dy):
        d.free()


# a short prompt (64-row tiles, cut K), a ragged one, and batches with 128-row and 128 x 256 tiles
@pytest.mark.parametrize("batch,n", [(1, 65), (1, 333), (5, 200), (16, 512)])
def test_bf16_rows_give_what_f32_rows_of_the_same_values_give(batch, n):
    # (two layers: behind the last one's keys and values a prompt goes on with its last row)
    cfg = Gpt2Config(vocab_size=300, n_positions=512, n_embd=768, n_layer=2, n_head=12)
    w = synth.bf16_rounded(synth.random_weights(cfg, 0x5EED0900, perturb=True))
    ids = synth.token_ids(batch * n, 0x70C00900 + n, cfg.vocab_size).reshape(batch, n)
    got = []
    for storage in (_lib.PG_STORE_BF16, _lib.PG_STORE_F32):
        model = Gpt2Model.new(cfg, w, Gpt2HipConfig(weight_storage=storage))
        cache = model.new_kv_cache(batch)
        got.append(np.atleast_2d(model.prefill_batch(ids, cache).to_host() if batch > 1 else model.prefill(ids[0], cache).to_host()))
    # (both multiply the same values: what differs is the order of f32 sums of at most 3072 terms)
    assert np.linalg.norm(got[0] - got[1]) <= 1e-5 * np.linalg.norm(got[1])


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, np.float32(3.4e38)])
def test_values_past_bf16_meet_the_weights_as_in_f32(value):
    """3.4e38 rounds to an infinite bf16: the tile is computed again in plain f32 arithmetic."""
    x, w, b = operands(300, 256, 1300)
    x = np.clip(x, -10, 10)
    w[:] = np.sign(w) * 0.25
    x[17, 3] = value
    got = np.empty((300, 1300), np.float32)
    ok(_lib.load().pg_op_dense(0, _lib.f32p(x.reshape(-1)), 300, 256, 1300, _lib.f32p(w.reshape(-1)), _lib.f32p(b),
                               _lib.f32p(got.reshape(-1))))
    others = np.arange(300) != 17
    within_f32_sums(got[others], x[others], w, b)
    want = x[17].astype(np.float64) @ w.astype(np.float64).T
    np.testing.assert_array_equal(np.isnan(got[17]), np.isnan(want))
    np.testing.assert_array_equal(np.isposinf(got[17]), np.isposinf(want))
    if np.isfinite(value):
        np.testing.assert_allclose(got[17], want, rtol=1e-6)


# ---- the tiles by name -------------------------------------------------------------------------
F32_TILES, BYTE_TILES = [(64, 128), (128, 128), (128, 128, 1), (256, 128)], [(64, 128), (128, 128), (128, 128, 1), (128, 256)]
STORED = {"f32": F32_TILES, "bf16": BYTE_TILES, "int8": BYTE_TILES}
TILES = [(s, t) for s, tiles in STORED.items() for t in tiles]
ONE_SUM = [(s, t) for s in ("bf16", "int8") for t in ((128, 128, 1), (128, 256))]


def stored_rows(w, storage):
    """(matrix as it is handed over, scales, the values it stands for)"""
    if storage == "f32":
        return w, None, w.astype(np.float64)
    if storage == "bf16":
        w = synth.round_bf16(w.reshape(-1)).reshape(w.shape)
        return as_bf16(w), None, w.astype(np.float64)
    q = np.random.default_rng(w.shape).integers(-127, 128, w.shape).astype(np.int8)
    scales = np.abs(w[:, 0]) + np.float32(1e-3)
    return q, scales, q * scales[:, None].astype(np.float64)


# one stage of K and the first few (32 columns; f32 rows 16), ragged rows and columns
@pytest.mark.parametrize("rows,k,n", [(65, 32, 129), (1, 64, 31), (127, 96, 257), (300, 160, 385), (257, 224, 640)])
@pytest.mark.parametrize("storage,tile", TILES)
def test_tiles_at_their_edges(storage, tile, rows, k, n):
    for k in ((k, k - 16) if storage == "f32" else (k,)):
        x, w, b = operands(rows, k, n)
        stored, scales, values = stored_rows(w, storage)
        within_f32_sums(product_dev(x, stored, b, scales, tile=tile), x, values, b)


@pytest.mark.parametrize("parts", [2, 5, 8])
@pytest.mark.parametrize("storage,tile", TILES)
def test_tiles_with_k_cut(storage, tile, parts):
    for rows, k, n in ((65, 256, 132), (200, 1088, 388)):
        x, w, b = operands(rows, k, n)
        stored, scales, values = stored_rows(w, storage)
        within_f32_sums(product_dev(x, stored, b, scales, tile=tile, parts=parts, ws_floats=parts * rows * n), x, values, b)


def one_sided(shape, seed, top):
    """Values whose three bf16 parts are all of the value's sign and nearly as large as they can be: 2^e (1 + a 2^-7
    + b 2^-8 + c 2^-17), so that every one of the products of parts adds to the same side."""
    r = np.random.default_rng(seed)
    m = 1.0 + r.integers(0, 32, shape) * 2.0 ** -7 + r.uniform(0.8, 0.99, shape) * 2.0 ** -8
    x = (m * 2.0 ** r.integers(-top, top + 1, shape)).astype(np.float32)
    return ((x.view(np.uint32) & ~np.uint32(0x7f)) | r.integers(0x30, 0x40, shape).astype(np.uint32)).view(np.float32)


@pytest.mark.parametrize("storage,tile", TILES)
def test_every_product_of_parts_counts(storage, tile):
    """With one sign throughout, leaving out lo or mid mid would show as at least 2^-18 of the result; what the
    six products leave out is 2^-24 of it, and each of the 2 K / 16 groups of hi hi products rounds the sum by at
    most 2^-24, the sum of the small products the same of a 2^-7th, two last additions once each."""
    for k in (32, 64):
        x, w = one_sided((160, k), 1, 1), one_sided((200, k), 2, 1)
        stored, scales, values = stored_rows(w, storage)
        if storage == "int8":
            stored = (64 + np.abs(stored) // 2).astype(np.int8)
            values = stored * scales[:, None].astype(np.float64)
        got = product_dev(x, stored, None, scales, tile=tile).astype(np.float64)
        want = x.astype(np.float64) @ values.T
        groups = k / 8 * (3 if (storage, tile) in ONE_SUM else 1)
        assert (np.abs(got - want) <= (1 + groups * 1.05 + 3) * 2.0 ** -24 * want).all()


@pytest.mark.parametrize("storage,tile", [c for c in TILES if c not in ONE_SUM])
def test_small_products_have_a_sum_of_their_own(storage, tile):
    """The 2-norm of the error over the result's: K / 8 roundings of the running sum s, whose mean square is k / K
    of the result's; a rounding is uniform in a unit of the last place, 2^-23 |s| times a square mean of 0.541.
    With the small products in the same sum (twelve or six roundings per 16 columns instead of two) it is 2.4 or 1.7 times this."""
    rows, k, n = 700, 1600, 520
    r = np.random.default_rng(8)
    x, w = r.standard_normal((rows, k)).astype(np.float32), r.standard_normal((n, k)).astype(np.float32)
    stored, scales, values = stored_rows(w, storage)
    want = x.astype(np.float64) @ values.T
    err = product_dev(x, stored, None, scales, tile=tile) - want
    expected = np.sqrt(k / 8 / 2 * 0.541 / 12) * 2.0 ** -23
    assert np.linalg.norm(err) <= 1.25 * expected * np.linalg.norm(want)
    # rows that are nearly alike: what their errors have in common is what the mean of independent ones is (three
    # times that), and what the roundings downward leave
    common = r.standard_normal(k)
    x = (common + 0.05 * r.standard_normal((rows, k))).astype(np.float32)
    want = x.astype(np.float64) @ values.T
    err = product_dev(x, stored, None, scales, tile=tile) - want
    size = np.sqrt((want ** 2).mean())
    assert np.sqrt((err.mean(0) ** 2).mean()) <= (3 * expected / np.sqrt(rows) + 3e-8) * size


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, np.float32(3.4e38)])
@pytest.mark.parametrize("storage,tile,parts", [(s, t, p) for s, t in TILES for p in (1, 3)])
def test_tiles_with_values_past_bf16(storage, tile, parts, value):
    x, w, b = operands(150, 192, 260)
    x = np.clip(x, -10, 10)
    w[:] = np.sign(w) * 0.25
    stored, scales, values = stored_rows(w, storage)
    if storage == "int8":
        stored, scales = np.sign(stored) + (stored == 0).astype(np.int8), np.full(260, 0.25, np.float32)
        values = stored * 0.25
    x[17, 3] = value
    got = product_dev(x, stored, b, scales, tile=tile, parts=parts, ws_floats=parts * 150 * 260 if parts > 1 else 0)
    others = np.arange(150) != 17
    within_f32_sums(got[others], x[others], values, b)
    want = x[17].astype(np.float64) @ values.T
    np.testing.assert_array_equal(np.isnan(got[17]), np.isnan(want))
    np.testing.assert_array_equal(np.isposinf(got[17]), np.isposinf(want))
    np.testing.assert_array_equal(np.isneginf(got[17]), np.isneginf(want))
    if np.isfinite(value):
        np.testing.assert_allclose(got[17], want, rtol=1e-6)


@pytest.mark.parametrize("storage,tile_rows", [("bf16", 32), ("bf16", 64), ("bf16", 128), ("f32", 32), ("f32", 64)])
def test_grouped_rows_past_four_gigabytes(storage, tile_rows):
    """Experts' slots (and the rows they take) whose offsets need more than 32 bits: only the last two tiles hold any."""
    lib, k, n = _lib.load(), 16000, 96
    slots = (1 << 32) // (4 * k) // 128 * 128 + 384
    first = slots - 2 * tile_rows
    assert first * k * 4 >= 1 << 32
    x, w, _ = operands(2 * tile_rows, k, 2 * n)
    stored, _, values = stored_rows(w, storage)
    a = ctypes.c_void_p()
    ok(lib.pg_device_alloc(0, slots * k * 4, ctypes.byref(a)))
    try:
        ok(lib.pg_device_upload(0, ctypes.c_void_p(a.value + first * k * 4), x.ctypes.data_as(ctypes.c_void_p), x.nbytes))
        tiles = np.full(slots // tile_rows, -1, np.int32)
        tiles[-2:] = (1, 0)
        got = grouped_dev(a, slots, stored.reshape(2, n, k), tiles, None, tile_rows)[first:]
        within_f32_sums(got[:tile_rows], x[:tile_rows], values[n:], 0.0)
        within_f32_sums(got[tile_rows:], x[tile_rows:], values[:n], 0.0)
        # few slots that take those rows, in another order
        order = np.random.default_rng(3).permutation(2 * tile_rows)
        got = grouped_dev(a, 2 * tile_rows, stored.reshape(2, n, k), [0, 1], first + order, tile_rows)
        within_f32_sums(got[:tile_rows], x[order[:tile_rows]], values[:n], 0.0)
        within_f32_sums(got[tile_rows:], x[order[tile_rows:]], values[n:], 0.0)
    finally:
        ok(lib.pg_device_free(0, a))
