"""Products of more than 64 rows on the bf16 matrix cores with f32 operands cut into three bf16 parts: every
tile shape at its edges, one to a few stages of K, whole tiles and cut K, each storage of the weights."""
import numpy as np
import pytest

from helpers import DeviceArray
from puppygrad_amd import Gpt2Config, Gpt2HipConfig, Gpt2Model, _lib, synth

pytestmark = pytest.mark.gpu


def ok(status):
    assert status == 0, _lib.load().pg_last_error_message().decode()


def within_f32_sums(got, x, w, b):
    """|error| <= (K + 8) 2^-24 sum |x w| + 2^-23 |result|: f32 sums of K exact products in any order, products
    right to 2^-25, the bias and (int8) the row scale each rounded once."""
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
    cfg = Gpt2Config(vocab_size=300, n_positions=512, n_embd=768, n_layer=1, n_head=12)
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
