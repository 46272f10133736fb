"""Prompts whose last layer goes on with the rows that logits are wanted of: both sides of where that begins, what the cache
holds afterwards, and the steps that follow."""
import numpy as np
import pytest

import oracle
import test_gpu_tarepel as other
from helpers import assert_logits_close
from oracle import movudra, tarepel
from puppygrad_amd import Gpt2Config, Gpt2HipConfig, Gpt2Model, synth
from stack_helpers import Pair, check
from test_gpu_movudra import MIXED, config, delta, latent, mamba, moe, weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", [0, 1, 2], ids=["f32", "bf16", "int8"])
@pytest.mark.parametrize("B,n", [(1, 127), (1, 128), (1, 300), (2, 63), (2, 64), (3, 70), (8, 33), (15, 8), (16, 8),
                                  (32, 7), (32, 9), (33, 9)])
def test_prompts(B, n, storage):
    cfg = Gpt2Config(vocab_size=131, n_positions=304, n_embd=128, n_layer=2, n_head=2)
    w = synth.random_weights(cfg, 0x5EED0D00, perturb=True)
    ids = synth.token_ids(B * n, 0x70C00D00 + n, cfg.vocab_size).reshape(B, n)
    model = Gpt2Model.new(cfg, w, Gpt2HipConfig(weight_storage=storage))
    ref = oracle.Model(cfg, synth.bf16_rounded(w) if storage == 1 else w, oracle.rust_config(8, quantized_weights=int(storage == 2)))
    cache = model.new_kv_cache(B)
    got = model.prefill_batch(ids, cache).to_host() if B > 1 else model.prefill(ids[0], cache).to_host()[None]
    some = sorted({0, B // 2, B - 1})
    rcs = {b: ref.new_kv_cache() for b in some}
    for b in some:
        assert_logits_close(got[b], ref.prefill(ids[b], rcs[b]))
        for kv in (0, 1):
            np.testing.assert_allclose(cache.read_layer(1, kv, b)[:, :n], rcs[b].read_layer(1, kv)[:, :n], atol=2e-5, rtol=1e-4)
    nxt = ids[:, 0]
    got = model.forward_one_batch(nxt, cache).to_host() if B > 1 else model.forward_one(int(nxt[0]), cache).to_host()[None]
    for b in some:
        assert_logits_close(got[b], ref.forward_one(int(nxt[b]), rcs[b]))


# (a last layer with experts, with a dense feed-forward and with none; one of parallel sublayers, of two kinds, without its MLP, and
# with one too wide for a launch together with the mixers)
LAST = {"experts": config([delta(), mamba(mlp=moe(5, 3, 20))]), "dense": MIXED, "none": config([mamba(), latent()]),
        "parallel": other.config([other.gla(), other.parallel()]), "gla": other.config([other.parallel(), other.gla()]),
        "no-mlp": other.config([other.gla(), other.parallel(ff=None)]), "wide": other.config([other.parallel(ff=16300)])}


@pytest.fixture(scope="module", params=LAST)
def pair(request, tmp_path_factory):
    cfg = LAST[request.param]
    orc, make = (movudra, weights) if cfg["architecture"] == "Movudra" else (tarepel, other.weights)
    return Pair(orc, tmp_path_factory.mktemp("last"), cfg, make(cfg, 17))


# (5e-5: what models of six layers are held to, whichever rows are wanted)
@pytest.mark.parametrize("n,wanted", [(40, []), (3, [2]), (4, [3]), (4, [0]), (7, [2, 5]), (8, [2, 5]), (131, range(99, 131)),
                                      (127, range(95, 127)), (140, range(0, 132, 4)),
                                      (2047, [1, 2046]), (2047, [1, 7, 2046]), (2048, [1, 2046]), (2048, [1, 7, 2046])])
def test_wanted_rows(pair, n, wanted):
    ids, wanted = pair.ids(n + 2, seed=n), list(wanted)
    want = pair.ref.run(ids)
    cache = pair.dev.new_kv_cache()
    got = pair.dev.extend(ids[:n], cache, wanted)
    if wanted:
        check(got.to_host().reshape(len(wanted), -1), want[wanted], 5e-5)
    check(pair.dev.extend(ids[n:], cache, [0, 1]).to_host(), want[n:], 5e-5)


@pytest.mark.parametrize("B,n", [(2, 3), (2, 4), (5, 21), (32, 5), (33, 5), (32, 63), (32, 64)])
def test_batches(pair, B, n):
    ids = np.array([pair.ids(n, seed=100 + b) for b in range(B)], np.uint32)
    cache = pair.dev.new_kv_cache(B)
    got = pair.dev.prefill_batch(ids, cache).to_host()
    for b in sorted({0, B // 2, B - 1}):
        check(got[b], pair.ref.run([int(t) for t in ids[b]])[-1:], 5e-5)


@pytest.mark.parametrize("ff", [40, None])
def test_the_last_row_is_booked_as_a_step_books_it(tmp_path, ff):
    """Both products back to the residual are one launch: the MLP's, where there is one."""
    cfg = other.config([other.parallel(ff=ff)])
    dev = Pair(tarepel, tmp_path, cfg, other.weights(cfg, 19)).dev
    prof = dev.prefill_profiled([3, 1, 4, 1, 5], dev.new_kv_cache())[1]
    assert (prof.attention_projection == 0) == (ff is not None) and (prof.mlp_projection > 0) == (ff is not None)
