"""Weights read ahead by a launch's spare blocks (pg_ahead.h): which words, and the steps that do it."""
import subprocess
from pathlib import Path

import numpy as np
import pytest

import oracle
from helpers import assert_logits_close
from oracle import tarepel
from puppygrad_amd import Gpt2Config, Gpt2HipConfig, Gpt2Model, synth
from stack_helpers import Pair, check, rounded

CSRC = Path(__file__).resolve().parents[1] / "puppygrad_amd" / "csrc"
DIES, LINE = 8, 128
PROGRAM = """
#include <cstdio>
#include <cstdlib>
#include "pg_ahead.h"
int main(int, char** v) {
  pgk::Ahead a;
  a.matrix(1, nullptr, atoi(v[1]), atoi(v[2]), atoi(v[3]));
  for (unsigned die = 0; die < pgk::kDies; ++die)
    for (unsigned w = 0; w < a.words[1]; ++w) {
      unsigned at;
      if (pgk::ahead_word(a, 1, die, w, &at)) printf("%u %u\\n", die, at);
    }
}
"""


@pytest.fixture(scope="module")
def words_of(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("ahead")
    (tmp / "words.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", f"-I{CSRC}", str(tmp / "words.cpp"), "-o", str(tmp / "words")], check=True)
    return lambda *args: np.loadtxt(subprocess.run([str(tmp / "words"), *map(str, args)], check=True, capture_output=True,
                                                   text=True).stdout.splitlines(), dtype=np.int64).reshape(-1, 2)


@pytest.mark.parametrize("row,rows,group", [(4096, 3072, 12), (3200, 4800, 19), (3200, 6400, 25), (7296, 1600, 7), (4, 3, 1),
                                            (128, 8, 1), (132, 9, 2), (5120, 15, 4), (64, 1000, 3), (3200, 8, 8)])
def test_every_line_of_a_group_is_read_by_its_own_die(words_of, row, rows, group):
    got = words_of(1, row * rows, row * group)
    assert (got[:, 1] % 4 == 0).all() and (got[:, 1] + 4 <= row * rows).all()
    assert len(np.unique(got[:, 1])) == len(got)
    size = row * group
    for g in range(0, -(-rows // group)):
        first, last = g * size, min((g + 1) * size, row * rows)
        mine = got[got[:, 1] // size == g]
        assert (mine[:, 0] == g % DIES).all()
        np.testing.assert_array_equal(np.sort(mine[:, 1]), np.arange(first, last, LINE))


# (1408: f32 rows of c_attn 23.8 MB, c_fc beyond what is read ahead; 1600: bf16 rows 15.4 and 20.5 MB)
@pytest.mark.gpu
@pytest.mark.parametrize("C,storage,B", [(1408, 0, 2), (1408, 0, 16), (1600, 1, 3), (1600, 1, 32)])
def test_batched_steps_that_read_ahead(C, storage, B):
    cfg = Gpt2Config(vocab_size=97, n_positions=16, n_embd=C, n_layer=2, n_head=C // 64)
    w = synth.random_weights(cfg, 0x5EED0C00 + C, perturb=True)
    ids = synth.token_ids(B * 3, 0x70C00C00 + B, cfg.vocab_size).reshape(B, 3)
    model = Gpt2Model.new(cfg, w, Gpt2HipConfig(weight_storage=storage))
    ref = oracle.Model(cfg, synth.bf16_rounded(w) if storage else w, oracle.rust_config(8))
    cache = model.new_kv_cache(B)
    model.prefill_batch(ids, cache)
    nxt = ids[:, 0]
    for _ in range(2):
        got = model.forward_one_batch(nxt, cache).to_host()
    for b in sorted({0, B // 2, B - 1}):
        rc = ref.new_kv_cache()
        ref.prefill(ids[b], rc)
        for _ in range(2):
            want = ref.forward_one(int(nxt[b]), rc)
        assert_logits_close(got[b], want)


# (1280: attention reads 16 MB ahead, the norm 10; 1600: 26 and 15; 1024: 10 and none)
@pytest.mark.gpu
@pytest.mark.parametrize("C,storage,n", [(1024, 1, 50), (1280, 1, 5), (1280, 2, 37), (1280, 1, 64), (1280, 1, 65), (1600, 2, 17), (1600, 1, 64)])
def test_prompts_that_read_ahead(C, storage, n):
    cfg = Gpt2Config(vocab_size=97, n_positions=72, n_embd=C, n_layer=3, n_head=C // 64)
    w = synth.random_weights(cfg, 0x5EED0C02 + C, perturb=True)
    ids = synth.token_ids(n, 0x70C00C02 + n, cfg.vocab_size)
    model = Gpt2Model.new(cfg, w, Gpt2HipConfig(weight_storage=storage))
    ref = oracle.Model(cfg, synth.bf16_rounded(w) if storage == 1 else w, oracle.rust_config(8, quantized_weights=int(storage == 2)))
    cache, rc = model.new_kv_cache(), ref.new_kv_cache()
    assert_logits_close(model.prefill(ids, cache).to_host(), ref.prefill(ids, rc))


@pytest.mark.gpu
def test_stack_step_that_reads_ahead(tmp_path):
    cfg = synth.tarepel_config(1600, 3, vocab=61)
    p = Pair(tarepel, tmp_path, cfg, rounded(dict(synth.stack_weights(cfg, 0x5EED0C01))))
    ids, cache, state = p.ids(5), p.dev.new_kv_cache(), p.ref.new_state()
    p.dev.prefill(ids[:3], cache)
    p.ref.run(ids[:3], state)
    for t in ids[3:]:
        check(p.dev.forward_one(t, cache).to_host(), p.ref.step(t, state))
