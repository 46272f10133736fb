"""Weights read ahead by a launch's spare blocks (pg_ahead.h): which words, and the steps that do it."""
import ctypes
import subprocess
from pathlib import Path

import numpy as np
import pytest

import oracle
from helpers import assert_logits_close
from oracle import tarepel
from puppygrad_amd import Gpt2Config, Gpt2HipConfig, Gpt2Model, _lib, synth
from stack_helpers import Pair, check, rounded

CSRC = Path(__file__).resolve().parents[1] / "puppygrad_amd" / "csrc"
DIES, LINE = 8, 128
ROWS = 4  # HALF_ROWS
PROGRAM = """
#include <cstdio>
#include <cstdlib>
#include "pg_ahead.h"
// every word that the spare blocks, the first of them block `first` of its launch, read: die and place
int main(int, char** v) {
  pgk::Ahead a;
  a.matrix(1, nullptr, atoi(v[1]), atoi(v[2]), atoi(v[3]));
  a.blocks = atoi(v[4]);
  const int first = atoi(v[5]), threads = atoi(v[6]);
  for (int block = 0; block < a.blocks; ++block)
    for (int tid = 0; tid < threads; ++tid) {
      auto load = [&](unsigned at) { return printf("%d %u\\n", (first + block) % 8, at), at; };
      pgk::ahead_words(a, 1, block, first + block, tid, threads, load, [](const unsigned (&)[pgk::kAheadAtOnce]) {});
    }
}
"""


@pytest.fixture(scope="module")
def words_of(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("ahead")
    (tmp / "words.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{CSRC}", str(tmp / "words.cpp"), "-o", str(tmp / "words")], check=True)
    return lambda *args: np.array(subprocess.run([str(tmp / "words"), *map(str, args)], check=True, capture_output=True).stdout.split(),
                                  np.int64).reshape(-1, 2)


# rows one after the other, and slabs; spare blocks behind any number of others
@pytest.mark.parametrize("slabs,slab,group", [
    (1, 4096 * 3072, 4096 * 12), (1, 3200 * 4800, 3200 * 19), (1, 3200 * 6400, 3200 * 25), (1, 7296 * 1600, 7296 * 7), (1, 12, 4),
    (1, 128 * 8, 128), (1, 132 * 9, 132 * 2), (1, 64 * 1000, 64 * 3), (1, 5120 * 15, 5120 * 4), (1, 3200 * 8, 3200 * 8), (160, 1280 * 16, 40 * 16), (160, 5120 * 16, 24 * 16),
    (200, 1600 * 16, 32 * 16), (67, 72 * 16, 8 * 16), (3, 30000 * 16, 8 * 16)])
@pytest.mark.parametrize("blocks,first,threads", [(8, 0, 64), (64, 57, 512), (128, 20, 256)])
def test_every_line_of_a_group_is_read_once_by_its_own_die(words_of, slabs, slab, group, blocks, first, threads):
    got = words_of(slabs, slab, group, blocks, first, threads)
    want = {s * slab + at: g % DIES for s in range(slabs) for g in range(-(-slab // group))
            for at in range(g * group, min((g + 1) * group, slab), LINE)}
    assert len(got) == len(want) and {int(at): int(die) for die, at in got} == want


@pytest.mark.parametrize("width", [1088, 1216, 1280, 1408, 1600])
@pytest.mark.parametrize("rows", [17, 37, 50, 64, 65])
def test_groups_of_short_prompts_products_are_their_blocks(width, rows):
    f = _lib.load().pg_testing_half_ahead
    f.argtypes, f.restype = [ctypes.c_int32] * 5 + [ctypes.POINTER(ctypes.c_uint32)], None
    for in_f, out_f, resid in ((width, width, 1), (width, 4 * width, 0), (width, 3 * width, 0)):
        out = (ctypes.c_uint32 * 7)()
        f(rows, in_f, out_f, resid, 256, out)
        tile, _, mt, block_rows, slabs, slab, group = out
        if tile == ROWS and rows <= 16 * mt:
            assert (slabs, slab, group) == (in_f // 8, out_f * 16, block_rows * 16)
        else:
            assert slabs == 0


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


# (1280: attention reads 16 MB ahead, the norm 10; 1600: 26 and 15; 1024: 10 and none; 5, 16 and 65 tokens: on the far sides of the lines)
@pytest.mark.gpu
@pytest.mark.parametrize("C,storage,n", [(1024, 1, 50), (1280, 1, 5), (1280, 1, 16), (1280, 1, 17), (1280, 2, 37), (1280, 1, 64), (1280, 1, 65), (1600, 2, 17), (1600, 1, 64)])
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
