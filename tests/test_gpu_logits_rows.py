"""Logits over large vocabularies: rows of the output matrix taken in turns by fewer blocks than there are rows."""
import numpy as np
import pytest

from puppygrad_amd import Gpt2Config, Gpt2HipConfig, Gpt2Model, _lib, synth
from stack_helpers import check
from test_gpu_movudra import Pair, config, mamba, weights

pytestmark = pytest.mark.gpu
STORAGES = {"f32": _lib.PG_STORE_F32, "bf16": _lib.PG_STORE_BF16, "int8": _lib.PG_STORE_INT8}


# the last size without turns and the first with them, a last turn of one row, three turns and a part
@pytest.mark.parametrize("vocab", [16376, 16384, 16385, 27001])
@pytest.mark.parametrize("storage", STORAGES)
def test_gpt2_rows_do_not_depend_on_the_vocabulary(vocab, storage):
    """The first and the last rows alone, too few of them for turns, give the same bits."""
    few, ids = 4500, synth.token_ids(9, 0x70C00A00, 100)

    def logits(w, rows):
        cfg = Gpt2Config(vocab_size=rows, n_positions=32, n_embd=192, n_layer=1, n_head=3)
        model = Gpt2Model.new(cfg, w, Gpt2HipConfig(weight_storage=STORAGES[storage]))
        return np.asarray(model.prefill(ids, model.new_kv_cache()).to_host()).reshape(-1)

    w = synth.random_weights(Gpt2Config(vocab_size=vocab, n_positions=32, n_embd=192, n_layer=1, n_head=3), 0x5EED0A00, perturb=True)
    got, table = logits(w, vocab), np.reshape(w.wte, (vocab, 192))
    w.wte = table[:few]
    np.testing.assert_array_equal(got[:few], logits(w, few))
    w.wte = np.concatenate([table[:100], table[-few:]])
    np.testing.assert_array_equal(got[-few:], logits(w, few + 100)[100:])


# (width 2304: more chunks to a row than are asked for ahead, in both storages)
@pytest.mark.parametrize("vocab,width", [(16385, 48), (24600, 136), (16401, 2304)])
@pytest.mark.parametrize("storage", ["f32", "bf16"])
def test_stack_rows_match_the_oracle(tmp_path, vocab, width, storage):
    cfg = config([mamba()], width=width, vocab=vocab)
    p = Pair(tmp_path, cfg, weights(cfg, 29), STORAGES[storage])
    ids = p.ids(12)
    check(p.portions(ids, [8, 1, 1, 1, 1]), p.ref.run(ids))
