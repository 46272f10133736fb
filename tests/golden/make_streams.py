"""Writes tests/golden/streams.npz: the ids of sampled streams as the loaded library draws them.

The file in the repository was written with a library from before prompts had activations in cut form, attention on the
bf16 matrix cores and tiles of 16 rows for experts (pg_gemm_rows.hip, pg_attn_cut.hip, pg_moe.hip): a seed's stream goes on
drawing these ids.  Write it anew only with a change that is meant to change what a seed draws.

Run from the repo root, on a GPU:  python tests/golden/make_streams.py [file]
"""
import sys
import tempfile
from pathlib import Path

import numpy as np

ROOT = Path(__file__).resolve().parents[2]
sys.path.insert(0, str(ROOT))

from puppygrad_amd import Gpt2Config, Gpt2HipConfig, Gpt2Model, TextGenerationConfig, _lib, load_model, synth  # noqa: E402

VOCAB, NEW = 50257, 60
# model: prompts.  Draws over the whole row, among its likeliest ids (top_p) and behind a repeat penalty.
PROMPTS = {"f32-768": (12, 33, 64, 100, 150, 400), "bf16-768": (12, 33, 50, 100, 300), "int8-768": (12, 17, 40, 100, 400),
           "f32-1600": (640,), "movudra-768": (3, 20, 48, 60), "tarepel-768": (3, 20, 60)}
SAMPLINGS = (dict(temperature=1.0), dict(temperature=0.8), dict(temperature=1.1, top_p=0.9), dict(temperature=1.0, repeat_penalty=1.2))


def model(name):
    kind, width = name.split("-")
    width = int(width)
    if kind in ("movudra", "tarepel"):
        cfg = getattr(synth, kind + "_config")(width, 3)
        with tempfile.TemporaryDirectory() as tmp:
            synth.write_model_dir(tmp, cfg, synth.stack_weights(cfg, 0x5EED0B00))
            return load_model(tmp, Gpt2HipConfig(weight_storage=_lib.PG_STORE_BF16))
    cfg = Gpt2Config(vocab_size=VOCAB, n_positions=720, n_embd=width, n_layer=2, n_head=width // 64)
    store = {"f32": _lib.PG_STORE_F32, "bf16": _lib.PG_STORE_BF16, "int8": _lib.PG_STORE_INT8}[kind]
    return Gpt2Model.new(cfg, synth.random_weights(cfg, 0x5EED0B00, perturb=True), Gpt2HipConfig(weight_storage=store))


def streams(m, n):
    """[sampling][NEW] ids behind a prompt of n tokens."""
    ids = [int(t) for t in synth.token_ids(n, 0x70C00B00 + n, VOCAB)]
    return np.array([m.stream_token_ids_with_stats(ids, TextGenerationConfig(NEW, seed=7 + i, **kw))[0][n:]
                     for i, kw in enumerate(SAMPLINGS)], np.uint16)


if __name__ == "__main__":
    out = {}
    for name, prompts in PROMPTS.items():
        m = model(name)
        for n in prompts:
            out[f"{name}.{n}"] = streams(m, n)
        print(name, flush=True)
    np.savez_compressed(sys.argv[1] if len(sys.argv) > 1 else Path(__file__).resolve().parent / "streams.npz", **out)
