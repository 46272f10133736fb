"""Experts behind a router whose product is cut along K: routing adds the raw parts (pg_moe.hip).  Widths, storages, numbers of
experts and rows on both sides of where it does, against the float64 oracle; with K not cut, and a row of experts padded."""
import numpy as np
import pytest

import oracle.movudra as orc
from puppygrad_amd import _lib, synth
from stack_helpers import Pair, check, rounded

pytestmark = pytest.mark.gpu
BF16, F32 = _lib.PG_STORE_BF16, _lib.PG_STORE_F32


def model(tmp_path, width, experts, top, storage, ff=32):
    layer = {"type": "channel_delta", "mixer": {"heads": 2, "kv_heads": 2, "dim": 16, "vdim": 16, "conv": 2},
             "mlp": {"kind": "moe", "router": {"experts": experts, "top": top}, "expert": {"ff": ff}}}
    cfg = {"architecture": "Movudra", "vocab": 97, "width": width, "norm": {"eps": 1e-6}, "layers": [layer]}
    g, w = np.random.default_rng([width, experts]), {}
    for name, shape in synth.stack_tensor_shapes(cfg, (8, 8)).items():
        last = name.split(".")[-1]
        scale = 1.0 if last in ("embed", "dt_bias", "A_log") else 3.0 / np.sqrt(shape[-1]) if last == "router" else 1.0 / np.sqrt(shape[-1])
        w[name] = 1.0 + 0.2 * g.standard_normal(shape) if last.startswith("norm") else scale * g.standard_normal(shape)
    return Pair(orc, tmp_path, cfg, rounded(w), storage)


# width 96: no K is cut; 70 and 130 experts: two and three logits a lane, rows padded to 72 and 132
@pytest.mark.parametrize("width,experts,top,storage", [(96, 8, 2, BF16), (768, 8, 2, BF16), (768, 8, 2, F32), (768, 64, 4, BF16), (768, 70, 3, BF16),
                                                       (768, 70, 3, F32), (1024, 130, 2, BF16)])
def test_batches_and_prompts(tmp_path, width, experts, top, storage):
    p = model(tmp_path, width, experts, top, storage)
    # (17 rows and more: a wavefront has a second row, 33 and more a third; rows past 64 leave the 32-row kernel)
    for batch in (2, 16, 17, 33, 64, 65):
        ids = np.array([p.ids(3, seed=7 * batch + b) for b in range(batch)], np.uint32)
        cache = p.dev.new_kv_cache(batch)
        got = [p.dev.prefill_batch(np.ascontiguousarray(ids[:, :1]), cache).to_host().reshape(batch, -1),
               p.dev.forward_one_batch(ids[:, 1], cache).to_host(), p.dev.forward_one_batch(ids[:, 2], cache).to_host()]
        for b in {0, 1, 15, 16, batch // 2, batch - 1} & set(range(batch)):
            check(np.stack([g[b] for g in got]), p.ref.run(ids[b]), what=f"sequence {b} of {batch}")
    for n in (2, 16, 33, 64, 127, 128, 129):  # (up to 128 rows one block routes)
        ids = p.ids(n, seed=n)
        check(p.portions(ids, [n]), p.ref.run(ids), what=f"prompt of {n}")
