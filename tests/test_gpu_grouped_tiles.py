"""Products of rows sorted by the matrix they meet, in tiles of 16 and 32 rows: empty tiles, slots without a row, ragged
columns, one step of K for eight wavefronts and more."""
import numpy as np
import pytest

from helpers import DeviceArray, as_bf16, grouped_dev
from puppygrad_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,n,tiles", [(32, 8, [0]), (96, 66, [2, -1, 0, 2]), (544, 130, [1, 1, -1]), (1600, 256, [0, 1, 2, 0, 1, 2, -1])])
@pytest.mark.parametrize("silu_pair", [False, True])
@pytest.mark.parametrize("storage", ["f32", "bf16"])
@pytest.mark.parametrize("tile_rows", [16, 32])
def test_tiles(tile_rows, storage, silu_pair, k, n, tiles):
    rng = np.random.default_rng([tile_rows, k, n])
    x = rng.standard_normal((50, k)).astype(np.float32)
    w = (rng.standard_normal((3, n, k)) / np.sqrt(k)).astype(np.float32)
    if storage == "bf16":
        w = synth.round_bf16(w.reshape(-1)).reshape(w.shape)
    rows = rng.integers(0, 50, len(tiles) * tile_rows)
    rows[rng.random(rows.size) < 0.3] = -1
    dx = DeviceArray(x)
    got = grouped_dev(dx.ptr, rows.size, as_bf16(w) if storage == "bf16" else w, tiles, rows, tile_rows, silu_pair)
    dx.free()
    for t, group in enumerate(tiles):
        if group < 0:
            continue
        at = np.arange(t * tile_rows, (t + 1) * tile_rows)
        at = at[rows[at] >= 0]
        a, m = x[rows[at]].astype(np.float64), w[group].astype(np.float64)
        # f32 sums of K products: (K + 8) 2^-24 of the sum of their sizes
        c, err = a @ m.T, (k + 8) * 2.0 ** -24 * (np.abs(a) @ np.abs(m).T)
        if not silu_pair:
            assert (np.abs(got[at] - c) <= err).all()
            continue
        gate, up = c[:, 0::2], c[:, 1::2]
        want = gate / (1 + np.exp(-gate)) * up
        # (the slope of c / (1 + e^-c) is at most 1.1)
        bound = 1.2 * err[:, 0::2] * np.abs(up) + err[:, 1::2] * np.abs(gate) + err[:, 0::2] * err[:, 1::2] + 1e-6 * np.abs(want)
        assert (np.abs(got[at] - want) <= bound).all()
