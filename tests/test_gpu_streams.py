"""What a seed draws stays what it was: streams over rows of 50257 logits, where a logit's last bit decides between ids
whose ranks lie next to each other, against the ids of a library from before prompts had other kernels
(golden/make_streams.py)."""
import sys

import numpy as np
import pytest

from helpers import GOLDEN

sys.path.insert(0, str(GOLDEN))
import make_streams  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", make_streams.PROMPTS)
def test_a_seeds_stream_is_what_it_was(name):
    want, m = np.load(GOLDEN / "streams.npz"), make_streams.model(name)
    for n in make_streams.PROMPTS[name]:
        np.testing.assert_array_equal(make_streams.streams(m, n), want[f"{name}.{n}"], err_msg=f"{name}, prompt of {n}")
