"""The operands of attn_parts.py show every product of the parts: all six are within the bound, none may be left out."""
import numpy as np
import pytest

import attn_parts


@pytest.mark.parametrize("which", ["scores", "weights"])
def test_no_product_may_be_left_out(which):
    qkv = attn_parts.operands(which)
    want = attn_parts.exact(qkv)

    def error(**chosen):
        got, size = attn_parts.attention(qkv, **chosen)
        return (np.abs(got - want) / (attn_parts.BOUND[which] * size)).max()

    assert error() < 0.25
    for left_out in attn_parts.PRODUCTS:
        assert error(**{which: [p for p in attn_parts.PRODUCTS if p != left_out]}) > 2.0, left_out
