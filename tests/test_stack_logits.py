"""The logits of one row of a prompt pass against those of several rows (another kernel), and tokens read from host
memory: calls of different lengths, and one of more tokens than a portion."""
import numpy as np
import pytest

import fazinex_util as U
from vkllama_amd import model as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,cap,dtype", [(64, 9.0, "float32"), (72, 30.0, "float32"),  # rows padded to 128
                                             (128, 2.0, "bfloat16"), (4160, 30.0, "bfloat16")])  # a second span
def test_one_row_of_logits(width, cap, dtype):
    cfg = U.config([U.attention(2, 1, 32, ff=96)], 321, width, cap=cap)
    m = M.CausalModel.create(cfg, U.weights(cfg, seed=width), dtype, 4200)
    rng = np.random.default_rng(width)
    # a normed row and a matrix of N(0, s): sums of `width` products with weights of 8 bits; bf16: the rows of several
    # are rounded to 2^-9 of themselves, each logit by no more than that of its sum of magnitudes, of which 1e-2 of the
    # largest logit is several times the spread
    bound = 1e-5 if dtype == "float32" else 1e-2
    for n in (3, 1, 40, 2):
        toks = rng.integers(0, 321, n).astype(np.uint32)
        many = m.forward_rows(toks, 0, np.arange(n)) if n > 1 else None
        one = m.forward_rows(toks, 0, [n - 1])
        if many is not None:
            assert np.abs(one[0] - many[-1]).max() < bound * np.abs(many[-1]).max(), n
    toks = rng.integers(0, 321, 4100).astype(np.uint32)
    whole = m.forward_rows(toks, 0, [4099])[0]
    m.forward_rows(toks[:4096], 0, [0])
    parts = m.forward_rows(toks[4096:], 4096, [3])[0]
    assert np.array_equal(whole, parts)
    m.close()
