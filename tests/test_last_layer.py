"""The last layer of a prompt pass that is asked for its last row only (the step's layer behind what is kept of the other
tokens) against the operators over all rows."""
import numpy as np
import pytest

import fazinex_util as Z
import fuzuvik_util as V
from vkllama_amd import model as M

pytestmark = pytest.mark.gpu

SHARED = Z.attention(4, 2, 32, q_temp=(0.2, 16), ff=96)
LATENT = Z.latent(4, 24, 40, 48, ff=104)  # sizes with padding on every side
CHUNKED = V.attention(4, 2, 40, 24, rot=24, size=50, v_mix=True, ff=104)
DELTA = V.delta(2, 2, 32, 32, ff=96)


# each mixer that can leave outputs out as the last layer, by itself, repeated, and behind a recurrence; one that cannot
@pytest.mark.parametrize("util,layers,loop", [(Z, [SHARED, LATENT], None), (Z, [LATENT, SHARED], None), (Z, [LATENT], (0, 1, 2)),
                                              (Z, [Z.attention(2, 2, 32)], None), (V, [CHUNKED, DELTA, CHUNKED], None),
                                              (V, [CHUNKED, DELTA], None)])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_last_row_equals_the_operators(util, layers, loop, dtype):
    cfg = Z.config(layers, 321, 72, loop=loop) if util is Z else V.config(layers, 321, 72)
    w = util.weights(cfg, seed=3)
    ms = [M.CausalModel.create(cfg, w, dtype, 512) for _ in range(2)]
    for m, fused in zip(ms, (0, 1)):
        m.set_option("fused_decode", fused)
    rng = np.random.default_rng(7)
    # fp32: sums of a few hundred products in another order; bf16: rows rounded to 2^-9 of themselves where the step
    # keeps them in fp32, of the largest logit several times what a few such roundings in a row give
    bound = 2e-5 if dtype == "float32" else 3e-2
    pos = 0
    for n in (2, 17, 1, 64, 130, 3):
        toks = rng.integers(0, 321, n).astype(np.uint32)
        a, b = (m.forward(toks, pos) for m in ms)
        pos += n
        assert np.abs(a).max() > 0
        assert np.abs(a - b).max() <= bound * np.abs(a).max(), n
    # rows besides the last one take the operators
    toks = rng.integers(0, 321, 9).astype(np.uint32)
    a, b = (m.forward_rows(toks, pos, [2, 8]) for m in ms)
    assert np.abs(a - b).max() <= bound * np.abs(a).max()
    for m in ms:
        m.close()


def test_arguments_are_checked(dev):
    from vkllama_amd import stack
    assert stack.lib().vkl_stack_layer_step(None, 0, None, 0, dev.stream) == 1
