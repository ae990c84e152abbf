"""The end of a prompt pass on the launches of a step's phases, against the operators it takes the place of."""
import numpy as np
import pytest

from vkllama_amd import model as M

pytestmark = pytest.mark.gpu

BASE = dict(dim=256, n_layers=3, n_heads=4, ffn=704, vocab=1024, maxlen=96, eps=1e-5, wtype=8)


# both formats, heads of 64 and 128; one layer (the residual row is the embedding's); rows beyond 4096 and 8192 values
@pytest.mark.parametrize("cfg", [BASE, dict(BASE, wtype=1), dict(BASE, n_heads=2, n_layers=1, vocab=642),
                                 dict(BASE, n_heads=2, n_layers=1, wtype=1), dict(BASE, dim=4160, n_heads=65, ffn=8224, n_layers=1, vocab=130)])
@pytest.mark.parametrize("operator_attention", [0, 1])
def test_tail_equals_the_operators(cfg, operator_attention):
    w = M.synth_weights(cfg, seed=5, std=cfg["dim"] ** -0.5)
    rng = np.random.default_rng(7)
    ms = [M.Llama2(cfg, w) for _ in range(2)]
    for m, fused in zip(ms, (0, 1)):
        m.set_option("fused_decode", fused)
        m.set_option("operator_attention", operator_attention)
    pos = 0
    for n in (2, 33, 1, 40, 3):
        toks = rng.integers(3, cfg["vocab"], n).astype(np.uint32)
        a, b = (m.forward(toks, pos) for m in ms)
        pos += n
        # fp16 values between them, a few roundings apart: of the largest logit, 2^-11 each
        assert np.abs(a - b).max() <= 8 * 2.0 ** -11 * np.abs(a).max(), n
        assert np.abs(a).max() > 0
    # the rows of the caches come before the tail, the last token of one apart, which the steps' launches write
    for layer in range(cfg["n_layers"]):
        for value in (0, 1):
            x, y = (m.read_kv_cache(layer, value).astype(np.float32) for m in ms)
            assert np.abs(x - y).max() <= 8 * 2.0 ** -11 * np.abs(x).max()
    # a generation goes on from the logits of the tail
    ids = [m.generate_greedy(toks, 4)[0] for m in ms]
    assert np.array_equal(ids[0], ids[1])
    for m in ms:
        m.close()
