"""The layer launch on either side of the rule for its number of workgroups: bit for bit the launches per phase."""
import numpy as np
import pytest

from vkllama_amd import model as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,ffn,heads,wtype", [(256, 352, 4, 8),        # the smallest
                                                 (2048, 5504, 32, 1),     # half: near the line by bytes, on it by heads
                                                 (2560, 6912, 20, 8),     # half
                                                 (2560, 6912, 40, 8),     # whole: too many heads
                                                 (2560, 6912, 20, 1)])    # whole: too many bytes
def test_either_number_of_workgroups(dim, ffn, heads, wtype):
    cfg = dict(dim=dim, n_layers=2, n_heads=heads, ffn=ffn, vocab=640, maxlen=64, eps=1e-5, wtype=wtype)
    m = M.Llama2(cfg, M.synth_weights(cfg, seed=9))
    prompt = np.random.default_rng(9).integers(3, 640, 5).astype(np.uint32)
    runs = []
    for mode in (0, 1):
        m.set_option("decode_mode", mode)
        for graph in (1, 0):
            m.set_option("decode_graph", graph)
            ids, _, _ = m.generate_greedy(prompt, 30)
            logits = m.forward([int(ids[-1])], 5 + 29)
            runs.append((list(ids), logits.view(np.uint32).copy()))
    assert m.decode_recoveries() == 0
    m.close()
    for ids, logits in runs[1:]:
        assert ids == runs[0][0] and np.array_equal(logits, runs[0][1])
