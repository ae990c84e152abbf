"""All layers of a step in one launch (narrow rows): bit for bit the launches per phase."""
import numpy as np
import pytest

from vkllama_amd import model as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,ffn,heads,wtype,prompt,maxlen", [
    (64, 192, 1, 8, 3, 64),        # one head, eight workgroups, three pairs for every wave
    (64, 32, 1, 1, 3, 64),         # fewer pairs than waves
    (128, 352, 1, 8, 3, 64),       # heads of 128 values; two or three pairs
    (512, 1376, 8, 8, 570, 640),   # cached rows beyond those a head requests ahead
    (576, 1536, 9, 1, 3, 64),      # fp16: a row's second step of loads in part
    (1024, 3072, 8, 1, 3, 64),     # fp16: the widest
    (1088, 2912, 17, 8, 3, 64),    # Q8_0: a second step of loads in part
    (1792, 4768, 28, 8, 3, 64),    # Q8_0: workgroups for all but four compute units
    (64, 192, 1, 8, 3, 15900),     # as many positions as half the LDS of a compute unit takes
    (1792, 5408, 14, 8, 3, 64),    # more than three pairs for a wave: a launch per layer
])
def test_all_layers_in_one_launch(dim, ffn, heads, wtype, prompt, maxlen):
    compare(dim, ffn, heads, wtype, prompt, maxlen, 642)


@pytest.mark.parametrize("dim,wtype,vocab", [
    (64, 8, 2),             # one wave has the vocabulary
    (64, 1, 95234),         # two rounds of what the waves hold, of no round number
    (512, 8, 32000),
    (512, 1, 40002),        # one row of each in every load, two rounds
    (512, 1, 70654),        # more than two rounds: a launch of its own
    (1024, 8, 30720),       # as many as the one launch takes
    (1024, 8, 30722),       # more: a launch of its own
    (1024, 8, 43006),
    (1024, 8, 43012),
])
def test_whole_step_in_one_launch(dim, wtype, vocab):
    compare(dim, 3 * dim // 64 * 32, max(1, dim // 128), wtype, 3, 64, vocab)


def compare(dim, ffn, heads, wtype, prompt, maxlen, vocab):
    cfg = dict(dim=dim, n_layers=3, n_heads=heads, ffn=ffn, vocab=vocab, maxlen=maxlen, eps=1e-5, wtype=wtype)
    m = M.Llama2(cfg, M.synth_weights(cfg, seed=dim))
    ids0 = np.random.default_rng(dim).integers(0, vocab, prompt).astype(np.uint32)
    runs = []
    for mode in (0, 1):
        m.set_option("decode_mode", mode)
        for graph in (1, 0):
            m.set_option("decode_graph", graph)
            ids, _, _ = m.generate_greedy(ids0, 40)
            logits = m.forward([int(ids[-1])], prompt + 39)
            runs.append((list(ids), logits.view(np.uint32).copy(), m.read_kv_cache(2, True)[:, :prompt + 40].copy()))
    assert m.decode_recoveries() == 0
    m.close()
    for ids, logits, rows in runs[1:]:
        assert ids == runs[0][0] and np.array_equal(logits, runs[0][1])
        assert np.array_equal(rows.view(np.uint16), runs[0][2].view(np.uint16))
