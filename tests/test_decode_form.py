"""What a step's launches are, and that measuring them measures those launches."""
import numpy as np
import pytest

from vkllama_amd import capi
from vkllama_amd import model as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,ffn,heads,wtype,vocab,form", [
    (512, 1376, 8, 8, 640, "step"), (512, 1376, 8, 1, 640, "step"), (1024, 2752, 8, 1, 32000, "layers"),
    (1088, 2912, 17, 8, 640, "step"), (1920, 5120, 15, 8, 640, "layers"), (1088, 2912, 17, 1, 640, "layer"), (256, 1024, 2, 8, 640, "layer")])
def test_forms_and_their_phases(dim, ffn, heads, wtype, vocab, form):
    cfg = dict(dim=dim, n_layers=3, n_heads=heads, ffn=ffn, vocab=vocab, maxlen=64, eps=1e-5, wtype=wtype)
    m = M.Llama2(cfg, M.synth_weights(cfg, seed=2))
    m.set_option("decode_mode", 0)
    assert m.decode_form(5) == "phases"
    m.set_option("decode_mode", 1)
    assert m.decode_form(5) == form and m.decode_form(64) == "phases"      # (beyond the context)
    m.set_option("attn_split_min", 40)
    assert m.decode_form(38) == form and m.decode_form(39) == "phases"
    m.set_option("attn_split_min", 0)
    prompt = np.arange(3, 9).astype(np.uint32)
    want, _, _ = m.generate_greedy(prompt, 20)
    m.set_option("decode_graph", 0)
    m.set_option("phase_timing", 1)
    m.phase_times()
    timed, _, _ = m.generate_greedy(prompt, 20)
    m.set_option("phase_timing", 0)
    times = {k: n for k, (ms, n) in m.phase_times().items() if n}
    assert times == {"step": {"step": 19}, "layers": {"layers": 19, "lm_head": 19}, "layer": {"layer": 57, "lm_head": 19}}[form]
    for kind in ("step", "layers", "layer"):
        if kind == form or kind == "layer":
            us, n = m.phase_replay(kind, 7, 4)
            assert us > 0 and n == (12 if kind == "layer" else 4)
        else:
            with pytest.raises(capi.VklError):
                m.phase_replay(kind, 7, 4)
    assert m.phase_bytes("layers", 8) == 3 * m.phase_bytes("layer", 8)
    assert 0.98 < m.phase_bytes("step", 8) / m.decode_step_bytes(8) < 1.02
    again, _, _ = m.generate_greedy(prompt, 20)
    assert list(timed) == list(want) and list(again) == list(want)
    assert m.decode_recoveries() == 0
    m.close()
