"""What vkl_stack_layer_step and vkl_stack_logits refuse beside a model that is covered, one bad argument at a time: before they touch
the GPU."""
import ctypes as C

import pytest

from vkllama_amd import stack

vp, i32, f32 = C.c_void_p, C.c_int, C.c_float
ROOM = (C.c_uint8 * 4096)()
AT = (C.addressof(ROOM) + 255) // 256 * 256
MAXLEN = 96


def fields(text):
    return [(n, t) for t, names in text for n in names.split()]


class Layer(C.Structure):
    """vkl_stack_layer"""
    _fields_ = fields([(i32, "mixer H G dim vdim rank rank_p"), (f32, "scale temp_coef"), (i32, "temp_every ff"), (vp, "norm w_in"),
                       (i32, "n_in kv0 g0 up0"), (vp, "w_out"), (i32, "k_out ff_col"), (vp, "w_ukt w_uv c_norm cache norm2 w_up w_down"),
                       (i32, "ff_p ff_act v0 n npair chunk sink"), (vp, "freq vcache vfirst"), (i32, "fdim"), (f32, "vmix"),
                       (i32, "b0 a0 taps vn r_a r_g"), (vp, "w_a2 w_g2 conv ring dt_bias rate log_decay gnorm"), (f32, "qscale unit_eps"),
                       (vp, "state")])


class Model(C.Structure):
    """vkl_stack_model"""
    _fields_ = fields([(i32, "width width_p vocab maxlen n_runs ctype"), (f32, "eps logit_cap"), (vp, "layers_h embed head"),
                       (f32, "embed_scale"), (vp, "embed_norm final_norm scratch")])


@pytest.fixture
def model():
    """two layers of shared rows, each 2 heads of 32 and 64 feed-forward values"""
    layers = (Layer * 2)()
    for l in layers:
        l.H, l.G, l.dim, l.vdim, l.ff, l.n_in, l.kv0, l.up0, l.k_out, l.ff_col = 2, 1, 32, 32, 64, 160, 64, 96, 128, 64
        l.norm = l.w_in = l.w_out = l.cache = AT
    m = Model(width=64, width_p=64, vocab=96, maxlen=MAXLEN, n_runs=2, ctype=stack.BF16, eps=1e-5)
    m.layers_h, m.embed, m.final_norm, m.scratch = C.addressof(layers), AT, AT, AT
    assert stack.lib().vkl_stack_supported(C.byref(m)) == 1
    yield m
    assert len(layers) == 2


@pytest.mark.parametrize("run,x,pos", [(-1, AT, 0), (2, AT, 0), (0, None, 0), (0, AT + 4, 0), (1, AT + 8, 0), (0, AT, MAXLEN), (1, AT, 2**32 - 1)])
def test_layer_step(model, run, x, pos):
    assert stack.lib().vkl_stack_layer_step(C.byref(model), run, x, pos, None) == 1


def test_layer_step_of_a_model_that_is_not_covered(model):
    model.width_p = 72
    assert stack.lib().vkl_stack_supported(C.byref(model)) == 0
    assert stack.lib().vkl_stack_layer_step(C.byref(model), 0, AT, 0, None) == 1


@pytest.mark.parametrize("x,logits", [(None, AT), (AT + 4, AT), (AT, None)])
def test_logits(model, x, logits):
    assert stack.lib().vkl_stack_logits(C.byref(model), x, logits, None) == 1
