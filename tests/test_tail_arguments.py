"""What vkl_decode_tail refuses, one bad argument at a time: before it touches the GPU or follows a pointer."""
import ctypes as C

import pytest

import decode_util as U

ROOM = (C.c_uint8 * 4096)()
AT = (C.addressof(ROOM) + 255) // 256 * 256


def model(**over):
    table = (U.Layer * 2)()
    for t in table:
        for n, _ in U.Layer._fields_:
            setattr(t, n, AT)
    m = U.Model(dim=256, n_layers=2, n_heads=4, head_dim=64, ffn=704, vocab=1024, maxlen=96, wtype=8, eps=1e-5, final_eps=1e-6)
    m.layers, m.layers_h, m.tok_embd, m.output, m.output_norm, m.freqc, m.freqs, m.scratch = (AT,) * 8
    m.layers_h = C.addressof(table)
    for k, v in over.items():
        setattr(m, k, v)
    return m, table


def refused(m):
    lib = U.lib()
    return lib.vkl_decode_tail(C.byref(m), AT, AT, None, None) == 1 and lib.vkl_decode_tail_supported(C.byref(m)) == 0


def test_a_model_that_is_covered():
    m, table = model()
    assert U.lib().vkl_decode_tail_supported(C.byref(m)) == 1
    m, table = model(wtype=1, maxlen=1 << 20)  # (a step's scores would not fit)
    assert U.lib().vkl_decode_tail_supported(C.byref(m)) == 1
    assert U.lib().vkl_decode_tail_supported(None) == 0


@pytest.mark.parametrize("field,value", [("dim", 0), ("dim", 260), ("dim", 16640), ("n_layers", 0), ("n_heads", 0), ("n_heads", -4), ("n_heads", 5),
                                         ("head_dim", 0), ("head_dim", 32), ("ffn", 0), ("ffn", 700), ("ffn", 16416), ("vocab", 0),
                                         ("vocab", 1023), ("maxlen", 0), ("wtype", 2), ("layers", None), ("layers_h", None),
                                         ("tok_embd", None), ("output", None), ("output_norm", None), ("freqc", None), ("scratch", None)])
def test_a_model_that_is_not(field, value):
    m, table = model(**{field: value})
    assert refused(m)


@pytest.mark.parametrize("field", ["wo", "w_gate", "w_up", "w_down", "ffn_norm"])
def test_a_last_layer_without_a_matrix(field):
    m, table = model()
    setattr(table[0], field, None)  # (the others are not read)
    assert U.lib().vkl_decode_tail_supported(C.byref(m)) == 1
    setattr(table[1], field, None)
    assert refused(m)


def test_rows():
    m, table = model()
    f = U.lib().vkl_decode_tail
    for att, row in ((None, AT), (AT, None), (AT + 8, AT), (AT, AT + 2)):
        assert f(C.byref(m), att, row, None, None) == 1
    assert f(None, AT, AT, None, None) == 1
