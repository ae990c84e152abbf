"""Scratch of the decode step: rows of tagged words only for shapes whose layers can share a launch; host arithmetic, no GPU needed."""
import ctypes as C

import pytest

import decode_util as U


def scratch_bytes(dim, heads, ffn, wtype):
    m = U.Model()
    m.dim, m.n_layers, m.n_heads, m.head_dim, m.ffn, m.vocab, m.maxlen, m.wtype = dim, 2, heads, dim // heads, ffn, 640, 64, wtype
    return U.lib().vkl_decode_scratch_bytes(C.byref(m))


@pytest.mark.parametrize("dim,heads,wtype,tagged", [(512, 8, 8, True), (512, 8, 1, True), (1024, 16, 1, True), (1088, 17, 8, True),
                                                    (1920, 15, 8, True), (1792, 28, 8, True), (1088, 17, 1, False),
                                                    (1920, 30, 8, False), (2048, 16, 8, False), (2048, 16, 1, False)])
def test_tagged_rows_where_they_are_used(dim, heads, wtype, tagged):
    # (one pair too many for a wave: no rows, and a little more of everything that grows with ffn)
    have = scratch_bytes(dim, heads, 3 * dim, wtype) - scratch_bytes(dim, heads, 3 * dim + 32, wtype)
    rows = 4 * (3 * dim + 3 * 8 * dim + 8 * 3 * dim + 2 * 512)
    assert rows - 1024 <= have <= rows if tagged else -1024 <= have <= 0
