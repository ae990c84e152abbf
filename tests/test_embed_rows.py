"""Embedding rows at widths and addresses where the wide accesses begin and end."""
import numpy as np
import pytest

import fazinex_ref as R
from oracle import oracle as O
from util import q8_weights
from vkllama_amd import capi
from vkllama_amd import stack

pytestmark = pytest.mark.gpu


def guarded(dev, n, W, skip):
    """(buffer of n rows behind `skip` values and before eight, reader of the rows that checks both guards)"""
    buf = dev.upload(np.full(skip + n * W + 8, 0x7e11, np.uint16))

    def rows():
        got = buf.read(np.uint16, (skip + n * W + 8,))
        assert np.all(got[:skip] == 0x7e11) and np.all(got[skip + n * W:] == 0x7e11)
        return got[skip:skip + n * W].reshape(n, W)
    return buf, rows


@pytest.mark.parametrize("skip", [0, 8, 1])
@pytest.mark.parametrize("W", [1, 7, 8, 32, 100, 2040, 2048, 2056, 2061, 4104])
def test_rows_of_both_tables(dev, rng, W, skip):
    V, toks = 9, np.array([0, 8, 3, 9, 2 ** 31 + 5], np.uint32)
    dt = dev.upload(toks)
    raw, _ = q8_weights(rng, V, W)
    table = dev.upload_q8_0(raw, V, W)
    out, rows = guarded(dev, len(toks), W, skip)
    capi.check(capi.lib().vkl_embed_q8_0(table.ptr, V, W, dt.ptr, len(toks), 2, out.ptr.value + 2 * skip, dev.stream))
    assert np.array_equal(rows(), O.embedding_q8_0(raw, W, toks, 2).view(np.uint16))
    half = rng.standard_normal((V, W)).astype(np.float16)
    for shift in (0, 1):
        table = dev.upload(np.concatenate([np.zeros(shift, np.float16), half.ravel()]))
        out, rows = guarded(dev, len(toks), W, skip)
        capi.check(capi.lib().vkl_embed_f16(table.ptr.value + 2 * shift, V, W, dt.ptr, len(toks), 2, out.ptr.value + 2 * skip, dev.stream))
        assert np.array_equal(rows(), O.embedding_f16(half, toks, 2).view(np.uint16))


@pytest.mark.parametrize("W", [8, 2040, 2048, 2049, 2056, 4096, 4104, 8192, 16384, 16392])
def test_normed_rows_by_block_size(dev, rng, W):
    Wp, V = (W + 63) // 64 * 64, 6
    vals = np.zeros((V, Wp), np.float32)
    vals[:, :W] = rng.standard_normal((V, W)).astype(np.float32)
    bits = (vals.view(np.uint32) >> 16).astype(np.uint16)
    vals = (bits.astype(np.uint32) << 16).view(np.float32)
    wn = rng.uniform(0.5, 1.5, W).astype(np.float32)
    toks = np.array([5, 0, 3, 6, 1], np.uint32)
    dt, dn, dk = dev.upload(bits), dev.upload(wn), dev.upload(toks)
    out = dev.upload(np.full((5, Wp), 7, np.float32))
    capi.check(stack.lib().vkl_embed_norm_bf16(dt.ptr, V, Wp, W, dk.ptr, 5, dn.ptr, 1e-3, out.ptr, Wp, dev.stream))
    got, want = out.read(np.float32, (5, Wp)), R.rms_norm(vals[[5, 0, 3, 0, 1], :W], wn, 1e-3)
    # the sum of squares: at most 64 additions deep; a square root, a division and two products behind it
    assert np.all(np.abs(got[:, :W] - want) <= (64 / 2 + 6) * 2.0 ** -24 * np.abs(want))
    assert np.all(got[:, W:] == 7)
    capi.check(stack.lib().vkl_embed_rows_bf16(dt.ptr, V, Wp, W, dk.ptr, 5, 3.0, out.ptr, Wp, dev.stream))
    assert np.array_equal(out.read(np.float32, (5, Wp))[:, :W], vals[[5, 0, 3, 0, 1], :W] * np.float32(3))
