"""Attention of many 32-bit query rows on the matrix cores, against 64 bits."""
import math

import pytest

from vkllama_amd import capi
from vkllama_amd import stack

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def attend(dev, q, k, v, H, G, D, pos0, chunk=0, sink=0, temp=(0.0, 1), pad=0):
    S, lib = q.shape[0], stack.lib()
    out = torch.full((S, H * D + pad), 7.0, device="cuda")
    shared = v is None
    need = (lib.vkl_attn_rows_scratch_bytes if shared else lib.vkl_attn_kv_rows_scratch_bytes)(stack.F32, H, G, D, S)
    scratch = torch.zeros(need, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    if shared:
        err = lib.vkl_attn_rows(q.data_ptr(), stack.F32, q.stride(0), k.data_ptr(), stack.F32, k.stride(0), H, G, D, S, pos0, 0.3,
                                *temp, out.data_ptr(), stack.F32, out.stride(0), scratch.data_ptr(), dev.stream)
    else:
        err = lib.vkl_attn_kv_rows(q.data_ptr(), stack.F32, q.stride(0), k.data_ptr(), v.data_ptr(), stack.F32, k.stride(0), H, G, D, S,
                                   pos0, 0.3, chunk, sink, out.data_ptr(), stack.F32, out.stride(0), scratch.data_ptr(), dev.stream)
    capi.check(err)
    dev.sync()
    assert bool((out[:, H * D:] == 7.0).all())
    return out[:, :H * D]


def reference(q, k, v, H, G, D, pos0, chunk=0, sink=0, temp=(0.0, 1)):
    S, L = q.shape[0], pos0 + q.shape[0]
    pos, key = torch.arange(pos0, L, device="cuda"), torch.arange(L, device="cuda")
    hidden = (key[None] > pos[:, None]) | (key[None] < (pos // chunk * chunk if chunk else pos * 0)[:, None])
    f = 0.3 * (1.0 + temp[0] * torch.log(torch.floor((pos + 1) / temp[1]).double() + 1.0))
    out, size = [], []
    for h in range(H):
        cols = slice(h // (H // G) * D, (h // (H // G) + 1) * D)
        x, y = k[:L, cols].double(), (k if v is None else v)[:L, cols].double()
        s = (q[:, h * D:(h + 1) * D].double() * f[:, None] @ x.t()).masked_fill(hidden, -math.inf)
        if sink:
            s = torch.cat([s, s.new_zeros(S, 1)], 1)
        w = torch.softmax(s, -1)[:, :L]
        out.append(w @ y), size.append(w @ y.abs())
    return torch.cat(out, 1), torch.cat(size, 1)


def inputs(S, L, H, G, D, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn((S, H * D + 8), generator=g, device="cuda")[:, :H * D], torch.randn((L, G * D + 8), generator=g, device="cuda")[:, :G * D],
            torch.randn((L, G * D + 8), generator=g, device="cuda")[:, :G * D])


# the smallest, a last tile of one row and of fifteen, waves without a block, a context in front; chunks that begin in a tile and in a block;
# 15 rows, few rows of few heads and few rows behind many (the row kernel)
@pytest.mark.parametrize("H,G,S,pos0,D,chunk,sink,tiles", [
    (8, 1, 16, 0, 128, 0, 1, 1), (3, 3, 17, 0, 64, 0, 0, 1), (16, 2, 31, 5, 128, 0, 1, 1), (8, 2, 300, 0, 64, 0, 1, 1), (5, 1, 130, 77, 128, 0, 0, 1),
    (2, 2, 200, 40, 64, 37, 1, 1), (4, 1, 97, 63, 128, 64, 0, 1), (2, 1, 64, 10, 128, 16, 1, 1), (2, 1, 15, 3, 128, 0, 1, 0),
    (2, 1, 16, 0, 128, 0, 1, 0), (4, 2, 31, 5, 128, 0, 1, 0), (2, 1, 18, 1500, 64, 0, 1, 0)])
def test_against_64_bits(dev, H, G, S, pos0, D, chunk, sink, tiles):
    assert stack.lib().vkl_attn_f32_tiles(1, H, G, D, S, pos0, chunk) == tiles
    q, k, v = inputs(S, pos0 + S + 3, H, G, D, S + D)
    q = q * torch.exp(torch.linspace(-3, 1.5, S, device="cuda"))[:, None]  # from flat to sharp
    q = torch.nn.functional.pad(q, (0, 8))[:, :H * D]
    k[pos0 + S:], v[pos0 + S:] = math.nan, math.nan                           # not there yet
    got = attend(dev, q, k, v, H, G, D, pos0, chunk, sink, pad=5)
    want, size = reference(q, k, v, H, G, D, pos0, chunk, sink)
    # scores of up to 0.3 |q| |k| (some 200): each off by D / 2 + 1 roundings of sums of that size, which is the relative error of a weight;
    # and the sums of weights and of values
    top = 0.3 * float(q.norm(dim=1).max() * k[:pos0 + S].norm(dim=1).max())
    assert bool(((got - want).abs() <= (top * 8 * 2.0 ** -24 + 64 * 2.0 ** -24) * size + 1e-9).all())


@pytest.mark.parametrize("S,pos0,D", [(16, 0, 64), (100, 30, 128)])
def test_shared_rows_and_a_temperature(dev, S, pos0, D):
    assert stack.lib().vkl_attn_f32_tiles(0, 4, 2, D, S, pos0, 0) == 1
    q, k, _ = inputs(S, pos0 + S, 4, 2, D, S)
    got = attend(dev, q, k, None, 4, 2, D, pos0, temp=(0.2, 16))
    want, size = reference(q, k, None, 4, 2, D, pos0, temp=(0.2, 16))
    top = 0.5 * float(q.norm(dim=1).max() * k.norm(dim=1).max())
    assert bool(((got - want).abs() <= (top * 8 * 2.0 ** -24 + 64 * 2.0 ** -24) * size + 1e-9).all())


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("odd", [math.inf, -math.inf, math.nan])
@pytest.mark.parametrize("chunk", [0, 24])
def test_values_that_are_not_finite_reach_those_who_see_them(dev, D, odd, chunk):
    """A value of a later position, or of an earlier chunk, changes nothing."""
    S, H = 60, 8
    assert stack.lib().vkl_attn_f32_tiles(1, H, 1, D, S, 0, chunk) == 1
    q, k, v = inputs(S, S, H, 1, D, D)
    clean = attend(dev, q, k, v, H, 1, D, 0, chunk, 1)
    bad = torch.nn.functional.pad(v, (0, 8))[:, :D]                          # (of the strides of k)
    bad[21, 3] = odd
    got = attend(dev, q, k, bad, H, 1, D, 0, chunk, 1)
    pos = torch.arange(S, device="cuda")
    sees = (pos >= 21) & ((pos // chunk == 21 // chunk) if chunk else (pos >= 0))
    column = torch.arange(H * D, device="cuda") % D == 3
    assert bool((~torch.isfinite(got[sees][:, column])).all())
    # (rows of such a block are added one by one: the last bits differ)
    assert bool(torch.isfinite(got[~sees]).all()) and bool(torch.isfinite(got[:, ~column]).all())
    assert bool(((got[~sees] - clean[~sees]).abs() <= 64 * 2.0 ** -24 * 4.0).all())
    assert bool(((got[:, ~column] - clean[:, ~column]).abs() <= 64 * 2.0 ** -24 * 4.0).all())
