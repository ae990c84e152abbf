"""Prompt attention over the numbers of query tiles, heads and keys at which its
order of work changes, against the same in float32."""
import math

import pytest

from vkllama_amd import capi

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# Per output value, relative to sum_l p[l] |v[l]|: a weight is rounded to 16 bits (2^-9 in bf16, 2^-12 in fp16), an fp16
# score of up to 8 moves its weight by 8 * 2^-12, the result is rounded once (2^-9 / 2^-12 of |o| <= the sum).
BOUND = 6e-3


def reference(q, k, v, scale):
    """q [S, H, d], k, v [L, G, d] -> (out, sum of p |v|), both [S, H, d] fp32; query s sees keys up to s + L - S"""
    S, H, d = q.shape
    L, G, _ = k.shape
    hidden = torch.arange(L, device="cuda")[None, :] > torch.arange(S, device="cuda")[:, None] + (L - S)
    out, size = torch.empty((S, H, d), device="cuda"), torch.empty((S, H, d), device="cuda")
    for h in range(H):
        kk, vv = k[:, h // (H // G)].float().contiguous(), v[:, h // (H // G)].float().contiguous()
        p = (q[:, h].float().contiguous() @ kk.t().contiguous() * scale).masked_fill(hidden, -math.inf).softmax(-1)
        out[:, h], size[:, h] = p @ vv, p @ vv.abs()
    return out, size


@pytest.mark.parametrize("dtype,H,G,S,L,hd", [
    ("f16", 16, 16, 17 * 128 - 5, 17 * 128 - 5, 64),    # 34 tiles of an XCD: the second layer of its queue is short
    ("f16", 40, 40, 3 * 128, 3 * 128, 128),             # 15: one layer, heads end inside it
    ("f16", 40, 40, 12 * 128 - 100, 2000, 128),         # 60, keys before the queries
    ("f16", 8, 8, 33 * 128 + 1, 33 * 128 + 1, 64),      # one head's tiles in two layers
    ("f16", 5, 5, 7 * 128, 7 * 128 + 33, 64),           # heads not dealt to XCDs
    ("f16", 32, 32, 2048, 2048, 128),
    ("bf16", 32, 8, 11 * 128 + 7, 11 * 128 + 7, 128),
    ("bf16", 16, 4, 1500, 2100, 128),
    ("bf16", 8, 1, 35 * 128, 35 * 128 + 1, 32),
    ("f16", 32, 32, 77, 1577, 128),                     # the keys in parts
    ("f16", 5, 5, 1, 4000, 128),
    ("bf16", 16, 4, 130, 900, 64),
])
def test_every_tile_of_every_head(dev, dtype, H, G, S, L, hd):
    t = torch.float16 if dtype == "f16" else torch.bfloat16
    gen = torch.Generator(device="cuda").manual_seed(S * 7 + L + H)
    q, k, v = (torch.randn(s, generator=gen, device="cuda").to(t) for s in ((S, H, hd), (L, G, hd), (L, G, hd)))
    out = torch.full((S, H, hd), math.nan, device="cuda", dtype=t)
    scale = hd ** -0.5
    torch.cuda.synchronize()
    if dtype == "f16":
        capi.check(capi.lib().vkl_attn_prefill_causal_f16(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), H, S, L, hd, hd, H * hd, hd, H * hd, hd, H * hd, scale,
            out.data_ptr(), H * hd, hd, dev.stream))
    else:
        from vkllama_amd import stack
        capi.check(stack.lib().vkl_attn_prefill_causal_bf16(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), H, G, S, L, hd, H * hd, G * hd, G * hd, scale, 0.0, 1, None, 0,
            out.data_ptr(), H * hd, dev.stream))
    dev.sync()
    want, size = reference(q, k, v, scale)
    err = (out.float() - want).abs() / size
    assert bool(torch.isfinite(out).all()) and float(err.max()) < BOUND, float(err.nan_to_num(9.0).max())


@pytest.mark.parametrize("chunk,sink", [(0, 1), (96, 1), (192, 0)])
@pytest.mark.parametrize("H,G,S,L,hd", [(16, 4, 33, 33, 128), (16, 2, 77, 700, 128), (8, 8, 5, 1300, 64), (4, 1, 300, 300, 64)])
def test_chunks_and_parts_of_the_keys(dev, H, G, S, L, hd, chunk, sink):
    """Keys divided among workgroups: parts that hold no key of a chunk, the sink in one part only."""
    from vkllama_amd import stack
    gen = torch.Generator(device="cuda").manual_seed(S + L + chunk)
    q, k, v = (torch.randn(s, generator=gen, device="cuda").to(torch.bfloat16) for s in ((S, H, hd), (L, G, hd), (L, G, hd)))
    out = torch.full((S, H, hd), math.nan, device="cuda", dtype=torch.bfloat16)
    scale = -0.1
    torch.cuda.synchronize()
    capi.check(stack.lib().vkl_attn_prefill_chunked_bf16(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), H, G, S, L, hd, H * hd, G * hd, G * hd, scale, chunk, sink,
        out.data_ptr(), H * hd, dev.stream))
    dev.sync()
    pos = torch.arange(S, device="cuda")[:, None] + (L - S)
    key = torch.arange(L, device="cuda")[None, :]
    hidden = (key > pos) | (key < (pos // chunk * chunk if chunk else 0 * pos))
    for h in range(H):
        kk, vv = k[:, h // (H // G)].float().contiguous(), v[:, h // (H // G)].float().contiguous()
        s = (q[:, h].float().contiguous() @ kk.t().contiguous() * scale).masked_fill(hidden, -math.inf)
        if sink:
            s = torch.cat([s, torch.zeros((S, 1), device="cuda")], 1)
        p = s.softmax(-1)[:, :L]
        err = (out[:, h].float() - p @ vv).abs() / (p @ vv.abs())
        assert float(err.nan_to_num(9.0).max()) < BOUND, (h, float(err.nan_to_num(9.0).max()))


@pytest.mark.parametrize("scale", [0.0, -0.25])
def test_any_score_factor(dev, scale):
    H, S, L, hd = 8, 70, 200, 64
    gen = torch.Generator(device="cuda").manual_seed(7)
    q, k, v = (torch.randn((n, H, hd), generator=gen, device="cuda").half() for n in (S, L, L))
    out = torch.empty((S, H, hd), device="cuda", dtype=torch.float16)
    torch.cuda.synchronize()
    capi.check(capi.lib().vkl_attn_prefill_causal_f16(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), H, S, L, hd, hd, H * hd, hd, H * hd, hd, H * hd, scale,
        out.data_ptr(), H * hd, hd, dev.stream))
    dev.sync()
    want, size = reference(q, k, v, scale)
    assert float(((out.float() - want).abs() / size).max()) < BOUND
