"""Prompt attention where query tiles get different numbers of parts of the keys: the rule, and results against fp32 attention."""
import pytest

from vkllama_amd import stack
import test_attention_tiles as tiles


def parts(H, S, L, chunk=0, hd=128):
    """of every query tile, and the most of any"""
    lib = stack.lib()
    each = [lib.vkl_attn_prefill_tile_parts(H, S, L, hd, chunk, q) for q in range(0, S, 128)]
    assert lib.vkl_attn_prefill_tile_parts(H, S, L, hd, chunk, S - 1) == each[-1]
    assert lib.vkl_attn_prefill_parts(H, S, L, hd, chunk) >= max(each)
    return each


# 12, 8 and 6 query tiles, two and three parts; 24 x 7: a last tile of one row
PLAIN = [(16, 1500, 1800), (16, 1500, 2700), (24, 1000, 2200), (24, 897, 2097), (32, 700, 3100), (32, 700, 1900), (40, 600, 3000),
         (7, 3200, 3201), (10, 2177, 2477)]
# rows whose chunk begins behind the first key, tiles that a chunk's end divides
CHUNKED = [(16, 4, 1500, 4400, 2500, 1), (16, 16, 1411, 5600, 2500, 0), (24, 8, 1000, 5200, 3000, 1), (8, 2, 2946, 5946, 3500, 1)]
UNEVEN = PLAIN + [(H, S, L, c) for H, _, S, L, c, _ in CHUNKED]


@pytest.mark.parametrize("shape", UNEVEN)
def test_longer_rows_have_more_parts(shape):
    H, S, L, chunk = (*shape, 0)[:4]
    each = parts(H, S, L, chunk)
    seen = [(min(L, q + 128 + L - S) + 63) // 64 - ((q + L - S) // chunk * chunk // 64 if chunk else 0) for q in range(0, S, 128)]
    assert set(each) in ({1, 3}, {2, 3}, {1, 2, 3})
    assert max(each[i] for i, n in enumerate(seen) if n == max(seen)) == 3
    # a span that gives every tile its parts: n tiles of keys in p parts, span * (p - 1) < n <= span * p
    assert any(all(s * (p - 1) < n <= s * p for n, p in zip(seen, each)) for s in range(1, max(seen) + 1))
    assert sum(each) * H <= 500


# too many groups; 192 groups of heads that are not dealt to XCDs; too many heads; heads of 64 values; 198 groups of heads that are not dealt
@pytest.mark.parametrize("H,S,L,hd", [(16, 2000, 3200, 128), (12, 2018, 3000, 128), (6, 3969, 6369, 128), (48, 448, 3648, 128),
                                      (96, 192, 3392, 128), (16, 1500, 2100, 64), (18, 1408, 2608, 128)])
def test_even_parts(H, S, L, hd):
    assert set(parts(H, S, L, 0, hd)) == {2}


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,S,L,chunk,sink", [(H, H // 2, S, L, 0, H % 3) for H, S, L in PLAIN if H % 2 == 0] + CHUNKED)
def test_chunks_and_sinks(dev, H, G, S, L, chunk, sink):
    assert len(set(parts(H, S, L, chunk))) > 1
    tiles.test_chunks_and_parts_of_the_keys(dev, H, G, S, L, 128, chunk, int(sink > 0))


@pytest.mark.gpu
@pytest.mark.parametrize("H,S,L", PLAIN)
def test_fp16(dev, H, S, L):
    assert len(set(parts(H, S, L))) > 1
    tiles.test_every_tile_of_every_head(dev, "f16", H, H, S, L, 128)
