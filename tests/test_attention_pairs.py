"""Prompt attention whose workgroups are two groups of waves, on every other tile of keys: many tiles of keys in one part and
a compute unit for each workgroup."""
import pytest

from vkllama_amd import stack
import test_attention_tiles as tiles

pytestmark = pytest.mark.gpu


# odd and even numbers of tiles, a last tile of one key
@pytest.mark.parametrize("dtype,H,G,S,L,hd", [("f16", 8, 8, 640, 640, 128), ("f16", 17, 17, 705, 705, 128), ("bf16", 16, 4, 1345, 1345, 128),
                                              ("bf16", 16, 8, 641, 641, 64), ("f16", 32, 32, 1000, 1000, 64), ("bf16", 16, 4, 2048, 2048, 128)])
def test_rows(dev, dtype, H, G, S, L, hd):
    assert stack.lib().vkl_attn_prefill_parts(H, S, L, hd, 0) == 1
    tiles.test_every_tile_of_every_head(dev, dtype, H, G, S, L, hd)


# chunks that begin in a tile and at one, whose first keys only one group sees; a last query tile of one tile of keys, of which the
# second group has none: one row, several
@pytest.mark.parametrize("H,G,S,L,hd,chunk,sink", [(16, 4, 1500, 1500, 128, 700, 1), (16, 2, 1100, 1100, 64, 640, 1), (16, 16, 1100, 1100, 128, 0, 1),
                                                   (16, 4, 1200, 1200, 128, 650, 0), (16, 4, 641, 641, 128, 640, 1), (16, 16, 641, 641, 64, 640, 0),
                                                   (16, 4, 1290, 1290, 128, 1280, 1), (16, 2, 1290, 1290, 128, 1280, 0)])
def test_chunks_and_sinks(dev, H, G, S, L, hd, chunk, sink):
    assert stack.lib().vkl_attn_prefill_parts(H, S, L, hd, chunk) == 1
    tiles.test_chunks_and_parts_of_the_keys(dev, H, G, S, L, hd, chunk, sink)
