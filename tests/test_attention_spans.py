"""Prompt attention where query tiles get different numbers of parts of the keys, against fp32 attention."""
import pytest

import test_attention_tiles as tiles

pytestmark = pytest.mark.gpu


# 12, 8 and 6 query tiles, two and three parts; 24 x 7: a last tile of one row; rows whose chunk begins behind the first key
@pytest.mark.parametrize("H,G,S,L,chunk,sink", [(16, 16, 1500, 1800, 0, 1), (24, 8, 1000, 2200, 0, 0), (32, 4, 700, 3100, 0, 1),
                                                (24, 4, 769, 2000, 1500, 1), (16, 4, 1411, 4000, 2500, 0)])
def test_chunks_and_sinks(dev, H, G, S, L, chunk, sink):
    tiles.test_chunks_and_parts_of_the_keys(dev, H, G, S, L, 128, chunk, sink)


@pytest.mark.parametrize("H,S,L", [(16, 1500, 2700), (24, 1000, 3400), (32, 700, 1900), (17, 1300, 2500)])
def test_fp16(dev, H, S, L):
    tiles.test_every_tile_of_every_head(dev, "f16", H, H, S, L, 128)
