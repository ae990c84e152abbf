"""Which attention of 32-bit rows goes to the matrix cores, as vkl_attn_f32_tiles tells it (the host function that the launcher follows;
no GPU): shapes that were measured on both kernels."""
import pytest

from vkllama_amd import stack


# few rows of few heads, which the tiles took up to 1.47 times as long for; long contexts behind few rows
@pytest.mark.parametrize("vals,H,G,D,S,pos0", [(0, 4, 4, 128, 111, 0), (0, 4, 4, 128, 97, 0), (0, 4, 4, 128, 176, 0), (0, 12, 12, 128, 25, 52), (0, 8, 8, 128, 39, 0),
                                               (0, 16, 16, 128, 31, 50), (0, 12, 12, 64, 61, 2519), (0, 4, 2, 128, 157, 30), (1, 4, 4, 128, 85, 0),
                                               (1, 4, 4, 128, 128, 0), (1, 8, 8, 128, 18, 44), (1, 2, 1, 128, 15, 0), (1, 16, 4, 128, 32, 2968)])
def test_the_row_kernel(vals, H, G, D, S, pos0):
    assert stack.lib().vkl_attn_f32_tiles(vals, H, G, D, S, pos0, 0) == 0


@pytest.mark.parametrize("vals,H,G,D,S,pos0,chunk", [(0, 16, 16, 128, 980, 0, 0), (0, 4, 4, 128, 708, 19, 0), (0, 16, 4, 64, 100, 0, 0), (1, 16, 4, 128, 300, 0, 0),
                                                     (1, 16, 4, 128, 800, 0, 256), (1, 16, 4, 128, 100, 0, 0), (1, 16, 4, 64, 300, 0, 0),
                                                     (1, 32, 8, 128, 2000, 0, 0), (1, 16, 2, 128, 16, 0, 0)])
def test_the_tiles(vals, H, G, D, S, pos0, chunk):
    assert stack.lib().vkl_attn_f32_tiles(vals, H, G, D, S, pos0, chunk) == 1


def test_arguments():
    f = stack.lib().vkl_attn_f32_tiles
    good = (1, 16, 4, 128, 300, 0, 0)
    assert f(*good) == 1
    for i, bad in ((1, 0), (1, 17), (2, 0), (3, 0), (3, 96), (4, 0), (4, 65536), (5, 2**32 - 1), (6, -1)):
        assert f(*(bad if j == i else v for j, v in enumerate(good))) == 0, (i, bad)
