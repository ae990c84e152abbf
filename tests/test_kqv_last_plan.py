"""When the other rows of Q are left out, as vkl_kqv_last_apart tells it (the host function that the launcher follows; no GPU)."""
from test_kqv_last import FORMED, LEFT_OUT
from vkllama_amd import capi


def test_which_form():
    """Only where the tiles of two matrices fill their rounds so that they save more than the second launch costs (Q8_0 1024 wide, 768 rows: 16.6 us
    with three matrices, 30.1 with two)."""
    apart = capi.lib().vkl_kqv_last_apart
    assert not any(apart(*c) for c in FORMED) and all(apart(*c) for c in LEFT_OUT)
    for w, M, W in ((1, 768, 1024), (1, 1557, 768), (1, 967, 2560), (1, 768, 3072), (8, 895, 1024), (8, 640, 1536), (8, 768, 3072), (8, 402, 2048)):
        assert not apart(w, M, W, W)
    for w, M, W in ((1, 2048, 4096), (1, 700, 4096), (1, 700, 2048), (8, 3967, 5120), (8, 700, 2048), (8, 640, 4096)):
        assert apart(w, M, W, W)
    for bad in ((2, 2048, 4096, 4096), (1, 0, 4096, 4096), (1, 2048, 0, 4096), (8, 2048, 4096, -32), (1, 2048, 4092, 4096)):
        assert not apart(*bad)
