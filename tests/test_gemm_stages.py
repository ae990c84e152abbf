"""Products of bf16 weights whose k range is shorter, as long as and longer than the stages of a tile, by every remainder."""
import pytest

from vkllama_amd import capi
from vkllama_amd import stack

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# tiles of 64 rows, one to a compute unit and more of them; 128 rows by four waves and, cut in two, by eight; 256 rows by
# four waves and by eight; planes in two and four stages
@pytest.mark.parametrize("M,N,xtype", [(40, 264, stack.BF16), (200, 264, stack.BF16), (130, 16384, stack.BF16), (650, 3080, stack.BF16),
                                       (160, 8056, stack.BF16), (750, 5448, stack.BF16), (1280, 6392, stack.BF16), (300, 8192, stack.BF16),
                                       (520, 12288, stack.BF16), (200, 1032, stack.F32), (800, 24584, stack.F32)])
def test_short_k_ranges(dev, M, N, xtype):
    g = torch.Generator(device="cuda").manual_seed(M + N)
    steps = (1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 13)
    xs = torch.randn((M, 64 * steps[-1]), generator=g, device="cuda")
    xs = xs if xtype == stack.F32 else xs.bfloat16()
    ws = torch.randn((N, 64 * steps[-1]), generator=g, device="cuda").bfloat16()
    for s in steps if M * N < 1 << 23 else steps[:6]:
        K = 64 * s
        x, w = xs[:, :K], ws[:, :K].contiguous()
        y = torch.full((M, N + 8), 7.0, device="cuda")
        torch.cuda.synchronize()
        capi.check(stack.lib().vkl_project_bf16w(x.data_ptr(), xtype, x.stride(0), w.data_ptr(), M, N, K,
                                                 stack.segments([(0, N, y.data_ptr(), N + 8, stack.F32, 0, None, 0.0)]), 1, dev.stream))
        dev.sync()
        # exact products, K of them (planes: and 2 K small ones) added in fp32: half of 2^-23 of the sum of magnitudes each
        xd, wd = x.double(), w.double()
        off = K / 2 * 2.0 ** -23 * (xd.abs() @ wd.abs().t())
        assert bool(((y[:, :N] - xd @ wd.t()).abs() <= off).all()), K
        assert bool((y[:, N:] == 7.0).all()), K
