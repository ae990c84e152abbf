"""Products of bf16 weights whose k range is divided: sums of the parts from the registers (rows of a multiple of eight
values) and through LDS (others), in any number of parts."""
import pytest

from vkllama_amd import capi
from vkllama_amd import stack

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# 64 rows and parts that are a power of two; three to seven parts of 128 and 256 rows; the last tile of rows or columns in
# part; rows of 4 n + 2 values
@pytest.mark.parametrize("xtype", [stack.BF16, stack.F32])
@pytest.mark.parametrize("M,N,K", [(40, 2056, 2048), (131, 264, 4160), (260, 4096, 5504), (300, 2056, 7552), (600, 2048, 5504),
                                   (1200, 2040, 7552), (300, 2050, 7552), (77, 518, 4096)])
def test_parts(dev, M, N, K, xtype):
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn((M, K), generator=g, device="cuda")
    x = x if xtype == stack.F32 else x.bfloat16()
    w = torch.randn((N, K), generator=g, device="cuda").bfloat16()
    runs = []
    for _ in range(2):
        y = torch.full((M, N + 8), 7.0, device="cuda")
        torch.cuda.synchronize()
        capi.check(stack.lib().vkl_project_bf16w(x.data_ptr(), xtype, K, w.data_ptr(), M, N, K,
                                                 stack.segments([(0, N, y.data_ptr(), N + 8, stack.F32, 0, None, 0.0)]), 1, dev.stream))
        dev.sync()
        runs.append(y)
    # exact products, K of them (planes: and 2 K small ones) added in fp32: half of 2^-23 of the sum of magnitudes each
    xd, wd = x.double(), w.double()
    off = K / 2 * 2.0 ** -23 * (xd.abs() @ wd.abs().t())
    assert bool(((y[:, :N] - xd @ wd.t()).abs() <= off).all())
    assert bool((y[:, N:] == 7.0).all())
    assert torch.equal(runs[0], runs[1])
