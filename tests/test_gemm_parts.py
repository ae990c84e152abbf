"""Products of bf16 weights whose k range is divided: sums of the parts from the registers (rows of a multiple of eight
values) and through LDS (others), in any number of parts."""
import pytest

from vkllama_amd import capi
from vkllama_amd import stack

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# (tile rows, parts) of bf16 rows, and parts of planes: 64 rows and powers of two; three and five parts of 128 rows, three of
# 256 (pairs of columns and none), five of 192; three, six and seven parts of planes; the last tile of rows or columns in part; rows of 4 n + 2 values
@pytest.mark.parametrize("M,N,K,bf16,f32", [(40, 2056, 2048, (64, 8), 8), (131, 264, 4160, (128, 16), 16), (260, 4096, 5504, (192, 4), 3),
                                            (300, 2056, 7552, (128, 5), 6), (600, 2048, 5504, (128, 3), 3), (1200, 2040, 7552, (128, 3), 4),
                                            (300, 2050, 7552, (128, 5), 6), (77, 518, 4096, (64, 16), 16), (1025, 2048, 5504, (256, 3), 2),
                                            (1030, 4096, 11008, (256, 3), 4), (528, 2048, 7552, (192, 5), 3), (300, 2048, 5504, (128, 5), 6), (193, 1100, 2816, (64, 4), 7)])
@pytest.mark.parametrize("xtype", [stack.BF16, stack.F32])
def test_parts(dev, M, N, K, bf16, f32, xtype):
    p = stack.project_plan(xtype, M, N, K)
    assert (p.tile_rows, p.ksplit, p.planes) == ((*bf16, 1) if xtype == stack.BF16 else (64, f32, 3))
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
    want = xd @ wd.t()
    assert bool(((y[:, :N] - want).abs() <= off).all())
    # (of the whole: a plane that is lost leaves 2^-16 / sqrt (3) of every value, 8e-6 and more; measured 1e-7 to 7e-7)
    assert float((y[:, :N] - want).norm() / want.norm()) < 1e-6
    assert bool((y[:, N:] == 7.0).all())
    assert torch.equal(runs[0], runs[1])
