"""Products of few rows in 64-row tiles (bf16 weights), at the edges of a tile, in one and several parts of the k range."""
import pytest

from vkllama_amd import capi
from vkllama_amd import stack

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(1, 8, 64), (12, 16136, 512), (31, 264, 2048), (63, 136, 576), (33, 2048, 2048), (64, 5504, 512),
                                   (65, 136, 5504), (128, 8064, 512), (192, 2048, 2048), (300, 5512, 1088),
                                   (520, 2048, 2048), (640, 16128, 576)])
@pytest.mark.parametrize("xtype", [stack.BF16, stack.F32])
def test_rows_in_tiles_of_64(dev, M, N, K, xtype):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn((M, K + 64), generator=g, device="cuda")
    x = (x if xtype == stack.F32 else x.bfloat16())[:, :K]
    w = torch.randn((N, K), generator=g, device="cuda").bfloat16()
    cut = (N // 2 + 7) // 8 * 8 if N > 8 else 8
    res = torch.randn((M, cut), generator=g, device="cuda")
    a, b = torch.full((M, cut), 7.0, device="cuda"), torch.full((M, max(N - cut, 1) + 3), 7.0, device="cuda")
    segs = [(0, cut, a.data_ptr(), cut, stack.F32, 0, res.data_ptr(), 0.0)]
    if N > cut:
        segs.append((cut, N - cut, b.data_ptr(), N - cut + 3, stack.F32, stack.ACT_RELU2, None, 0.0))
    torch.cuda.synchronize()
    capi.check(stack.lib().vkl_project_bf16w(x.data_ptr(), xtype, x.stride(0), w.data_ptr(), M, N, K,
                                             stack.segments(segs), len(segs), dev.stream))
    dev.sync()
    xd, wd = x.double(), w.double()
    want, mag = xd @ wd.t(), xd.abs() @ wd.abs().t()
    # exact products, K (planes: and 2 K small ones) of them added sixteen at a time, the 32-bit instructions two: 2^-23 of the sum of
    # magnitudes each; a square doubles that
    bound = K / 2 * 2.0 ** -23 * mag + 2.0 ** -23
    assert bool(((a - res - want[:, :cut]).abs() <= bound[:, :cut] + 2.0 ** -23 * (res.abs() + mag[:, :cut])).all())
    if xtype == stack.F32 and (K > 512 or M * N * K > 1 << 30):
        # In planes.  Without the third x loses 2.4e-6 of itself, without the second 1.6e-3 (in 64 bits, over these shapes).  All
        # three are exact; each step of 16 products rounds its partial sum by up to 2^-24 of itself, 3 K / 16 of them where
        # the planes share their accumulators: sqrt (3 K / 16) 2^-24 / sqrt (3) or less, 1.1e-6 at K = 5504 (seen: 2e-7)
        off = (a - res - want[:, :cut]).norm() / want[:, :cut].norm()
        assert float(off) < (K / 16) ** 0.5 * 2.0 ** -24, float(off)
    if N > cut:
        y, e = want[:, cut:].clamp_min(0), bound[:, cut:]
        assert bool(((b[:, :N - cut] - y * y).abs() <= 2 * y * e + e * e + 2.0 ** -22 * y * y).all())
        assert bool((b[:, N - cut:] == 7.0).all())
