"""The 32-bit product on the bf16 matrix cores, against 64 bits."""
import math

import pytest

from vkllama_amd import capi
from vkllama_amd import stack

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def project(dev, x, w, segs):
    M, K = x.shape
    torch.cuda.synchronize()
    capi.check(stack.lib().vkl_project_bf16w(x.data_ptr(), stack.F32, x.stride(0), w.data_ptr(), M, w.shape[0], K,
                                             stack.segments(segs), len(segs), dev.stream))
    dev.sync()


# rows: one, around a tile, several; inner sizes on both sides of the rule; more rows than the planes' scratch holds
@pytest.mark.parametrize("M,N,K", [(1, 40, 576), (2, 128, 512), (127, 264, 640), (129, 72, 1024), (257, 512, 2048),
                                   (1100, 200, 5504), (4100, 2048, 256), (33, 1000, 64)])
def test_three_planes(dev, M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn((M, K + 64), generator=g, device="cuda")[:, :K]
    x = x * torch.exp(2 * torch.randn((M, 1), generator=g, device="cuda"))
    x = torch.nn.functional.pad(x, (0, 64))[:, :K]                 # rows further apart than they are long
    w = torch.randn((N, K), generator=g, device="cuda").bfloat16()
    cut = N // 2 // 8 * 8
    res = torch.randn((M, cut + 3), generator=g, device="cuda")
    a, b = torch.full((M, cut + 3), 7.0, device="cuda"), torch.full((M, N - cut), math.nan, device="cuda")
    project(dev, x, w, [(0, cut, a.data_ptr(), cut + 3, stack.F32, 0, res.data_ptr(), 0.0),
                        (cut, N - cut, b.data_ptr(), N - cut, stack.F32, 0, None, 0.0)])
    xd, wd = x.double(), w.double()
    want, mag = xd @ wd.t(), xd.abs() @ wd.abs().t()
    # products are exact; of the 3 K of them sixteen enter an fp32 sum at a time (the 32-bit instructions: two), each of
    # which is off by at most 2^-23 of the sum of magnitudes; one more rounding for the residual
    bound = (3 * K / 16 if K > 512 else K / 2) * 2.0 ** -23 * mag + 2.0 ** -23
    assert bool((a[:, cut:] == 7.0).all())
    assert bool(((a[:, :cut] - res[:, :cut] - want[:, :cut]).abs() <= bound[:, :cut] + 2.0 ** -23 * (res[:, :cut].abs() + mag[:, :cut])).all())
    assert bool(((b - want[:, cut:]).abs() <= bound[:, cut:]).all())


def test_values_without_a_fraction_of_three_planes(dev):
    """Infinities and NaN stay where they are; the largest numbers do not overflow a plane."""
    x = torch.randn((6, 1024), device="cuda")
    x[1, 3], x[2, 5], x[3, 7] = math.inf, math.nan, -math.inf
    x[4] = 3.4e38                                                   # rounds to infinity in bf16
    w = torch.zeros((128, 1024), device="cuda", dtype=torch.bfloat16)
    w[:, 3], w[:, 5], w[:, 7], w[:, 0] = 1.0, 1.0, 1.0, 0.5
    y = torch.zeros((6, 128), device="cuda")
    project(dev, x, w, [(0, 128, y.data_ptr(), 128, stack.F32, 0, None, 0.0)])
    want = (x[:, 3] + x[:, 5] + x[:, 7] + 0.5 * x[:, 0]).unsqueeze(1).expand(6, 128)
    x4 = torch.tensor(math.inf)                                     # 3.5 times 3.4e38
    assert torch.equal(torch.isnan(y), torch.isnan(want)) and torch.equal(torch.isinf(y[:4]), torch.isinf(want[:4]))
    assert bool((y[4] == x4.to(y.device)).all()) and float(y[3, 0]) == -math.inf
    assert bool(((y[[0, 5]] - want[[0, 5]]).abs() < 1e-6).all())
