"""The GELU of a product against 64 bits: the unit matrix brings every x to the activation as it is (the planes of an fp32
value add up to it without a rounding)."""
import math

import pytest

from vkllama_amd import capi
from vkllama_amd import stack

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

EDGES = [-13, -9, -6, -3, -2, -1.5, -1, -0.5, -0.1, 0, 0.1, 0.5, 1, 1.5, 2, 3, 6, 9, 13]


def gelu(dev, x):
    """x [M, 64] fp32"""
    w = torch.eye(64, device="cuda").bfloat16()
    y = torch.full_like(x, 7.0)
    torch.cuda.synchronize()
    capi.check(stack.lib().vkl_project_bf16w(x.data_ptr(), stack.F32, 64, w.data_ptr(), x.shape[0], 64, 64,
                                             stack.segments([(0, 64, y.data_ptr(), 64, stack.F32, stack.ACT_GELU, None, 0.0)]), 1, dev.stream))
    dev.sync()
    return y


@pytest.mark.parametrize("low,high", list(zip(EDGES, EDGES[1:])))
def test_gelu(dev, low, high):
    g = torch.Generator().manual_seed(EDGES.index(low))
    x = low + (high - low) * torch.rand(64 * 2000, generator=g, dtype=torch.float64)
    if 0 in (low, high):
        x = torch.cat([x, (low + high) * torch.logspace(-30, 0, 64 * 200, dtype=torch.float64)])
    x = x.float().cuda().view(-1, 64)
    y, xd = gelu(dev, x).double(), x.double()
    z = xd / math.sqrt(2.0)
    want = 0.5 * xd * torch.erfc(-z)
    # x (1 + erf z) / 2: two roundings of z, 2^-24 each, times the slope of erf; erf off by two units of its last place at most;
    # a rounding of the sum and one of the product
    erf, slope, u = torch.erf(z).abs(), 2 / math.sqrt(math.pi) * torch.exp(-z * z), 2.0 ** -24
    bound = 0.5 * xd.abs() * (2 * u * z.abs() * slope + 4 * u * erf + 2 * u * torch.erfc(-z))
    assert bool(((y - want).abs() <= bound + 2.0 ** -126).all())


def test_gelu_of_the_odd(dev):
    x = torch.zeros((1, 64), device="cuda")
    x[0, 0] = 3.0e38
    y = gelu(dev, x)
    assert float(y[0, 0]) == float(x[0, 0]) and bool((y[0, 1:] == 0).all())
    x[0, 0] = -3.0e38
    assert float(gelu(dev, x)[0, 0]) == 0.0
