"""The GELU of a product against 64 bits: the unit matrix brings every x to the activation as it is."""
import math

import pytest

from vkllama_amd import capi
from vkllama_amd import stack

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def gelu(dev, x):
    """x [M, 64] fp32 of bf16 values"""
    w = torch.eye(64, device="cuda").bfloat16()
    y = torch.full_like(x, 7.0)
    torch.cuda.synchronize()
    capi.check(stack.lib().vkl_project_bf16w(x.data_ptr(), stack.F32, 64, w.data_ptr(), x.shape[0], 64, 64,
                                             stack.segments([(0, 64, y.data_ptr(), 64, stack.F32, stack.ACT_GELU, None, 0.0)]), 1, dev.stream))
    dev.sync()
    return y


def test_gelu(dev):
    x = torch.cat([torch.linspace(-13, 13, 64 * 4000), torch.logspace(-30, 1, 64 * 100), -torch.logspace(-30, 1, 64 * 100)]).cuda()
    x = x.bfloat16().float().view(-1, 64)
    y, xd = gelu(dev, x).double(), x.double()
    want = 0.5 * xd * torch.erfc(-xd / math.sqrt(2.0))
    err = (y - want).abs()
    # the polynomial is off by 2.1e-7 of h, its argument's power by x^2 / 2 roundings; the rest are some four roundings
    assert bool((err <= (2.1e-7 + (6 + 0.5 * xd.square()) * 2.0 ** -24) * want.abs() + 2.0 ** -126).all())
    assert float(err.max()) < 4.5e-7 * 13 / 9                     # 1 + erff: 4.5e-7 over |x| < 9


def test_gelu_of_the_odd(dev):
    x = torch.zeros((1, 64), device="cuda")
    x[0, 0] = 3.0e38
    y = gelu(dev, x)
    assert float(y[0, 0]) == float(x[0, 0]) and bool((y[0, 1:] == 0).all())
    x[0, 0] = -3.0e38
    assert float(gelu(dev, x)[0, 0]) == 0.0
