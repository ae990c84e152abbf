"""The fused fp16 projections against 64 bits, over the row counts at which the kernel families hand over."""
import math

import pytest

from vkllama_amd import capi

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 2, 3, 32, 33, 64, 65, 130, 300])
@pytest.mark.parametrize("N,K", [(512, 512), (520, 1376), (4096, 256)])
def test_kqv_f16(dev, M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M * 7 + N + K)
    x = torch.randn((M, K), generator=g, device="cuda").half()
    w = [(torch.randn((N, K), generator=g, device="cuda") * K ** -0.5).half() for _ in range(3)]
    y = [torch.full((M, N), math.nan, device="cuda", dtype=torch.float16) for _ in range(3)]
    torch.cuda.synchronize()
    capi.check(capi.lib().vkl_kqv_f16(x.data_ptr(), w[0].data_ptr(), w[1].data_ptr(), w[2].data_ptr(), M, N, K,
                                      y[0].data_ptr(), y[1].data_ptr(), y[2].data_ptr(), dev.stream))
    dev.sync()
    for i in range(3):
        want, mag = x.double() @ w[i].double().t(), x.double().abs() @ w[i].double().abs().t()
        # one rounding to fp16 and at most K of fp32 sums
        bound = 2.0 ** -11 * want.abs() + K * 2.0 ** -24 * mag + 2.0 ** -25
        assert bool(((y[i].double() - want).abs() <= bound).all()), i


def test_arguments_are_checked(dev):
    b = dev.alloc(64)
    lib = capi.lib()
    assert lib.vkl_kqv_f16(b.ptr, b.ptr, None, b.ptr, 1, 1, 8, b.ptr, b.ptr, b.ptr, dev.stream) != 0
    assert lib.vkl_kqv_f16(b.ptr, b.ptr, b.ptr, b.ptr, 0, 1, 8, b.ptr, b.ptr, b.ptr, dev.stream) != 0
