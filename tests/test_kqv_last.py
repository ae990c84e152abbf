"""K, V and one row of Q against 64 bits, on both sides of the sizes from which the other rows are left out."""
import math

import numpy as np
import pytest

import util as U
from vkllama_amd import capi

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


FORMED = [(w, M, N, K) for w, N, K in ((1, 1152, 1024), (1, 1160, 1064), (1, 1150, 1030), (8, 1152, 1024), (8, 1160, 1056), (8, 1154, 1088))
          for M in (1, 2, 70, 639, 700, 1025)] + [(8, 768, 1024, 1024)]
# rows that end inside a tile, columns too
LEFT_OUT = [(1, 641, 4096, 512), (1, 515, 4104, 640), (1, 1300, 2056, 576), (1, 3001, 1152, 1024), (8, 257, 4104, 576), (8, 1025, 1160, 512),
            (8, 641, 2176, 512), (8, 1500, 1152, 1024)]


@pytest.mark.parametrize("wtype,M,N,K", FORMED + LEFT_OUT)
def test_kqv_last(dev, wtype, M, N, K):
    rng = np.random.default_rng(M * 7 + N + K)
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float16)).cuda()
    if wtype == 8:
        raw = [U.q8_weights(rng, N, K) for _ in range(3)]
        held = [dev.upload_q8_0(r[0], N, K) for r in raw]
        ptr, w = [h.ptr for h in held], [torch.from_numpy(r[1][:, :K]).cuda() for r in raw]
    else:
        held = [torch.from_numpy((rng.standard_normal((N, K)) * K ** -0.5).astype(np.float16)).cuda() for _ in range(3)]
        ptr, w = [h.data_ptr() for h in held], [h.double() for h in held]
    y = [torch.full((M, N), math.nan, device="cuda", dtype=torch.float16) for _ in range(3)]
    torch.cuda.synchronize()
    capi.check(capi.lib().vkl_kqv_last(x.data_ptr(), *ptr, wtype, M, N, K, *(t.data_ptr() for t in y), dev.stream))
    dev.sync()
    for i in range(3):
        rows = slice(M - 1, M) if i == 1 else slice(0, M)
        want, mag = x[rows].double() @ w[i].t(), x[rows].double().abs() @ w[i].abs().t()
        # one rounding to fp16 and at most K of fp32 sums
        bound = 2.0 ** -11 * want.abs() + K * 2.0 ** -24 * mag + 2.0 ** -25
        assert bool(((y[i][rows].double() - want).abs() <= bound).all()), i


def test_arguments_are_checked(dev):
    b = dev.alloc(64)
    lib = capi.lib()
    assert lib.vkl_kqv_last(b.ptr, b.ptr, None, b.ptr, 1, 1, 1, 8, b.ptr, b.ptr, b.ptr, dev.stream) != 0
    assert lib.vkl_kqv_last(b.ptr, b.ptr, b.ptr, b.ptr, 2, 1, 1, 8, b.ptr, b.ptr, b.ptr, dev.stream) != 0
    assert lib.vkl_kqv_last(b.ptr, b.ptr, b.ptr, b.ptr, 8, 0, 1, 32, b.ptr, b.ptr, b.ptr, dev.stream) != 0
