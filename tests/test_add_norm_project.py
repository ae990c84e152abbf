"""A product added into the residual rows, their norm and the next product in one call: the same as the three calls, bit for
bit, whichever launches it takes."""
import ctypes as C
import math

import pytest

from vkllama_amd import capi
from vkllama_amd import stack

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

EPS = 1e-5


def pad(n):
    return (n + 63) // 64 * 64


class Rows:
    """Operands of a call, and two copies of what it writes"""

    def __init__(self, M, W, K, N, dtype):
        g = torch.Generator(device="cuda").manual_seed(M + W + K)
        self.M, self.W, self.K, self.N, self.Wp = M, W, K, N, pad(W)
        self.type = stack.F32 if dtype == torch.float32 else stack.BF16
        r = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
        self.x, self.w = r(M, K).to(dtype), r(W, K).bfloat16()
        self.norm = torch.nn.functional.pad(r(W), (0, self.Wp - W))
        self.next = r(N, self.Wp).bfloat16()
        self.y0 = r(M, self.Wp)
        self.y = [self.y0.clone() for _ in range(2)]
        self.h = [torch.full((M, self.Wp), 7.0, device="cuda", dtype=dtype) for _ in range(2)]
        self.out = [torch.full((M, N), 7.0, device="cuda") for _ in range(2)]

    def seg(self, i):
        return stack.segments([(0, self.N, self.out[i].data_ptr(), self.N, stack.F32, stack.ACT_GELU, None, 0.0)])

    def together(self, stream, add=True):
        p = stack.AddNormProject(x=self.x.data_ptr() if add else None, xs=self.K, w=self.w.data_ptr(), K=self.K,
                                 y=self.y[0].data_ptr(), ys=self.Wp, W=self.W, norm=self.norm.data_ptr(), eps=EPS,
                                 h=self.h[0].data_ptr(), hs=self.Wp, Wp=self.Wp, w_next=self.next.data_ptr(), N=self.N,
                                 segs=self.seg(0), nseg=1)
        capi.check(stack.lib().vkl_add_norm_project_bf16w(C.byref(p), self.type, self.M, stream))

    def apart(self, stream, add=True):
        y, h = self.y[1].data_ptr(), self.h[1].data_ptr()
        if add:
            back = stack.segments([(0, self.W, y, self.Wp, stack.F32, 0, y, 0.0)])
            capi.check(stack.lib().vkl_project_bf16w(self.x.data_ptr(), self.type, self.K, self.w.data_ptr(), self.M, self.W,
                                                     self.K, back, 1, stream))
        capi.check(stack.lib().vkl_rmsnorm_f32(y, self.Wp, None, self.M, self.W, self.norm.data_ptr(), EPS, h, self.type,
                                               self.Wp, self.Wp, stream))
        capi.check(stack.lib().vkl_project_bf16w(h, self.type, self.Wp, self.next.data_ptr(), self.M, self.N, self.Wp,
                                                 self.seg(1), 1, stream))

    def same(self):
        return all(torch.equal(a.view(torch.uint8), b.view(torch.uint8)) for a, b in (self.y, self.h, self.out))


# rows of parts and of one part, widths of one to eight loads per thread, padding, widths that no vector covers; planes in 64
# and in 256 rows, short products that take none
SHAPES = [(1, 2048, 5504, 512), (33, 2048, 2048, 1024), (300, 2048, 5504, 2048), (600, 1024, 1024, 512), (77, 4096, 4096, 512),
          (40, 5120, 1024, 256), (130, 2040, 2048, 264), (50, 2044, 1024, 128), (64, 512, 256, 128), (2048, 2048, 2048, 2048),
          (1500, 2048, 7552, 512)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,W,K,N", SHAPES)
def test_the_same_as_three_calls(dev, M, W, K, N, dtype):
    r = Rows(M, W, K, N, dtype)
    torch.cuda.synchronize()
    r.together(dev.stream)
    r.apart(dev.stream)
    dev.sync()
    assert r.same()
    want = r.y0[:, :W].double() + r.x.double() @ r.w.double().t()
    # products are exact, an fp32 sum of K of them is off by 2^-23 of the magnitudes for each addition at most
    bound = K * 2.0 ** -23 * (r.x.double().abs() @ r.w.double().abs().t()) + 2.0 ** -23 * want.abs() + 2.0 ** -23
    assert bool(((r.y[0][:, :W] - want).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_nothing_to_add(dev, dtype):
    r = Rows(300, 2048, 2048, 1024, dtype)
    torch.cuda.synchronize()
    r.together(dev.stream, add=False)
    r.apart(dev.stream, add=False)
    dev.sync()
    assert r.same() and torch.equal(r.y[0], r.y0)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_without_scratch(dev, dtype):
    r = Rows(300, 2048, 5504, 512, dtype)
    torch.cuda.synchronize()
    poor = C.c_void_p()
    capi.check(capi.lib().vkl_stream_create(C.byref(poor)))
    capi.check(capi.lib().vkl_debug_refuse_scratch(poor))
    r.together(poor)
    r.apart(poor)
    capi.check(capi.lib().vkl_stream_sync(poor))
    capi.check(capi.lib().vkl_stream_destroy(poor))
    assert r.same()


def test_values_that_planes_do_not_hold(dev):
    """Infinities, NaN and numbers below the planes' smallest, in rows of parts: the sums are formed again, the others stay."""
    r = Rows(40, 2048, 5504, 512, torch.float32)
    r.x[3, 5], r.x[7, 9], r.x[11] = math.inf, math.nan, 2.0 ** -120 * r.x[11]
    r.x[20, :] = 3.4e38
    torch.cuda.synchronize()
    r.together(dev.stream)
    r.apart(dev.stream)
    dev.sync()
    assert r.same()
    bad = ~torch.isfinite(r.y[0][:, :2048]).all(1)
    assert bad.nonzero().flatten().tolist() == [3, 7, 20]
