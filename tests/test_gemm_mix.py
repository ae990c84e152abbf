"""Products of many token rows in tiles of 256, 128 and half as many rows and 256 or 128 columns, against 64 bits.

The sizes reach every kind of tile and their edges: whole rounds of column pairs with what is left in tiles of 128
columns, whole and cut; pairs alone; an odd last column; last rows and columns that fill part of a tile; fewer k-steps
than a tile has stages, and a remainder of them."""
import ctypes as C

import pytest

from vkllama_amd import capi
from vkllama_amd import stack

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def numbers(seed, *shape, dtype=torch.float16):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, generator=g, device="cuda").to(dtype)


def sums(x, w):
    """x w^T in 64 bits, and how far an fp32 sum of exact products may be off it"""
    xd, wd = x.double(), w.double()
    return xd @ wd.t(), x.shape[1] * 2.0 ** -23 * (xd.abs() @ wd.abs().t())


def rounded(v, bits):
    """error of rounding to a type of so many significant bits (and, of fp16, its smallest steps)"""
    return 2.0 ** -bits * v.abs() * 1.01 + 2.0 ** -24


# (2049, 8200): 256 pairs, then cut tiles and the odd column; (2300, 8320): the same with more k-steps than stages; (770, 12416):
# all pairs and an odd column; (384, 16500): pairs of 128-row tiles; (1025, 4100, 1088): tiles of 128 columns, 17 k-steps
F16 = [(2049, 8200, 64), (2300, 8320, 192), (770, 12416, 128), (384, 16500, 320), (200, 12292, 64), (1025, 4100, 1088),
       (66, 12000, 256), (256, 24577, 128)]


@pytest.mark.parametrize("M,N,K", F16)
def test_fp16(dev, M, N, K):
    x, w = numbers(1, M, K + 8)[:, :K], numbers(2, N, K)
    ys = (N + 7) // 8 * 8 + 8
    y = torch.full((M, ys), 7.0, device="cuda", dtype=torch.float16)
    torch.cuda.synchronize()
    capi.check(capi.lib().vkl_matmul_f16_tb(x.data_ptr(), w.data_ptr(), 1, M, N, K, M * (K + 8), K + 8, N * K, K, M * ys, ys,
                                            1.0, 0.0, 0, None, y.data_ptr(), None, dev.stream))
    dev.sync()
    want, off = sums(x, w)
    assert bool((y[:, N:] == 7.0).all())
    assert bool(((y[:, :N] - want).abs() <= off + rounded(want, 11)).all())


@pytest.mark.parametrize("M,N,K", [(600, 8200, 128), (512, 4096, 64)])
def test_fp16_scale_residual_and_wide_copy(dev, M, N, K):
    """What is parked in LDS: a scale, an activation, a residual and an fp32 copy."""
    x, w, r = numbers(1, M, K), numbers(2, N, K), numbers(3, M, N)
    y, y32 = torch.empty((M, N), device="cuda", dtype=torch.float16), torch.empty((M, N), device="cuda")
    torch.cuda.synchronize()
    capi.check(capi.lib().vkl_matmul_f16_tb(x.data_ptr(), w.data_ptr(), 1, M, N, K, M * K, K, N * K, K, M * N, N,
                                            0.25, 0.5, 1, r.data_ptr(), y.data_ptr(), y32.data_ptr(), dev.stream))
    dev.sync()
    v, off = sums(x, w)
    v, off = v * 0.25 + 0.5, off * 0.25 + 2.0 ** -22 * (v.abs() + 1)
    v = v * torch.sigmoid(v)
    off = 1.1 * off + 2.0 ** -20 * v.abs()                       # the slope of SiLU is at most 1.1
    off = off + rounded(v, 11)
    want = v + r.double()
    assert bool(((y - want).abs() <= off + rounded(want, 11)).all())
    assert torch.equal(y32, y.float())


@pytest.mark.parametrize("M,N,K", [(1300, 4096, 128), (2049, 4104, 64), (130, 4096, 192)])
def test_fp16_three_matrices(dev, M, N, K):
    x, ws = numbers(1, M, K), [numbers(2 + i, N, K) for i in range(3)]
    ys = [torch.empty((M, N), device="cuda", dtype=torch.float16) for _ in range(3)]
    torch.cuda.synchronize()
    capi.check(capi.lib().vkl_kqv_f16(x.data_ptr(), *[w.data_ptr() for w in ws], M, N, K, *[y.data_ptr() for y in ys], dev.stream))
    dev.sync()
    for w, y in zip(ws, ys):
        want, off = sums(x, w)
        assert bool(((y - want).abs() <= off + rounded(want, 11)).all())


# 86 and 17 blocks of 64 output columns, an odd number of them, columns that fill part of one
@pytest.mark.parametrize("M,N,K", [(2051, 5504, 192), (300, 8200, 64), (2300, 6208, 128), (100, 11392, 128)])
def test_fp16_up_and_gate(dev, M, N, K):
    x, up, gate = numbers(1, M, K), numbers(2, N, K), numbers(3, N, K)
    y = torch.empty((M, N), device="cuda", dtype=torch.float16)
    torch.cuda.synchronize()
    capi.check(capi.lib().vkl_ffn_upgate_f16(x.data_ptr(), up.data_ptr(), gate.data_ptr(), M, N, K, y.data_ptr(), dev.stream))
    dev.sync()
    (u, uo), (g, go) = sums(x, up), sums(x, gate)
    s = g * torch.sigmoid(g)
    want = s * u
    off = 1.1 * go * u.abs() + s.abs() * uo + go * uo + 2.0 ** -20 * want.abs() + rounded(want, 11)
    # (the largest products lie beyond fp16)
    ok = want.abs() < 65000
    assert bool(((y - want).abs() <= off)[ok].all()) and bool(torch.isinf(y[want.abs() > 66000]).all())


# segments: bf16, bf16 with an activation, fp32 with a residual in place, an unaligned one (parked); parts of the k range
# (512 x 2048 with 32 k-steps); 8064 columns: an odd number of 128
@pytest.mark.parametrize("M,N,K,act", [(1500, 8064, 192, stack.ACT_NONE), (2100, 8064, 64, stack.ACT_RELU2), (2049, 4104, 128, stack.ACT_GELU),
                                       (512, 2048, 2048, stack.ACT_GELU), (700, 16128, 64, stack.ACT_NONE), (300, 2048, 1088, stack.ACT_NONE)])
def test_bf16_segments(dev, M, N, K, act):
    x, w = numbers(1, M, K, dtype=torch.bfloat16), numbers(2, N, K, dtype=torch.bfloat16)
    n0, n1 = N // 3 // 8 * 8, N // 2 // 8 * 8
    a = torch.empty((M, n0), device="cuda", dtype=torch.bfloat16)
    b = torch.full((M, n1 - n0 + 3), 7.0, device="cuda", dtype=torch.bfloat16)
    c = numbers(3, M, N - n1, dtype=torch.float32)
    r = c.double()
    torch.cuda.synchronize()
    capi.check(stack.lib().vkl_project_bf16w(
        x.data_ptr(), stack.BF16, K, w.data_ptr(), M, N, K,
        stack.segments([(0, n0, a.data_ptr(), n0, stack.BF16, act, None, 0.0),
                        (n0, n1 - n0, b.data_ptr(), n1 - n0 + 3, stack.BF16, stack.ACT_NONE, None, 0.0),
                        (n1, N - n1, c.data_ptr(), N - n1, stack.F32, stack.ACT_NONE, c.data_ptr(), 0.0)]), 3, dev.stream))
    dev.sync()
    v, off = sums(x, w)
    va, oa = v[:, :n0], off[:, :n0]
    if act == stack.ACT_RELU2:
        oa, va = 2 * va.abs() * oa + oa * oa, va.clamp_min(0).square()
    elif act == stack.ACT_GELU:
        oa, va = 1.13 * oa + 2.0 ** -20 * va.abs() + 2.0 ** -22, torch.nn.functional.gelu(va)  # its slope is at most 1.13
    assert bool(((a - va).abs() <= oa + 2.0 ** -22 * va.abs() + rounded(va, 8)).all())
    assert bool((b[:, n1 - n0:] == 7.0).all())
    assert bool(((b[:, :n1 - n0] - v[:, n0:n1]).abs() <= off[:, n0:n1] + rounded(v[:, n0:n1], 8)).all())
    want = v[:, n1:] + r
    assert bool(((c - want).abs() <= off[:, n1:] + 2.0 ** -23 * want.abs()).all())


# what is parked in LDS in tiles whose loads go on past the end of the k range, at inner sizes of models: 256 x 256
# (GELU), 256 x 128 in two and four parts, 128 x 256 (a scale), a fused pair of an odd width
@pytest.mark.parametrize("kind,M,N,K", [("gelu", 2048, 11008, 4096), ("bf16", 1500, 2048, 7552), ("f16", 300, 4096, 11008),
                                        ("f16", 512, 5120, 13824), ("scale", 384, 16500, 320), ("pair", 2300, 6201, 1024)])
def test_parked_sums(dev, kind, M, N, K):
    bf = kind in ("gelu", "bf16")
    x, w = (numbers(1 + i, n, K, dtype=torch.bfloat16 if bf else torch.float16) for i, n in enumerate((M, N)))
    gate = numbers(3, N, K) if kind == "pair" else None
    if not bf:                                                   # (bf16 products have no such plan to ask for)
        p = capi.GemmPlan()
        assert capi.lib().vkl_gemm_plan(M, N, K, 1, 1, int(kind == "pair"), 0, C.byref(p)) == 0
        assert (p.family, p.tile_rows, p.ksplit) == (5, 128 if kind == "scale" else 256, {11008: 4, 13824: 2}.get(K, 1))
    scale = 2.0 ** -6 if kind == "scale" else 1.0
    out = []
    for _ in range(3):
        y = torch.full((M, N), 7.0, device="cuda", dtype=torch.float32 if bf else torch.float16)
        torch.cuda.synchronize()
        if bf:
            act = stack.ACT_GELU if kind == "gelu" else stack.ACT_NONE
            e = stack.lib().vkl_project_bf16w(x.data_ptr(), stack.BF16, K, w.data_ptr(), M, N, K,
                                              stack.segments([(0, N, y.data_ptr(), N, stack.F32, act, None, 0.0)]), 1, dev.stream)
        elif kind == "pair":
            e = capi.lib().vkl_ffn_upgate_f16(x.data_ptr(), w.data_ptr(), gate.data_ptr(), M, N, K, y.data_ptr(), dev.stream)
        else:
            e = capi.lib().vkl_matmul_f16_tb(x.data_ptr(), w.data_ptr(), 1, M, N, K, M * K, K, N * K, K, M * N, N, scale, 0.0, 0,
                                             None, y.data_ptr(), None, dev.stream)
        capi.check(e)
        dev.sync()
        out.append(y)
    assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])
    want, off = sums(x, w)
    if kind == "gelu":
        off, want = 1.13 * off + 2.0 ** -20 * want.abs() + 2.0 ** -22, torch.nn.functional.gelu(want)  # its slope is at most 1.13
    elif kind == "pair":
        g, go = sums(x, gate)
        s = g * torch.sigmoid(g)
        off = 1.1 * go * want.abs() + s.abs() * off + go * off + 2.0 ** -20 * (s * want).abs()
        want = s * want
    want, off = want * scale, off * scale
    off = off + (0 if bf else rounded(want, 11))
    ok = want.abs() < 65000 if kind == "pair" else torch.ones_like(want, dtype=torch.bool)
    assert bool(((out[0] - want).abs() <= off)[ok].all())


class Q8:
    """A Q8_0 matrix of random quants and scales, in the library's layout and in 64 bits"""

    def __init__(self, dev, seed, n, k):
        g = torch.Generator(device="cuda").manual_seed(seed)
        q = torch.randint(-127, 128, (n, k // 32, 32), generator=g, device="cuda", dtype=torch.int8)
        d = (torch.rand((n, k // 32, 1), generator=g, device="cuda") * 0.01 + 0.001).half()
        raw = torch.cat([d.view(torch.uint8).view(n, k // 32, 2), q.view(torch.uint8)], -1)
        self.wide = (q.double() * d.double()).view(n, k)
        self.buf = dev.upload_q8_0(raw.view(n, -1).cpu().numpy(), n, k)


# (2049, 8200): 256 pairs of columns, then cut tiles and the odd column; (2300, 8320): the same with more k-steps than
# stages; (1025, 16390): pairs, then whole tiles of 128 columns; the last two: tiles of 128 rows
@pytest.mark.parametrize("M,N,K", [(2049, 8200, 64), (2300, 8320, 320), (1025, 16390, 192), (770, 16500, 128), (512, 4096, 256)])
def test_q8_0(dev, M, N, K):
    x, w = numbers(1, M, K), Q8(dev, 2, N, K)
    ys = (N + 7) // 8 * 8 + 8
    y = torch.full((M, ys), 7.0, device="cuda", dtype=torch.float16)
    torch.cuda.synchronize()
    capi.check(capi.lib().vkl_matmul_q8_0(x.data_ptr(), w.buf.ptr, M, N, K, K, ys, 1.0, 0.0, 0, None, y.data_ptr(), None, dev.stream))
    dev.sync()
    want, off = sums(x, w.wide)
    assert bool((y[:, N:] == 7.0).all())
    assert bool(((y[:, :N] - want).abs() <= off + rounded(want, 11)).all())


# with and without what is parked in LDS
@pytest.mark.parametrize("M,N,K,scale,act,copy", [(2049, 8200, 64, 1.0, 0, False), (2049, 8200, 128, 0.25, 1, False), (1030, 16384, 64, 1.0, 0, True)])
def test_q8_0_with_a_residual(dev, M, N, K, scale, act, copy):
    x, w, r = numbers(1, M, K), Q8(dev, 2, N, K), numbers(3, M, N)
    y, y32 = torch.empty((M, N), device="cuda", dtype=torch.float16), torch.empty((M, N), device="cuda")
    torch.cuda.synchronize()
    capi.check(capi.lib().vkl_matmul_q8_0(x.data_ptr(), w.buf.ptr, M, N, K, K, N, scale, 0.0, act, r.data_ptr(), y.data_ptr(),
                                          y32.data_ptr() if copy else None, dev.stream))
    dev.sync()
    v, off = sums(x, w.wide)
    v, off = v * scale, off * scale + 2.0 ** -22 * v.abs()
    if act:
        v = v * torch.sigmoid(v)
        off = 1.1 * off + 2.0 ** -20 * v.abs()
    off = off + rounded(v, 11)
    want = v + r.double()
    assert bool(((y - want).abs() <= off + rounded(want, 11)).all())
    assert not copy or torch.equal(y32, y.float())


@pytest.mark.parametrize("M,N,K", [(2049, 4104, 64), (1300, 4096, 192)])
def test_q8_0_three_matrices(dev, M, N, K):
    x, ws = numbers(1, M, K), [Q8(dev, 2 + i, N, K) for i in range(3)]
    ys = [torch.empty((M, N), device="cuda", dtype=torch.float16) for _ in range(3)]
    torch.cuda.synchronize()
    capi.check(capi.lib().vkl_kqv_q8_0(x.data_ptr(), *[w.buf.ptr for w in ws], M, N, K, *[y.data_ptr() for y in ys], dev.stream))
    dev.sync()
    for w, y in zip(ws, ys):
        want, off = sums(x, w.wide)
        assert bool(((y - want).abs() <= off + rounded(want, 11)).all())


@pytest.mark.parametrize("M,N,K", [(2051, 5504, 192), (2300, 6208, 128), (1030, 8212, 64)])
def test_q8_0_up_and_gate(dev, M, N, K):
    x, up, gate = numbers(1, M, K), Q8(dev, 2, N, K), Q8(dev, 3, N, K)
    y = torch.empty((M, N), device="cuda", dtype=torch.float16)
    torch.cuda.synchronize()
    capi.check(capi.lib().vkl_ffn_upgate_q8_0(x.data_ptr(), up.buf.ptr, gate.buf.ptr, M, N, K, y.data_ptr(), dev.stream))
    dev.sync()
    (u, uo), (g, go) = sums(x, up.wide), sums(x, gate.wide)
    s = g * torch.sigmoid(g)
    want = s * u
    off = 1.1 * go * u.abs() + s.abs() * uo + go * uo + 2.0 ** -20 * want.abs() + rounded(want, 11)
    assert bool(((y - want).abs() <= off).all())


# 88 to 128 tiles of 128 x 128, each of which is cut by its columns: k ranges shorter than the six stages, as long and longer;
# columns that end in the first and in the second half of the last tile (of the fused pair 64 of either), and none in its second half
@pytest.mark.parametrize("kind,M,N,K", [("one", 128, 12300, 64), ("one", 100, 12280, 320), ("one", 66, 12352, 384), ("one", 128, 12300, 448),
                                        ("one", 256, 8008, 1088), ("three", 128, 4104, 64), ("three", 100, 4096, 320), ("three", 250, 1944, 832),
                                        ("pair", 500, 1376, 64), ("pair", 250, 4040, 192), ("pair", 128, 5600, 384), ("pair", 400, 2048, 512)])
def test_fp16_few_tiles(dev, kind, M, N, K):
    p = capi.GemmPlan()
    assert capi.lib().vkl_gemm_plan(M, N, K, 1, 3 if kind == "three" else 1, int(kind == "pair"), 0, C.byref(p)) == 0
    tiles = -(-M // 128) * -(-N // (64 if kind == "pair" else 128)) * (3 if kind == "three" else 1)
    assert (p.family, p.tile_rows, p.ksplit) == (5, 128, 1) and tiles <= 128
    if kind == "pair":
        test_fp16_up_and_gate(dev, M, N, K)
    elif kind == "three":
        test_fp16_three_matrices(dev, M, N, K)
    else:
        test_fp16(dev, M, N, K)
        if N % 8 == 0:
            test_fp16_scale_residual_and_wide_copy(dev, M, N, K)
