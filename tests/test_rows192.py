"""bf16 products in tiles of 192 token rows: whole and partly filled ones, pairs of 128 columns and the odd one, sums straight
from the registers, parked in LDS, and of parts of the k range."""
import pytest

from vkllama_amd import capi
from vkllama_amd import stack

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# one row beyond three tiles, rows that just fill tiles, a column range that ends inside a tile; with a residual in place
# (fp32) or an activation that is parked; four and eight parts; pairs of 128 columns with an odd column behind them (8064) or a
# last one in part, straight from the registers, parked, with a residual
@pytest.mark.parametrize("M,N,K,f32,act,parts,pairs", [
    (577, 8190, 512, False, stack.ACT_NONE, 1, 0), (768, 8192, 512, True, stack.ACT_NONE, 1, 0), (768, 5504, 1024, False, stack.ACT_GELU, 1, 0),
    (1300, 4232, 512, False, stack.ACT_RELU2, 1, 0), (1500, 3080, 1024, True, stack.ACT_NONE, 1, 0), (1153, 4096, 512, False, stack.ACT_NONE, 1, 0),
    (750, 2048, 6144, True, stack.ACT_NONE, 4, 0), (768, 1024, 11008, False, stack.ACT_GELU, 8, 0),
    (1500, 8064, 2048, False, stack.ACT_NONE, 1, 248), (1500, 8064, 1024, False, stack.ACT_GELU, 1, 248), (1300, 8190, 576, True, stack.ACT_NONE, 1, 224)])
def test_tiles_of_192_rows(dev, M, N, K, f32, act, parts, pairs):
    p = stack.project_plan(stack.BF16, M, N, K, stack.F32 if f32 else stack.BF16, act)
    assert (p.tile_rows, p.ksplit, p.pairs) == (192, parts, pairs)
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn((M, K), generator=g, device="cuda").bfloat16()
    w = torch.randn((N, K), generator=g, device="cuda").bfloat16()
    r = torch.randn((M, N + 8), generator=g, device="cuda")
    runs = []
    for _ in range(3):
        y = r.clone() if f32 else torch.full((M, N + 8), 7.0, device="cuda", dtype=torch.bfloat16)
        torch.cuda.synchronize()
        capi.check(stack.lib().vkl_project_bf16w(
            x.data_ptr(), stack.BF16, K, w.data_ptr(), M, N, K,
            stack.segments([(0, N, y.data_ptr(), N + 8, stack.F32 if f32 else stack.BF16, act, y.data_ptr() if f32 else None,
                             0.0)]), 1, dev.stream))
        dev.sync()
        runs.append(y)
    assert torch.equal(runs[0], runs[1]) and torch.equal(runs[0], runs[2])
    # exact products, K of them added in fp32: half of 2^-23 of the sum of magnitudes each
    xd, wd = x.double(), w.double()
    want, off = xd @ wd.t(), K / 2 * 2.0 ** -23 * (xd.abs() @ wd.abs().t())
    if act == stack.ACT_RELU2:
        off, want = 2 * want.abs() * off + off * off, want.clamp_min(0).square()
    elif act == stack.ACT_GELU:
        off, want = 1.13 * off + 2.0 ** -20 * want.abs() + 2.0 ** -22, torch.nn.functional.gelu(want)  # its slope is at most 1.13
    if f32:
        want = want + r[:, :N].double()
        off = off + 2.0 ** -23 * want.abs()
    else:
        # one rounding to bf16: seven bits behind the first one, half of the last is 2^-8 of the value at most
        off = off + 2.0 ** -22 * want.abs() + 2.0 ** -8 * (want.abs() + off) + 2.0 ** -133
    assert bool(((y[:, :N].double() - want).abs() <= off).all())
    assert torch.equal(y[:, N:], r[:, N:] if f32 else torch.full_like(y[:, N:], 7.0))
