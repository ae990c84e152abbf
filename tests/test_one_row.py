"""The fused up/gate product of one row, Q8_0 weights, against 64 bits."""
import numpy as np
import pytest

from vkllama_amd import capi

pytestmark = pytest.mark.gpu


def blocks(q, d):
    n, k = q.shape
    raw = np.empty((n, k // 32, 34), np.uint8)
    raw[:, :, :2] = d.view(np.uint8).reshape(n, -1, 2)
    raw[:, :, 2:] = q.view(np.uint8).reshape(n, -1, 32)
    return raw.reshape(n, -1)


@pytest.mark.parametrize("N,K", [(2, 32), (30, 64), (700, 1376), (4098, 512), (1376, 4128), (64, 12320)])
def test_up_gate_q8_0(dev, N, K):
    rng = np.random.default_rng(N + K)
    x = rng.standard_normal(K).astype(np.float16)
    ws, want = [], []
    for _ in range(2):
        q = rng.integers(-127, 128, (N, K), dtype=np.int8)
        d = rng.uniform(0.5, 1.5, (N, K // 32)).astype(np.float16) * np.float16(K ** -0.5 / 64)
        ws.append(dev.upload_q8_0(blocks(q, d), N, K))
        w = q.astype(np.float64).reshape(N, -1, 32) * d.astype(np.float64)[:, :, None]
        want.append(w.reshape(N, K) @ x.astype(np.float64))
    up, gate = want
    y, dx = dev.alloc(N * 2), dev.upload(x)
    capi.check(capi.lib().vkl_ffn_upgate_q8_0(dx.ptr, ws[0].ptr, ws[1].ptr, 1, N, K, y.ptr, dev.stream))
    dev.sync()
    got = y.read(np.uint16, (N,)).view(np.float16).astype(np.float64)
    want = gate / (1 + np.exp(-gate)) * up
    # sums of order one: fp32 roundings of some 1e-6 of them, one rounding to fp16
    assert (np.abs(got - want) <= 2.0 ** -11 * np.abs(want) + 2e-5).all()


@pytest.mark.parametrize("N", [(1 << 23) - 2, 1 << 23, (1 << 23) + 4096])   # on either side of what the step's kernel deals
@pytest.mark.parametrize("fused", [False, True])
def test_more_rows_than_32_bits_deal(dev, N, fused):
    """N rows times 512 workgroups no longer fit 32 bits: every row is written all the same."""
    K, P = 32, 4094
    rng = np.random.default_rng(N)
    x = rng.standard_normal(K).astype(np.float16)
    ws, want = [], []
    for _ in range(2):
        q = rng.integers(-127, 128, (P, K), dtype=np.int8)
        d = rng.uniform(0.5, 1.5, (P, 1)).astype(np.float16) * np.float16(K ** -0.5 / 64)
        ws.append(dev.upload_q8_0(np.resize(blocks(q, d), (N, 34)), N, K))
        want.append((q.astype(np.float64) * d.astype(np.float64)) @ x.astype(np.float64))
    y, dx = dev.alloc(N * 2), dev.upload(x)
    y.write(np.full(N, 0x7E00, np.uint16))
    if fused:
        capi.check(capi.lib().vkl_ffn_upgate_q8_0(dx.ptr, ws[0].ptr, ws[1].ptr, 1, N, K, y.ptr, dev.stream))
        want = want[1] / (1 + np.exp(-want[1])) * want[0]
    else:
        capi.check(capi.lib().vkl_matmul_q8_0(dx.ptr, ws[0].ptr, 1, N, K, K, N, 1.0, 0.0, 0, None, y.ptr, None, dev.stream))
        want = want[0]
    dev.sync()
    got = y.read(np.uint16, (N,)).view(np.float16).astype(np.float64)
    want = np.resize(want, N)
    assert (np.abs(got - want) <= 2.0 ** -11 * np.abs(want) + 2e-5).all()


@pytest.mark.parametrize("N,K", [(2, 32), (2, 64), (6, 96), (14, 64)])      # less than 1 KiB
@pytest.mark.parametrize("fused", [False, True])
def test_matrices_at_the_end_of_their_memory(dev, N, K, fused):
    """Waves without rows of their own request nothing behind a small matrix."""
    rng = np.random.default_rng(N * K)
    x, room = rng.standard_normal(K).astype(np.float16), 1 << 21
    bufs, ptrs, want = [], [], []
    for _ in range(2):
        q = rng.integers(-127, 128, (N, K), dtype=np.int8)
        d = rng.uniform(0.5, 1.5, (N, K // 32)).astype(np.float16) * np.float16(K ** -0.5 / 64)
        planar = q.tobytes() + d.tobytes()
        at = (room - len(planar)) // 16 * 16
        whole = np.zeros(room, np.uint8)
        whole[at:at + len(planar)] = np.frombuffer(planar, np.uint8)
        bufs.append(dev.upload(whole))
        ptrs.append(bufs[-1].ptr.value + at)
        want.append((q.reshape(N, -1, 32) * d.astype(np.float64)[:, :, None]).reshape(N, K) @ x.astype(np.float64))
    y, dx = dev.alloc(N * 2), dev.upload(x)
    if fused:
        capi.check(capi.lib().vkl_ffn_upgate_q8_0(dx.ptr, ptrs[0], ptrs[1], 1, N, K, y.ptr, dev.stream))
        want = want[1] / (1 + np.exp(-want[1])) * want[0]
    else:
        capi.check(capi.lib().vkl_matmul_q8_0(dx.ptr, ptrs[0], 1, N, K, K, N, 1.0, 0.0, 0, None, y.ptr, None, dev.stream))
        want = want[0]
    dev.sync()
    got = y.read(np.uint16, (N,)).view(np.float16).astype(np.float64)
    assert (np.abs(got - want) <= 2.0 ** -11 * np.abs(want) + 2e-5).all()
