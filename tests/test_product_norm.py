"""A product with the norm of its rows against the product and the norm, over every family of products."""
import numpy as np
import pytest

from vkllama_amd import capi

pytestmark = pytest.mark.gpu


def weights(dev, rng, N, K, q8):
    if not q8:
        return dev.upload((rng.standard_normal((N, K)) * K ** -0.5).astype(np.float16))
    raw = np.empty((N, K // 32, 34), np.uint8)
    raw[:, :, :2] = rng.uniform(0.5, 1.5, (N, K // 32)).astype(np.float16).view(np.uint8).reshape(N, -1, 2)
    raw[:, :, :2] = (rng.uniform(0.5, 1.5, (N, K // 32)) / 64 * K ** -0.5).astype(np.float16).view(np.uint8).reshape(N, -1, 2)
    raw[:, :, 2:] = rng.integers(-127, 128, (N, K // 32, 32), dtype=np.int8).view(np.uint8)
    return dev.upload_q8_0(raw.reshape(N, -1), N, K)


# one row, slices of up to 32 rows, whole inner sizes, the general tiles and the wide ones with and without parts; rows of
# up to 2048, 4096, 6144, 8192 values and more, and of an odd number; few rows of as many parts as one launch takes, and of more
@pytest.mark.parametrize("q8", [True, False])
@pytest.mark.parametrize("M,N,K", [(1, 512, 1376), (2, 520, 64), (12, 2048, 2048), (31, 4096, 1408), (33, 4104, 4096), (77, 2056, 5504),
                                   (77, 4096, 11008), (130, 5120, 5120), (300, 4096, 4096), (40, 8200, 2048), (9, 130, 96), (200, 1000, 2048),
                                   (3, 5120, 5120), (33, 6144, 2048), (33, 6152, 2048), (64, 8192, 2048), (3, 5120, 11008), (3, 5120, 13824), (5, 4096, 11008),
                                   (3, 8192, 8192)])
def test_product_norm(dev, M, N, K, q8):
    rng = np.random.default_rng(M + N + K)
    L, w = capi.lib(), weights(dev, rng, N, K, q8)
    x, res = (dev.upload(rng.standard_normal(s).astype(np.float16)) for s in ((M, K), (M, N)))
    g = dev.upload(rng.uniform(0.5, 1.5, N).astype(np.float32))
    out = [dev.alloc(M * N * 2) for _ in range(4)]
    for r in (res.ptr, None):
        for o in out:
            o.write(np.full(M * N, 0x7e00, np.uint16))
        if q8:
            capi.check(L.vkl_matmul_q8_0(x.ptr, w.ptr, M, N, K, K, N, 1.0, 0.0, 0, r, out[0].ptr, None, dev.stream))
            fused = L.vkl_matmul_norm_q8_0
        else:
            capi.check(L.vkl_matmul_f16_tb(x.ptr, w.ptr, 1, M, N, K, 0, K, 0, K, 0, N, 1.0, 0.0, 0, r, out[0].ptr, None, dev.stream))
            fused = L.vkl_matmul_norm_f16
        capi.check(L.vkl_rmsnorm_f16(out[0].ptr, g.ptr, M, N, 1e-5, out[1].ptr, dev.stream))
        capi.check(fused(x.ptr, w.ptr, M, N, K, r, out[2].ptr, g.ptr, 1e-5, out[3].ptr, dev.stream))
        dev.sync()
        a, b, c, d = (o.read(np.uint16, (M, N)) for o in out)
        assert not (b == 0x7e00).any()
        assert np.array_equal(a, c)
        # (the same fp32 value before the last rounding; a tie of it between two fp16 numbers may go either way)
        assert (np.abs(b.astype(np.int32) - d.astype(np.int32)) <= 1).all()
        assert (b != d).mean() <= 2e-3
