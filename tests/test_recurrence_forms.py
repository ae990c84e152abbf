"""Which form a recurrence of few tokens takes by itself, with and without scratch memory, on either side of the rule."""
import numpy as np
import pytest

from test_fuzuvik_ops import F32, K, R, ok, recur_case, recur_plain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,at", [(12, 8), (23, 20), (60, 37), (100, 90)])
@pytest.mark.parametrize("delta", [True, False])
@pytest.mark.parametrize("what", ["k", "v"])
def test_how_far_a_value_that_is_not_finite_reaches(dev, rng, T, at, delta, what):
    H, dim, vdim = 3, 64, 32
    c = recur_case(rng, F32, T, H, 1, dim, vdim, delta)
    want = recur_plain(c, H, 1, dim, delta)
    bad = np.array(c[what][0]).reshape(T, -1)
    bad[at, 3] = np.nan
    d = {x: dev.upload(bad if x == what else c[x][0] if x in "qkv" else c[x]) for x in
         ("q", "k", "v", "z", "b", "dt", "rate", "log") if x in c}
    for form in (K.RECUR_TOKENS, K.RECUR_CHUNKS):
        state, y = dev.upload(np.zeros((H, dim, vdim), np.float32)), dev.alloc(T * H * vdim * 4)
        a = K.RecurrenceArgs()
        a.H, a.rep, a.dim, a.vdim, a.type, a.qscale = H, 1, dim, vdim, F32, 0.25
        a.q, a.k, a.v, a.qs, a.ks, a.vs = d["q"].ptr, d["k"].ptr, d["v"].ptr, H * dim, H * dim, H * vdim
        a.state, a.out, a.os = state.ptr, y.ptr, H * vdim
        if delta:
            a.z, a.zs, a.b, a.bs, a.unit_eps = d["z"].ptr, H * dim, d["b"].ptr, H, R.UNIT_EPS
            a.dt_bias, a.rate = d["dt"].ptr, d["rate"].ptr
        else:
            a.log_decay = d["log"].ptr
        n = K.lib().vkl_recurrence_scratch_bytes(a, T)
        scratch = dev.alloc(n)
        ok(K.lib().vkl_recurrence(a, T, 0, form, scratch.ptr, n, dev.stream))
        got = y.read(np.float32, (T, H, vdim))
        first = at if form == K.RECUR_TOKENS else at // 16 * 16
        assert np.isnan(got[at:, 0]).any(axis=1).all()                       # (values 3 are those of the first head)
        assert np.abs(got[:first] - want[:first]).max(initial=0) < 2e-5 * np.abs(want).max()
        assert np.abs(got[:, 1:] - want[:, 1:]).max() < 2e-5 * np.abs(want).max()


@pytest.mark.parametrize("T", [1, 4, 5, 16, 23, 24])
@pytest.mark.parametrize("delta", [True, False])
def test_few_tokens(dev, rng, T, delta):
    H, dim, vdim = 3, 64, 32
    c = recur_case(rng, F32, T, H, 1, dim, vdim, delta)
    want = recur_plain(c, H, 1, dim, delta)
    got = {}
    for form in ("tokens", "chunks", "auto", "auto without scratch"):
        state = dev.upload(np.zeros((H, dim, vdim), np.float32))
        d = {x: dev.upload(c[x][0] if x in "qkv" else c[x]) for x in ("q", "k", "v", "z", "b", "dt", "rate", "log") if x in c}
        y = dev.alloc(T * H * vdim * 4)
        a = K.RecurrenceArgs()
        a.H, a.rep, a.dim, a.vdim, a.type, a.qscale = H, 1, dim, vdim, F32, 0.25
        a.q, a.k, a.v, a.qs, a.ks, a.vs = d["q"].ptr, d["k"].ptr, d["v"].ptr, H * dim, H * dim, H * vdim
        a.state, a.out, a.os = state.ptr, y.ptr, H * vdim
        if delta:
            a.z, a.zs, a.b, a.bs, a.unit_eps = d["z"].ptr, H * dim, d["b"].ptr, H, R.UNIT_EPS
            a.dt_bias, a.rate = d["dt"].ptr, d["rate"].ptr
        else:
            a.log_decay = d["log"].ptr
        n = K.lib().vkl_recurrence_scratch_bytes(a, T)
        scratch = dev.alloc(n)
        chunked = T >= (5 if delta else 24)
        assert K.lib().vkl_recurrence_chunked(a, T) == chunked
        way = {"tokens": K.RECUR_TOKENS, "chunks": K.RECUR_CHUNKS}.get(form, K.RECUR_AUTO)
        rc = K.lib().vkl_recurrence(a, T, 0, way, None if "without" in form else scratch.ptr, 0 if "without" in form else n,
                                    dev.stream)
        if "without" in form and T >= 24:
            assert rc == 1
            continue
        ok(rc)
        got[form] = y.read(np.float32, (T, H, vdim))
        assert np.abs(got[form] - want).max() < 2e-5 * np.abs(want).max(), form
    assert np.array_equal(got["auto"], got["chunks" if chunked else "tokens"])
    if T < 24:
        assert np.array_equal(got["auto without scratch"], got["tokens"])
