"""Attention of few query rows over many keys (the key-split kernel) vs the f64 oracle: edges of
its 16-row and 16-key blocks and of its splits, every head dimension class, strided operands,
masks of the type's extremes, and a capture whose workspace may not grow."""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import pytest

from barracuda_amd import Tensor
from barracuda_amd import _native as N
from oracle import bc_oracle as O
from tests.test_gpu_graph import CAPTURE_RELAXED, _FreshCtx, _hip

pytestmark = pytest.mark.gpu
TOL = 1e-5  # f32 softmax and sums over N(0, 1) inputs: about 1e-6 of the largest output


def _run(dev, q, k, v, pad=0, ctx=None):
    """bch_sdpa_fwd_ex on [B, H, S, D] arrays; pad > 0 stores them [B, S, H * D + pad]."""
    def put(x):
        b, h, s, d = x.shape
        if not pad:
            return Tensor.from_data(x, [x.size], dev), N.AttnLayout(h * s * d, s * d, d)
        buf = np.full((b, s, h * d + pad), np.nan, np.float32)
        buf[:, :, :h * d] = x.transpose(0, 2, 1, 3).reshape(b, s, h * d)
        return Tensor.from_data(buf, [buf.size], dev), N.AttnLayout(s * (h * d + pad), d, h * d + pad)

    (b, h, sq, d), (_, hkv, skv, _) = q.shape, k.shape
    (tq, lq), (tk, lk), (tv, lv) = put(q), put(k), put(v)
    to, lo = put(np.full_like(q, 7.0))
    st = dev._lib.bch_sdpa_fwd_ex(ctx or dev.ctx, b, h, hkv, sq, skv, d, float(1.0 / np.sqrt(np.float32(d))), 0,
                                  C.c_void_p(tq.ptr), lq, C.c_void_p(tk.ptr), lk, C.c_void_p(tv.ptr), lv,
                                  C.c_void_p(to.ptr), lo)
    if ctx is not None:
        return st, to
    dev.check(st, "attention")
    out = to.to_numpy()
    if not pad:
        return out.reshape(q.shape)
    out = out.reshape(b, sq, h * d + pad)
    assert np.all(np.isnan(out[:, :, h * d:])), "padding written"
    return out[:, :, :h * d].reshape(b, sq, h, d).transpose(0, 2, 1, 3)


def _inputs(b, h, hkv, sq, skv, d):
    rng = np.random.default_rng(b + h * 3 + sq * 7 + skv + d)
    return (rng.standard_normal((b, h, sq, d), dtype=np.float32), rng.standard_normal((b, hkv, skv, d), dtype=np.float32),
            rng.standard_normal((b, hkv, skv, d), dtype=np.float32))


@pytest.mark.parametrize("pad", [0, 4])
@pytest.mark.parametrize("b,h,hkv,sq,skv,d", [
    (1, 1, 1, 1, 128, 64), (1, 1, 1, 1, 129, 128), (2, 4, 4, 1, 143, 4), (1, 4, 1, 1, 144, 36), (1, 15, 1, 1, 191, 68),
    (2, 16, 1, 1, 256, 100), (1, 17, 1, 1, 1000, 128), (3, 8, 2, 4, 777, 80), (1, 8, 1, 16, 1025, 128),
    (1, 2, 2, 16, 4099, 64), (8, 32, 8, 1, 2048, 128), (1, 32, 8, 1, 8191, 128), (40, 16, 16, 3, 130, 32)])
def test_decode_vs_f64(dev, b, h, hkv, sq, skv, d, pad):
    print(f"decode b={b} h={h} hkv={hkv} sq={sq} skv={skv} d={d} pad={pad}", flush=True)
    q, k, v = _inputs(b, h, hkv, sq, skv, d)
    got = _run(dev, q, k, v, pad)
    group = h // hkv
    want = O.sdpa_f64(q, np.repeat(k, group, 1), np.repeat(v, group, 1), False)
    assert O.max_rel_err(got, want) <= TOL
    assert np.array_equal(got, _run(dev, q, k, v, pad)), "not deterministic"


def test_decode_extreme_scores(dev):
    """Keys whose scores are the type's lowest value, -inf or far above the rest leave the
    others' weights as they are; a row of nothing but -inf, or with +inf or NaN in it, is NaN; an
    infinite value reaches its column."""
    b, h, sq, skv, d = 1, 4, 1, 600, 64
    q, k, v = _inputs(b, h, h, sq, skv, d)
    q[..., 0] = 1.0
    k[..., 0] = 0.0
    k[0, 0, 100:, 0] = -np.finfo(np.float32).max
    k[0, 1, :, 0] = -np.inf
    k[0, 2, 37, 0] = np.inf
    k[0, 3, ::2, 0] = -np.inf
    v[0, 0, 5, 3] = np.inf
    got = _run(dev, q, k, v)
    s = np.einsum("bhid,bhjd->bhij", q.astype(np.float64), k.astype(np.float64)) / math.sqrt(d)
    with np.errstate(invalid="ignore"):
        p = np.exp(s - s.max(-1, keepdims=True))
        want = (p / p.sum(-1, keepdims=True)) @ v.astype(np.float64)
    assert np.isinf(got[0, 0, 0, 3]) and np.all(np.isnan(got[0, 1])) and np.all(np.isnan(got[0, 2]))
    fin = np.isfinite(want)
    assert np.max(np.abs(got[fin] - want[fin])) <= 1e-5
    assert np.all(np.isfinite(got[0, 3]))


def test_decode_under_capture_without_workspace(dev):
    """A first call under capture may not grow the workspace: it runs unsplit, and replays."""
    hip = _hip()
    b, h, hkv, sq, skv, d = 1, 8, 2, 1, 2048, 128
    q, k, v = _inputs(b, h, hkv, sq, skv, d)
    want = O.sdpa_f64(q, np.repeat(k, 4, 1), np.repeat(v, 4, 1), False)
    tq, tk, tv, to = (Tensor.from_data(x, list(x.shape), dev) for x in (q, k, v, np.zeros_like(q)))
    lay = lambda heads, s: N.AttnLayout(heads * s * d, s * d, d)
    with _FreshCtx(dev) as f:
        call = lambda: f.lib.bch_sdpa_fwd_ex(f.ctx, b, h, hkv, sq, skv, d, 1.0 / math.sqrt(d), 0, C.c_void_p(tq.ptr),
                                             lay(h, sq), C.c_void_p(tk.ptr), lay(hkv, skv), C.c_void_p(tv.ptr),
                                             lay(hkv, skv), C.c_void_p(to.ptr), lay(h, sq))
        graph, exe = C.c_void_p(), C.c_void_p()
        assert hip.hipStreamBeginCapture(f.stream, CAPTURE_RELAXED) == 0
        st = call()
        assert hip.hipStreamEndCapture(f.stream, C.byref(graph)) == 0
        assert st == N.BCH_OK and f.ws_bytes() == 0
        try:
            assert hip.hipGraphInstantiate(C.byref(exe), graph, None, None, 0) == 0
            for _ in range(3):
                assert hip.hipGraphLaunch(exe, f.stream) == 0
                assert f.lib.bch_sync(f.ctx) == N.BCH_OK
                assert O.max_rel_err(to.to_numpy(), want) <= TOL
                assert call() == N.BCH_OK and f.lib.bch_sync(f.ctx) == N.BCH_OK  # eager: split
                assert O.max_rel_err(to.to_numpy(), want) <= TOL
                dev.upload(to.ptr, np.full(q.shape, np.nan, np.float32))
        finally:
            hip.hipGraphExecDestroy(exe)
            hip.hipGraphDestroy(graph)
