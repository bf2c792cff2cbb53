"""The fused attention's three-part bf16 products (D <= 128) vs the f64 oracle: every head
dimension class, remainders of queries and keys, grids on both workgroup shapes and with split
keys, and operands whose parts cannot stand for them."""
from __future__ import annotations

import math

import numpy as np
import pytest

from barracuda_amd import Tensor
from oracle import bc_oracle as O

pytestmark = pytest.mark.gpu
TOL = 1e-5  # f32 softmax and sums over N(0, 1) inputs: about 1e-6 of the largest output


def _run(dev, q, k, v, causal):
    t = [Tensor.from_data(x, list(x.shape), dev) for x in (q, k, v)]
    return (t[0].causal_attention(t[1], t[2]) if causal else t[0].attention(t[1], t[2])).to_numpy()


def _inputs(b, h, sq, skv, d):
    rng = np.random.default_rng(b + h * 3 + sq * 7 + skv + d)
    return (rng.standard_normal((b, h, sq, d), dtype=np.float32), rng.standard_normal((b, h, skv, d), dtype=np.float32),
            rng.standard_normal((b, h, skv, d), dtype=np.float32))


@pytest.mark.parametrize("b,h,sq,skv,d", [
    (1, 1, 33, 33, 1), (1, 2, 129, 129, 7), (2, 3, 100, 100, 31), (1, 4, 256, 256, 32), (1, 3, 300, 300, 33),
    (1, 2, 512, 512, 64), (2, 2, 257, 257, 80), (1, 2, 95, 95, 96), (1, 5, 200, 200, 97), (1, 3, 700, 700, 127),
    (1, 4, 1024, 1024, 128), (4, 64, 256, 256, 128), (4, 64, 255, 255, 128), (4, 64, 257, 257, 72), (16, 16, 31, 31, 64)])
def test_parts_causal_vs_f64(dev, b, h, sq, skv, d):
    print(f"sdpa parts causal b={b} h={h} s={sq} d={d}", flush=True)
    q, k, v = _inputs(b, h, sq, skv, d)
    got = _run(dev, q, k, v, True)
    heads = range(min(h, 4))
    assert O.max_rel_err(got[:1, heads], O.sdpa_f64(*(np.ascontiguousarray(x[:1, heads]) for x in (q, k, v)), True)) <= TOL
    assert O.max_rel_err(got[-1:, -1:], O.sdpa_f64(*(np.ascontiguousarray(x[-1:, -1:]) for x in (q, k, v)), True)) <= TOL
    assert np.array_equal(got, _run(dev, q, k, v, True)), "not deterministic"


@pytest.mark.parametrize("b,h,sq,skv,d", [
    (1, 1, 17, 1, 128), (1, 2, 40, 31, 64), (1, 2, 130, 63, 40), (1, 1, 128, 4097, 128), (2, 2, 64, 1000, 96),
    (1, 3, 300, 65, 80), (4, 64, 250, 97, 128), (4, 64, 256, 128, 64)])
def test_parts_cross_vs_f64(dev, b, h, sq, skv, d):
    print(f"sdpa parts cross b={b} h={h} sq={sq} skv={skv} d={d}", flush=True)
    q, k, v = _inputs(b, h, sq, skv, d)
    got = _run(dev, q, k, v, False)
    for sl in (np.s_[:1, :2], np.s_[-1:, -1:]):
        assert O.max_rel_err(got[sl], O.sdpa_f64(*(np.ascontiguousarray(x[sl]) for x in (q, k, v)), False)) <= TOL


@pytest.mark.parametrize("sq", [300, 2048])  # split keys; whole
def test_parts_extreme_operands(dev, sq):
    """-inf and the type's lowest value in K mask keys, NaN or +inf scores and rows of nothing but
    -inf give NaN rows, an infinite value reaches its column, subnormal values keep their bits."""
    h, d = 6 if sq == 300 else 40, 64
    q, k, v = _inputs(1, h, sq, sq, d)
    q[..., 0] = 1.0
    k[..., 0] = 0.0
    k[0, 0, 100:, 0] = -np.finfo(np.float32).max
    k[0, 1, :, 0] = -np.inf
    k[0, 2, 37, 0] = np.inf
    k[0, 3, ::2, 0] = -np.inf
    v[0, 0, 5, 3] = np.inf
    v[0, 4] *= np.float32(2.0**-130)
    v[0, 5, :, 7] *= np.float32(2.0**-110)
    got = _run(dev, q, k, v, False)[:, :6]
    q, k, v = (x[:, :6].astype(np.float64) for x in (q, k, v))
    s = (q @ k.transpose(0, 1, 3, 2)) / math.sqrt(d)
    with np.errstate(invalid="ignore"):
        p = np.exp(s - s.max(-1, keepdims=True))
        want = (p / p.sum(-1, keepdims=True)) @ v
    assert np.all(np.isinf(got[0, 0, :, 3])) and np.all(np.isnan(got[0, 1])) and np.all(np.isnan(got[0, 2]))
    for head, cols in ((0, [0, 1, 2] + list(range(4, d))), (3, list(range(d))), (4, list(range(d))), (5, list(range(d)))):
        x, y = got[0, head][:, cols], want[0, head][:, cols]
        # sums of sq terms of magnitude up to the largest value of the column, and half of the
        # smallest subnormal a term
        bound = 2e-6 * np.abs(v[0, head][:, cols]).max(0) + sq * 2.0**-150
        assert np.all(np.isfinite(x)) and np.all(np.abs(x - y) <= bound), head


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("sq,d", [(300, 64), (300, 128), (2048, 128)])  # split keys; split keys; whole
@pytest.mark.parametrize("e", [-120, -126, 90, 120])
def test_parts_scaled_operands(dev, sq, d, e, causal):
    """q scaled by 2^e against K scaled by 2^-e: ordinary scores of operands at the ends of the range."""
    print(f"scaled operands sq={sq} d={d} 2^{e} causal={causal}", flush=True)
    h = 6 if sq == 300 else 40
    q, k, v = _inputs(1, h, sq, sq, d)
    q, k = q * np.float32(2.0**e), k * np.float32(0.125) * np.float32(2.0**-e)
    want = O.sdpa_f64(*(np.ascontiguousarray(x[:, :2]) for x in (q, k, v)), causal)
    assert O.max_rel_err(_run(dev, q, k, v, causal)[:, :2], want) <= TOL


@pytest.mark.parametrize("sq", [300, 2048])
def test_parts_tiny_elements_beside_ordinary_ones(dev, sq):
    """Half of each row of q ordinary against zeros in K, the other half 2^-122 against 2^122; a key of
    probability 2^-124 with the only nonzero value."""
    print(f"tiny elements beside ordinary ones sq={sq}", flush=True)
    h, d = 6 if sq == 300 else 40, 64
    q, k, v = _inputs(1, h, sq, sq, d)
    k[..., ::2] = 0.0
    q[..., 1::2] *= np.float32(2.0**-122)
    k[..., 1::2] *= np.float32(2.0**122)
    want = O.sdpa_f64(*(np.ascontiguousarray(x[:, :2]) for x in (q, k, v)), False)
    assert O.max_rel_err(_run(dev, q, k, v, False)[:, :2], want) <= TOL
    q[...], k[...], v[...] = 0.0, 0.0, 0.0
    q[..., 0] = 8.0
    k[..., 17, 0] = -86.0  # scores / sqrt(64): probability e^-86 / (sq - 1 + e^-86)
    v[..., 17, :] = np.float32(2.0**100) * np.arange(1, d + 1, dtype=np.float32)
    want = math.exp(-86.0) / (sq - 1) * v[..., 17, :].astype(np.float64)
    got = _run(dev, q, k, v, False)
    # the exponent's f32 rounding: 124 2^-24 ln 2 and as much again for the score and the sum
    assert np.max(np.abs(got / want[:, :, None, :] - 1.0)) <= 2e-5


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("sq,d", [(300, 64), (300, 128), (299, 80), (130, 33), (2048, 32), (2047, 96), (2048, 128)])
def test_parts_computed_again_in_f32(dev, sq, d, causal):
    """Infinite and NaN operands and magnitudes past the parts' range, each in a head of its own, on split
    and whole keys: what f32 arithmetic gives, and the other heads as they are."""
    print(f"again in f32 sq={sq} d={d} causal={causal}", flush=True)
    h = 40 if sq > 1000 else 6
    q, k, v = _inputs(1, h, sq, sq, d)
    v[0, 0, 0, 3] = np.inf
    k[0, 1, sq - 1, 1] = np.nan
    q[0, 2, 7, d - 1] = np.nan
    q[0, 3] *= np.float32(2.0**50)
    k[0, 3] *= np.float32(2.0**-50)
    v[0, 4] *= np.float32(2.0**110)
    got = _run(dev, q, k, v, causal)[0, :6].astype(np.float64)
    q, k, v = (x[0, :6].astype(np.float64) for x in (q, k, v))
    s = (q @ k.transpose(0, 2, 1)) / math.sqrt(d)
    if causal:
        s = np.where(np.triu(np.ones((sq, sq), bool), 1), -np.inf, s)
    with np.errstate(invalid="ignore"):
        p = np.exp(s - s.max(-1, keepdims=True))
        want = (p / p.sum(-1, keepdims=True)) @ v
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isinf(got), np.isinf(want))
    fin = np.isfinite(want)
    got, want = np.where(fin, got, 0.0), np.where(fin, want, 0.0)
    for head in range(6):
        assert np.max(np.abs(got[head] - want[head])) <= TOL * max(np.max(np.abs(want[head])), 1e-30), head
