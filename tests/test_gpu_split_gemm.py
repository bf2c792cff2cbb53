"""The tile GEMM's three-part bf16 products (bch_sgemm, bch_sgemm_ex) where they can go wrong:
operands whose parts cannot stand for them (infinities, NaN, magnitudes at both ends of the f32
range), remainders of k at every tile and load mode, and misaligned rows."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from barracuda_amd import Tensor
from tests.test_gpu_graph import CAPTURE_RELAXED, _FreshCtx, _hip

pytestmark = pytest.mark.gpu


def _ex(dev, a, b, transb, lda=None, ldb=None, a_off=0, b_off=0, bias=None, act=0):
    """bch_sgemm_ex on copies of a and b with the given leading dimensions and start offsets."""
    m, k = a.shape
    n = b.shape[0] if transb else b.shape[1]
    lda, ldb = lda or k, ldb or b.shape[1]

    def put(x, ld, off):
        buf = np.zeros(off + x.shape[0] * ld, dtype=np.float32)
        buf[off:].reshape(x.shape[0], ld)[:, :x.shape[1]] = x
        return Tensor.from_data(buf, [buf.size], dev)

    ta, tb, tc = put(a, lda, a_off), put(b, ldb, b_off), Tensor.empty([m, n], dev)
    tbias = None if bias is None else Tensor.from_data(bias, [n], dev)
    dev.check(dev._lib.bch_sgemm_ex(dev.ctx, transb, m, n, k, C.c_void_p(ta.ptr + 4 * a_off), lda,
                                    C.c_void_p(tb.ptr + 4 * b_off), ldb, tbias and C.c_void_p(tbias.ptr), act,
                                    C.c_void_p(tc.ptr), n), "linear")
    return tc.to_numpy()


def _check_f32_sums(got, a, b):
    """The bound of a sum of k products in f32: k 2^-24 of the sum of their magnitudes, and half
    the smallest subnormal a term."""
    k = a.shape[1]
    want = a.astype(np.float64) @ b.astype(np.float64)
    bound = k * 2.0**-24 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)) + k * 2.0**-150
    worst = float(np.max(np.abs(got - want) / bound))
    assert worst <= 1.0, worst


# (m, n) and the kernel from 64 k on: few tiles (below 64 k 128 x 128 ones), 128 x 128, 256 x 128, 256 x 256
TILES = [(192, 128, b"sgemm_small_kernel"), (200, 136, b"sgemm_small_kernel"), (2040, 2044, b"sgemm_mfma_kernel<128,128,32"),
         (8190, 1020, b"sgemm_mfma_kernel<256,128,32"), (4095, 4090, b"sgemm_mfma_kernel<256,256,32")]


@pytest.mark.parametrize("transb", [0, 1])
@pytest.mark.parametrize("m,n,kernel", TILES)
@pytest.mark.parametrize("k", [1, 7, 15, 16, 17, 31, 32, 33, 47, 65, 95])
def test_k_remainders_exact(dev, m, n, kernel, k, transb):
    """Integers below 2^12: products below 2^24 and their sums are exact in f32, so three parts
    have to give every bit, whatever the remainder of k."""
    print(f"k remainder m={m} n={n} k={k} transb={transb}", flush=True)
    name = dev._lib.bch_sgemm_kernel_name(m, n, k)
    assert name.startswith(kernel if k >= 64 or kernel != b"sgemm_small_kernel" else b"sgemm_mfma_kernel<128,128,32")
    rng = np.random.default_rng(m + n + k)
    a = rng.integers(-400, 401, (m, k)).astype(np.float32)
    b = rng.integers(-400, 401, (n, k) if transb else (k, n)).astype(np.float32)
    want = a.astype(np.float64) @ (b.T if transb else b).astype(np.float64)
    assert np.abs(want).max() < 2**24
    assert np.array_equal(_ex(dev, a, b, transb), want.astype(np.float32))


@pytest.mark.parametrize("m,n,k,a_off,b_off,lda_pad,ldb_pad", [
    # the small kernel
    (260, 300, 100, 1, 3, 0, 0), (260, 300, 100, 0, 0, 1, 3), (300, 260, 67, 2, 1, 2, 2), (128, 128, 64, 1, 1, 0, 0),
    # 128 x 128, 256 x 128 and 256 x 256 tiles, and slices, that aligned operands would take unguarded or by 16 bytes
    (2048, 2048, 96, 1, 3, 0, 0), (2040, 2044, 100, 0, 0, 1, 3), (8192, 1024, 64, 2, 1, 2, 2), (8190, 1020, 65, 0, 1, 3, 0),
    (4096, 4096, 64, 1, 1, 0, 0), (4096, 4096, 64, 0, 0, 4, 1), (300, 260, 4096, 1, 3, 1, 3), (512, 512, 4096, 0, 2, 0, 0)])
@pytest.mark.parametrize("transb", [0, 1])
def test_misaligned_rows_exact(dev, m, n, k, a_off, b_off, lda_pad, ldb_pad, transb):
    print(f"misaligned m={m} n={n} k={k} transb={transb}", flush=True)
    rng = np.random.default_rng(k)
    a = rng.integers(-400, 401, (m, k)).astype(np.float32)
    b = rng.integers(-400, 401, (n, k) if transb else (k, n)).astype(np.float32)
    want = (a.astype(np.float64) @ (b.T if transb else b).astype(np.float64)).astype(np.float32)
    assert np.array_equal(_ex(dev, a, b, transb, k + lda_pad, b.shape[1] + ldb_pad, a_off, b_off), want)


@pytest.mark.parametrize("m,n,k", [(128, 128, 64), (200, 136, 100), (300, 260, 4096), (2048, 2048, 96)])
@pytest.mark.parametrize("transb", [0, 1])
def test_non_finite_operands(dev, m, n, k, transb):
    """Infinities and NaN give what IEEE arithmetic gives: an infinite a reaches its row with the
    sign of each b (NaN where b is zero or infinities meet), and no other row changes."""
    print(f"non-finite m={m} n={n} k={k} transb={transb}", flush=True)
    rng = np.random.default_rng(m + k)
    a = rng.integers(-8, 9, (m, k)).astype(np.float32)
    b = rng.integers(-8, 9, (k, n)).astype(np.float32)
    a[3, 5], a[70, 0], a[100, k - 1] = np.inf, -np.inf, np.nan
    b[7, 11], b[k - 1, 90] = -np.inf, np.nan
    with np.errstate(invalid="ignore"):
        want = np.einsum("mk,kn->mn", a.astype(np.float64), b.astype(np.float64)) if k <= 100 else None
        if want is None:
            want = a.astype(np.float64) @ b.astype(np.float64)
    got = _ex(dev, a, np.ascontiguousarray(b.T) if transb else b, transb)
    assert np.array_equal(got, want.astype(np.float32), equal_nan=True)


# m, n, k and what bch_sgemm runs there
KERNELS = [(256, 256, 256, "sgemm_mfma_kernel<64,64,64,false>"), (160, 144, 128, "sgemm_small_kernel"),
           (300, 260, 4096, "sgemm_mfma_kernel<128,128,32,true,v4>+sgemm_splitk_reduce"),
           (2048, 2048, 96, "sgemm_mfma_kernel<128,128,32,false>"),
           (2047, 2045, 95, "sgemm_mfma_kernel<128,128,32,true>"),
           (8192, 1024, 64, "sgemm_mfma_kernel<256,128,32,false>"), (4096, 4096, 64, "sgemm_mfma_kernel<256,256,32,false>"),
           (4095, 4090, 95, "sgemm_mfma_kernel<256,256,32,true>"),
           (3072, 3072, 512, "sgemm_mfma_kernel<128,128,32,false,hyb>+sgemm_tail_reduce"),
           (20, 301, 333, "sgemm_rows_kernel<1>+sgemm_splitk_reduce"),
           (50, 301, 2049, "sgemm_rows_kernel<2>+sgemm_splitk_reduce")]


@pytest.mark.parametrize("sa,sb", [(2.0**-120, 1.0), (2.0**-120, 2.0**100), (1.0, 2.0**-126), (2.0**-70, 2.0**-60),
                                   (2.0**60, 2.0**56), (2.0**-149, 2.0**120), (2.0**124, 2.0**-20)])
@pytest.mark.parametrize("m,n,k,kernel", KERNELS)
def test_ends_of_the_range(dev, m, n, k, kernel, sa, sb):
    """Rows scaled by powers of two to both ends of the f32 range, subnormals among them: the
    f32 product to 2^-24 a term (and half the smallest subnormal), as the f32 instruction gives."""
    assert dev._lib.bch_sgemm_kernel_name(m, n, k).decode() == kernel
    print(f"range m={m} n={n} k={k} sa={sa} sb={sb}", flush=True)
    rng = np.random.default_rng(5)
    a = (rng.standard_normal((m, k)) * sa).astype(np.float32)
    b = (rng.standard_normal((k, n)) * sb).astype(np.float32)
    _check_f32_sums(_ex(dev, a, b, 0), a, b)


@pytest.mark.parametrize("transb", [0, 1])
@pytest.mark.parametrize("m,n,k,kernel", KERNELS)
def test_tiny_elements_beside_ordinary_ones(dev, m, n, k, kernel, transb):
    """Elements down to the subnormals in rows (columns) that also hold ordinary ones, against zeros
    there and large elements elsewhere: every element counts to f32 accuracy, whatever else its
    row holds."""
    assert dev._lib.bch_sgemm_kernel_name(m, n, k).decode() == kernel
    rng = np.random.default_rng(m + k)
    for e, f, swap in ((-118, 100, False), (-125, 120, False), (-140, 120, False), (-125, 120, True)):
        print(f"tiny elements m={m} n={n} k={k} transb={transb} 2^{e} 2^{f} swap={swap}", flush=True)
        a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
        tiny = rng.random(k) < 0.5
        tiny[0], tiny[k - 1] = False, True
        if swap:
            b[tiny] *= np.float32(2.0**e)
            a[:, ~tiny], a[:, tiny] = 0.0, a[:, tiny] * np.float32(2.0**f)
        else:
            a[:, tiny] *= np.float32(2.0**e)
            b[~tiny], b[tiny] = 0.0, b[tiny] * np.float32(2.0**f)
        _check_f32_sums(_ex(dev, a, np.ascontiguousarray(b.T) if transb else b, transb), a, b)


@pytest.mark.parametrize("epilogue", [False, True])
@pytest.mark.parametrize("transb", [0, 1])
@pytest.mark.parametrize("m,n,k,kernel", KERNELS)
def test_values_computed_again_in_f32(dev, m, n, k, kernel, transb, epilogue):
    """What the parts cannot stand for, on every kernel and k-slice: infinities and NaN anywhere in k,
    a row and a column of nothing but NaN, operands from 2^111 and sums from 2^96.  Integers times
    powers of two, so every value is exact; its neighbours keep theirs."""
    assert dev._lib.bch_sgemm_kernel_name(m, n, k).decode() == kernel
    print(f"again in f32 m={m} n={n} k={k} transb={transb} epilogue={epilogue}", flush=True)
    rng = np.random.default_rng(m + k)
    a, b = (rng.integers(-8, 9, s).astype(np.float32) for s in ((m, k), (k, n)))
    a[3, k // 3], a[m - 2, 0], a[m // 2, k - 1], a[m // 3] = np.inf, -np.inf, np.nan, np.nan
    b[k // 2, 7], b[k - 1, n - 1], b[:, n // 2] = -np.inf, np.nan, np.nan
    a[5] *= np.float32(2.0**108)
    a[m - 1, k // 2] = np.float32(2.0**112)
    b[:, 40] *= np.float32(2.0**100)
    bias = rng.integers(-8, 9, n).astype(np.float32) if epilogue else None
    with np.errstate(invalid="ignore", over="ignore"):
        want = np.empty((m, n))
        fa, fb = np.where(np.isfinite(a), a, 0.0).astype(np.float64), np.where(np.isfinite(b), b, 0.0).astype(np.float64)
        want[:] = fa @ fb
        # rows and columns that hold infinities or NaN, term by term
        for r in np.flatnonzero(~np.isfinite(a).all(1)):
            want[r] = (a[r].astype(np.float64)[:, None] * b.astype(np.float64)).sum(0)
        for c in np.flatnonzero(~np.isfinite(b).all(0)):
            want[:, c] = (a.astype(np.float64) * b[:, c].astype(np.float64)).sum(1)
        want = want.astype(np.float32)
        if epilogue:
            want = want + bias
            want = np.where(want > 0, want, np.where(np.isnan(want), want, np.float32(0.0)))
    got = _ex(dev, a, np.ascontiguousarray(b.T) if transb else b, transb, bias=bias, act=1 if epilogue else 0)
    if epilogue:  # the activation's own treatment of NaN: what a product of few k gives
        nan = _ex(dev, np.full((1, 1), np.nan, np.float32), np.ones((1, 1), np.float32), 0, bias=np.ones(1, np.float32), act=1)
        want = np.where(np.isnan(want), nan[0, 0], want)
    got[5, 40] = want[5, 40] = 0.0  # products beyond the range of f32, of either sign
    assert np.array_equal(got, want, equal_nan=True)


def test_values_computed_again_in_f32_batched(dev):
    """Batches of each kernel that takes them: every batch's own operands."""
    for batch, m, n, k in ((3, 192, 128, 192), (5, 77, 90, 270), (40, 256, 256, 96), (3, 300, 260, 2111)):
        print(f"again in f32 batched {batch} {m} {n} {k}", flush=True)
        rng = np.random.default_rng(k)
        a, b = (rng.integers(-8, 9, s).astype(np.float32) for s in ((batch, m, k), (batch, k, n)))
        for i in range(batch):
            a[i, (7 * i) % m, (11 * i) % k] = np.inf if i % 2 else np.nan
            b[i, :, (3 * i) % n] *= np.float32(2.0**100)
        with np.errstate(invalid="ignore"):
            want = np.matmul(a.astype(np.float64), b.astype(np.float64)).astype(np.float32)
            for i in range(batch):
                r = (7 * i) % m
                want[i, r] = (a[i, r].astype(np.float64)[:, None] * b[i].astype(np.float64)).sum(0)
        got = Tensor.from_data(a, list(a.shape), dev).batch_matmul(Tensor.from_data(b, list(b.shape), dev)).to_numpy()
        assert np.array_equal(got, want, equal_nan=True)


def test_one_huge_element_in_a_row(dev):
    """Parts keep each element's own exponent: a row with one element 2^60 times the others, and a
    zero in B against it, still has the others' product to f32 accuracy."""
    m, n, k = 256, 256, 512
    rng = np.random.default_rng(9)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    a[:, 17] *= 2.0**60
    b[17, :] = 0.0
    _check_f32_sums(_ex(dev, a, b, 0), a, b)


@pytest.mark.parametrize("transb", [0, 1])
@pytest.mark.parametrize("m,n,k", [(171, 455, 1472), (67, 1536, 3056), (128, 150, 2624), (185, 192, 521), (3, 8001, 642),
                                   (1, 130, 4097), (260, 129, 255), (515, 1030, 1999), (300, 260, 2999), (700, 1200, 1501)])
def test_uneven_k_slices_exact(dev, m, n, k, transb):
    """Split-K where the slices do not divide K: the last slice is shorter and takes the remainder.  Of the
    sizes that now run the small kernel, every eighth unit a wavefront."""
    print(f"uneven slices m={m} n={n} k={k} transb={transb}", flush=True)
    small = (m, n, k) in ((171, 455, 1472), (185, 192, 521), (260, 129, 255))
    name = dev._lib.bch_sgemm_kernel_name(m, n, k)
    assert name == b"sgemm_small_kernel" if small else name.endswith(b"+sgemm_splitk_reduce")
    rng = np.random.default_rng(m + n + k)
    a = rng.integers(-40, 41, (m, k)).astype(np.float32)
    b = rng.integers(-40, 41, (n, k) if transb else (k, n)).astype(np.float32)
    want = (a.astype(np.float64) @ (b.T if transb else b).astype(np.float64)).astype(np.float32)
    assert np.array_equal(_ex(dev, a, b, transb), want)


@pytest.mark.parametrize("batch,m,n,k", [(3, 150, 70, 1001), (3, 150, 70, 2999), (3, 300, 260, 2111)])
def test_uneven_k_slices_batched(dev, batch, m, n, k):
    """The small kernel; slices of 4 k-tiles and of 8, the last with the remainder."""
    # a batch of one of these sizes splits too: k from 2048 on is not the small kernel's
    assert dev._lib.bch_sgemm_kernel_name(m, n, k).endswith(b"+sgemm_splitk_reduce" if k >= 2048 else b"sgemm_small_kernel")
    rng = np.random.default_rng(4)
    a, b = (rng.integers(-40, 41, s).astype(np.float32) for s in ((batch, m, k), (batch, k, n)))
    got = Tensor.from_data(a, list(a.shape), dev).batch_matmul(Tensor.from_data(b, list(b.shape), dev)).to_numpy()
    assert np.array_equal(got, (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32))


@pytest.mark.parametrize("m,n,k,kernel", [(171, 455, 1471, b"sgemm_small_kernel"),
                                          (300, 260, 2999, b"sgemm_mfma_kernel<128,128,32,true>+sgemm_splitk_reduce"),
                                          (20, 5247, 1001, b"sgemm_rows_kernel<1>+sgemm_splitk_reduce")])
def test_capture_without_workspace_runs_unsplit(dev, m, n, k, kernel):
    """A shape whose K no slices divide, first called under capture: no workspace may grow, the call
    runs unsplit (the small kernel as ever, few rows on tiles), and its graph replays to the product."""
    assert dev._lib.bch_sgemm_kernel_name(m, n, k) == kernel
    hip = _hip()
    rng = np.random.default_rng(6)
    a, b = rng.integers(-40, 41, (m, k)).astype(np.float32), rng.integers(-40, 41, (k, n)).astype(np.float32)
    want = (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32)
    ta, tb, tc = (Tensor.from_data(x, list(x.shape), dev) for x in (a, b, np.zeros((m, n), np.float32)))
    with _FreshCtx(dev) as f:
        graph, exe = C.c_void_p(), C.c_void_p()
        assert hip.hipStreamBeginCapture(f.stream, CAPTURE_RELAXED) == 0
        st = f.lib.bch_sgemm(f.ctx, m, n, k, C.c_void_p(ta.ptr), k, C.c_void_p(tb.ptr), n, C.c_void_p(tc.ptr), n)
        assert hip.hipStreamEndCapture(f.stream, C.byref(graph)) == 0
        assert st == 0 and f.ws_bytes() == 0
        try:
            assert hip.hipGraphInstantiate(C.byref(exe), graph, None, None, 0) == 0
            for _ in range(3):
                dev.upload(tc.ptr, np.full((m, n), np.nan, np.float32))
                assert hip.hipGraphLaunch(exe, f.stream) == 0
                assert f.lib.bch_sync(f.ctx) == 0
                assert np.array_equal(tc.to_numpy(), want)
        finally:
            hip.hipGraphExecDestroy(exe)
            hip.hipGraphDestroy(graph)


@pytest.mark.parametrize("transb", [0, 1])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (1, 127, 31), (3, 129, 33), (20, 5247, 1001), (31, 257, 65), (32, 2890, 5249),
                                   (33, 131, 4099), (64, 1021, 130), (48, 8192, 4096)])
def test_few_rows_exact(dev, m, n, k, transb):
    """Up to 64 rows that the skinny kernels do not take (and large [n][k] weights): one 32-column
    pass, remainders of k, columns and rows, split and unsplit."""
    print(f"few rows m={m} n={n} k={k} transb={transb}", flush=True)
    rng = np.random.default_rng(m + n + k)
    a = rng.integers(-40, 41, (m, k)).astype(np.float32)
    b = rng.integers(-40, 41, (n, k) if transb else (k, n)).astype(np.float32)
    want = (a.astype(np.float64) @ (b.T if transb else b).astype(np.float64)).astype(np.float32)
    assert np.array_equal(_ex(dev, a, b, transb), want)


@pytest.mark.parametrize("transb", [0, 1])
@pytest.mark.parametrize("m,k", [(20, 333), (50, 2049)])
def test_few_rows_extreme_operands(dev, m, k, transb):
    """As the tiles: infinities and NaN as in IEEE arithmetic, rows at the low end of the range."""
    n = 301
    rng = np.random.default_rng(m)
    a, b = rng.integers(-8, 9, (m, k)).astype(np.float32), rng.integers(-8, 9, (k, n)).astype(np.float32)
    a[3, 5], a[10, 0], b[7, 11], b[k - 1, 90] = np.inf, np.nan, -np.inf, np.nan
    with np.errstate(invalid="ignore"):
        want = np.einsum("mk,kn->mn", a.astype(np.float64), b.astype(np.float64)).astype(np.float32)
    bt = (lambda x: np.ascontiguousarray(x.T)) if transb else (lambda x: x)
    assert np.array_equal(_ex(dev, a, bt(b), transb), want, equal_nan=True)
    a, b = (rng.standard_normal(s).astype(np.float32) for s in ((m, k), (k, n)))
    _check_f32_sums(_ex(dev, a * np.float32(2.0**-120), bt(b * np.float32(2.0**100)), transb),
                    a * np.float32(2.0**-120), b * np.float32(2.0**100))
    _check_f32_sums(_ex(dev, a, bt(b * np.float32(2.0**-140)), transb), a, b * np.float32(2.0**-140))


# sgemm_small_kernel: 32 x 32 tiles, the 32-k units of a tile over eight wavefronts
SMALL = [(65, 65), (70, 33), (96, 100), (128, 160), (255, 257)]


@pytest.mark.parametrize("transb", [0, 1])
@pytest.mark.parametrize("m,n", SMALL)
@pytest.mark.parametrize("k", [64, 65, 96, 127, 255, 256, 257, 289, 511, 520, 777])
def test_small_kernel_every_unit_count(dev, m, n, k, transb):
    """Fewer units than wavefronts, one to four each, and a remainder on each wavefront; every element to
    the bound of f32 sums, and integers to the last bit."""
    assert dev._lib.bch_sgemm_kernel_name(m, n, k) == b"sgemm_small_kernel"
    print(f"small kernel m={m} n={n} k={k} transb={transb}", flush=True)
    rng = np.random.default_rng(m * n + k)
    for ints in (False, True):
        a = rng.integers(-120, 121, (m, k)) if ints else rng.standard_normal((m, k))
        b = rng.integers(-120, 121, (k, n)) if ints else rng.standard_normal((k, n))
        a, b = a.astype(np.float32), b.astype(np.float32)
        got = _ex(dev, a, np.ascontiguousarray(b.T) if transb else b, transb)
        if ints:  # |sums| <= 777 * 120^2 < 2^24
            assert np.array_equal(got, (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32))
        else:
            _check_f32_sums(got, a, b)


@pytest.mark.parametrize("transb", [0, 1])
def test_small_kernel_operands_without_parts(dev, transb):
    """Infinities, NaN, the largest floats and rows of tiny magnitudes, in a unit that the fourth
    wavefront holds: as the f32 instruction gives them."""
    print(f"small kernel, operands without parts, transb={transb}", flush=True)
    rng = np.random.default_rng(5)
    m, n, k = 96, 64, 300
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    a[3] *= np.float32(2.0**-120)
    b[:, 40] *= np.float32(2.0**-110)
    a[70, 100] = np.inf
    a[71, 101] = np.nan
    a[33], b[:, 9] = 0.0, 1.0
    a[33, 110] = np.float32(3.4e38)
    got = _ex(dev, a, np.ascontiguousarray(b.T) if transb else b, transb)
    with np.errstate(invalid="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[70], want[70].astype(np.float32))
    assert got[33, 9] == np.float32(3.4e38)
    rows = [r for r in range(m) if r not in (33, 70, 71)]
    _check_f32_sums(got[rows], a[rows], b)


def test_small_kernel_misaligned_strided_batched_with_epilogue(dev):
    """Odd leading dimensions and start offsets, a bias with an activation, and batches."""
    print("small kernel, misaligned, epilogue, batched", flush=True)
    rng = np.random.default_rng(6)
    m, n, k = 77, 90, 270
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((n, k)).astype(np.float32)
    _check_f32_sums(_ex(dev, a, b, 1, lda=k + 3, ldb=k + 1, a_off=1, b_off=3), a, b.T)
    bt = np.ascontiguousarray(b.T)
    _check_f32_sums(_ex(dev, a, bt, 0, lda=k + 3, ldb=n + 1, a_off=1, b_off=3), a, bt)
    bias = rng.standard_normal(n).astype(np.float32)
    ta, tb, tbias = (Tensor.from_data(x, list(x.shape), dev) for x in (a, b, bias))
    out = Tensor.empty([m, n], dev)
    dev.check(dev._lib.bch_sgemm_ex(dev.ctx, 1, m, n, k, C.c_void_p(ta.ptr), k, C.c_void_p(tb.ptr), k,
                                    C.c_void_p(tbias.ptr), 1, C.c_void_p(out.ptr), n), "linear")
    want = np.maximum(a.astype(np.float64) @ b.T.astype(np.float64) + bias, 0.0)
    # k + 1 roundings of sums of magnitudes below |a| |b| + |bias|
    bound = (k + 1) * 2.0**-24 * (np.abs(a).astype(np.float64) @ np.abs(b.T) + np.abs(bias))
    assert np.all(np.abs(out.to_numpy() - want) <= bound)
    xs, ys = rng.standard_normal((5, m, k)).astype(np.float32), rng.standard_normal((5, k, n)).astype(np.float32)
    got = Tensor.from_data(xs, [5, m, k], dev).batch_matmul(Tensor.from_data(ys, [5, k, n], dev)).to_numpy()
    for g, x, y in zip(got, xs, ys):
        _check_f32_sums(g, x, y)


@pytest.mark.parametrize("m,n,k", [(256, 256, 256), (185, 192, 521), (300, 260, 67), (320, 320, 448)])
def test_small_kernels_ask_for_no_workspace(dev, m, n, k):
    """Neither the 64 x 64 tiles nor the small kernel have partials; what they replaced had none here."""
    print(f"no workspace m={m} n={n} k={k}", flush=True)
    rng = np.random.default_rng(k)
    a, b = (rng.integers(-40, 41, s).astype(np.float32) for s in ((m, k), (k, n)))
    ta, tb, tc = (Tensor.from_data(x, list(x.shape), dev) for x in (a, b, np.zeros((m, n), np.float32)))
    with _FreshCtx(dev) as f:
        assert f.lib.bch_sgemm(f.ctx, m, n, k, C.c_void_p(ta.ptr), k, C.c_void_p(tb.ptr), n, C.c_void_p(tc.ptr), n) == 0
        assert f.lib.bch_sync(f.ctx) == 0 and f.ws_bytes() == 0
        assert f.lib.bch_sgemm_strided_batched(f.ctx, 1, m, n, k, C.c_void_p(ta.ptr), m * k, C.c_void_p(tb.ptr), k * n,
                                               C.c_void_p(tc.ptr), m * n) == 0
        assert f.lib.bch_sync(f.ctx) == 0 and f.ws_bytes() == 0
    assert np.array_equal(tc.to_numpy(), (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32))
