"""Weight Gemms on fp16 digit pairs (F32Weight.gemm) against float64, at the
edges of their 64 x 64 tiles and 64-k padding, over every plan of the digit
split, over wide exponent ranges within a row (outputs that lost parts of small
elements could show in) and with Inf and NaN operands, both on the fp32 form of
the tile, and without the workspace they would like to have (the fp32 MFMA
kernel)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from onnx_runtime_dart_amd import ops as _ops
    return _ops


def check(y, a, w, c=0.0, alpha=1.0, beta=1.0):
    """Element by element: the digits leave 2^-23 of an operand, lo lo' 2^-22
    of a product, what small elements lose 2^-21 of the sum, and each of the
    K / 16 additions per output (and the few that join the shares, scale and add
    C) at most 2^-23 of what has been added, all of it at most sum |a| |w|."""
    a, w = a.astype(np.float64), w.astype(np.float64)
    want = alpha * (a @ w.T) + beta * c
    size = abs(alpha) * (np.abs(a) @ np.abs(w).T) + np.abs(beta * c)
    bound = (a.shape[1] / 16 + 12) * 2.0**-23 * size + 2.0**-148
    assert (np.abs(y - want) <= bound).all()


@pytest.mark.parametrize("m,k,n", [(1, 1, 1), (63, 15, 65), (65, 64, 63), (64, 65, 64),
                                   (1, 2049, 130), (130, 8200, 70), (2049, 513, 65),
                                   (1030, 1025, 33), (700, 1537, 129), (4096, 384, 200),
                                   # The sizes that take pairs, to either side of each line.
                                   (1, 256, 1), (63, 257, 65), (65, 319, 63), (64, 320, 64),
                                   (128, 192, 64), (129, 192, 64), (64, 191, 64), (700, 200, 6000),
                                   (690, 200, 6000), (1024, 256, 3), (1025, 257, 66),
                                   (1030, 260, 767), (1030, 260, 768), (2049, 260, 383),
                                   (2049, 260, 384), (1025, 384, 65), (2049, 384, 128),
                                   (2049, 513, 127), (8193, 384, 191), (8193, 385, 192),
                                   (2050, 4100, 255), (2050, 4096, 255), (2050, 4096, 256),
                                   (2050, 4100, 511), (2050, 4100, 512), (30, 9000, 65)])
def test_tile_edges(ops, m, k, n):
    rng = np.random.default_rng(m + k + n)
    a = rng.standard_normal((m, k)).astype(np.float32)
    w = rng.standard_normal((n, k)).astype(np.float32)
    fw = ops.F32Weight(w, trans_b=True)
    check(fw.gemm(a), a, w)
    bias = rng.standard_normal(n).astype(np.float32)
    check(fw.gemm(a, bias, alpha=0.5, beta=2.0), a, w, bias, 0.5, 2.0)
    full = rng.standard_normal((m, n)).astype(np.float32)
    check(fw.gemm(a, full), a, w, full)
    col = rng.standard_normal((m, 1)).astype(np.float32)
    check(fw.gemm(a, col), a, w, col)
    fw.release()


def test_exponent_ranges(ops):
    # Rows and columns from 2^-140 to 2^60, elements of a row over 2^40, zeros.
    rng = np.random.default_rng(3)
    a = rng.standard_normal((70, 200)) * 2.0 ** rng.integers(-20, 21, (70, 200))
    a *= 2.0 ** np.linspace(-120, 60, 70)[:, None]
    a[5] = 0
    w = rng.standard_normal((66, 200)) * 2.0 ** np.linspace(-60, 40, 66)[:, None]
    w[7] = 0
    a, w = a.astype(np.float32), w.astype(np.float32)
    fw = ops.F32Weight(w, trans_b=True)
    check(fw.gemm(a), a, w)
    fw.release()


def test_inf_and_nan(ops):
    # An Inf or NaN touches its own row's (column's) outputs, as the sum in
    # fp32 gives them; the other outputs are those without it.
    rng = np.random.default_rng(4)
    a = rng.standard_normal((100, 150)).astype(np.float32)
    w = rng.standard_normal((90, 150)).astype(np.float32)
    fw = ops.F32Weight(w, trans_b=True)
    clean = fw.gemm(a)
    b = a.copy()
    b[3, 7], b[40, 100], b[77, 149], b[77, 0] = np.inf, np.nan, -np.inf, np.inf
    y = fw.gemm(b)
    fw.release()
    rows = np.setdiff1d(np.arange(100), [3, 40, 77])
    np.testing.assert_array_equal(y[rows], clean[rows])
    np.testing.assert_array_equal(y[3], np.sign(w[:, 7]) * np.float32(np.inf))
    assert np.isnan(y[40]).all()
    same = np.sign(w[:, 149]) == -np.sign(w[:, 0])
    np.testing.assert_array_equal(np.isnan(y[77]), ~same)
    v = w.copy()
    v[11, 2], v[64, 64] = np.inf, np.nan
    fw = ops.F32Weight(v, trans_b=True)
    z = fw.gemm(a)
    fw.release()
    cols = np.setdiff1d(np.arange(90), [11, 64])
    np.testing.assert_array_equal(z[:, cols], clean[:, cols])
    np.testing.assert_array_equal(z[:, 11], np.sign(a[:, 2]) * np.float32(np.inf))
    assert np.isnan(z[:, 64]).all()


def test_without_workspace(ops):
    # A byte budget below the images of A: the call still runs (fp32 MFMA).
    rng = np.random.default_rng(5)
    a = rng.standard_normal((70, 96)).astype(np.float32)
    w = rng.standard_normal((40, 96)).astype(np.float32)
    ctx = ops.default_context()
    fw = ops.F32Weight(w, trans_b=True, ctx=ctx)
    ad, yd = ops.DeviceBuffer.from_array(a), ops.DeviceBuffer(70 * 40 * 4)
    ctx.set_control(None, max_bytes=64)
    try:
        fw.gemm_dev(ad.ptr, 70, yd.ptr)
    finally:
        ctx.set_control(None, max_bytes=-1)
    check(yd.to_array((70, 40), np.float32), a, w)
    for b in (ad, yd):
        b.free()
    fw.release()


def test_long_k(ops):
    # Above the K of pair images (32-bit fragment offsets, one chunk of A):
    # whole numbers whose sums are exact.
    rng = np.random.default_rng(6)
    for m, k, n in ((33, (1 << 23) + 40, 1), (65, (1 << 18) - 64, 40), (65, (1 << 18) - 63, 40)):
        a = rng.integers(-1, 2, (m, k), dtype=np.int8).astype(np.float32)
        w = rng.integers(-1, 2, (n, k), dtype=np.int8).astype(np.float32)
        fw = ops.F32Weight(w, trans_b=True)
        y = fw.gemm(a)
        fw.release()
        np.testing.assert_array_equal(y, a @ w.T)


def test_image_bytes(ops):
    # Images are bounded by the weight's size, whatever their padding.
    for n, k in ((1, 1 << 20), (1, 4), (7, 5000), (32, 8192), (100, 300), (40, 1 << 18)):
        fw = ops.F32Weight(np.zeros((n, k), np.float32), trans_b=True)
        assert 4 * n * k <= fw.info()[2] <= 12 * n * k + (1 << 20)
        fw.release()


# Two elements of a row, two of a column: the large one meets a zero or a small
# factor, so that the small one is the result.
LOST = [((1e20, 1), (0, 1)), ((3.4028235e38, 1.5), (0, 1)), ((1e8, 1e-8), (1e-8, 1e8)),
        ((1e12, 1.2345678), (0, 1)), ((1e6, 1.2345678e-6), (0, 1)), ((1e-30, 1e-45), (0, 1e30)),
        ((0, 1), (1e20, 1))]


@pytest.mark.parametrize("k", [256, 259, 513])
def test_large_beside_small(ops, k):
    rng = np.random.default_rng(k)
    n = len(LOST)
    a, w = np.zeros((66, k), np.float32), np.zeros((n, k), np.float32)
    for i, (x, y) in enumerate(LOST):
        at = rng.choice(k, 2, replace=False)
        a[i, at], a[-1 - i, at] = x, x
        w[i, at] = y
    fw = ops.F32Weight(w, trans_b=True)
    y = fw.gemm(a)
    fw.release()
    check(y, a, w)
    for i, (x, z) in enumerate(LOST):
        want = np.dot(np.float32(x).astype(np.float64), np.float32(z).astype(np.float64))
        assert y[i, i] == y[-1 - i, i] == np.float32(want), (i, y[i, i], want)


@pytest.mark.parametrize("k,off", [(256, 0), (320, 1), (301, 0)])
def test_ranges_within_a_row(ops, k, off):
    # Elements of a row over 2^80 against single elements (a permutation) and
    # against columns of the opposite range, whose products are all alike; a
    # zero row and a row whose one large element meets a zero.
    rng = np.random.default_rng(8)
    m = 70
    s = rng.integers(-40, 41, k)
    a = (rng.standard_normal((m, k)) * 2.0**s).astype(np.float32)
    a[3], a[40, 5] = 0, 3e38
    one = np.eye(k, dtype=np.float32)[rng.permutation(k)]
    w = (rng.standard_normal((130, k)) * 2.0**-s).astype(np.float32)
    w[:, 5] = 0
    ad = ops.DeviceBuffer.from_array(np.concatenate([np.zeros(off, np.float32), a.ravel()]))
    for b in (one, w):
        fw = ops.F32Weight(b, trans_b=True)
        yd = ops.DeviceBuffer(m * len(b) * 4)
        fw.gemm_dev(ad.ptr + 4 * off, m, yd.ptr)
        y = yd.to_array((m, len(b)), np.float32)
        check(y, a, b)
        assert (y[3] == 0).all()
        if b is one:
            want = a.astype(np.float64) @ one.T
            assert (np.abs(y - want) <= 2.0**-22 * np.abs(want)).all()
        fw.release()
        yd.free()
    ad.free()


@pytest.mark.parametrize("c_shape", [(1,), (130,), (70, 1), (70, 130)])
def test_redone_outputs_with_c(ops, c_shape):
    # alpha and beta C on outputs of both forms in one tile, C also in place.
    rng = np.random.default_rng(11)
    m, k, n = 70, 320, 130
    s = rng.integers(-40, 41, k)
    a = (rng.standard_normal((m, k)) * 2.0**s).astype(np.float32)
    w = (rng.standard_normal((n, k)) * 2.0**-s).astype(np.float32)
    a[::3], w[::2] = rng.standard_normal((24, k)), rng.standard_normal((65, k))
    a[::6, 9], w[:, 9] = 1e30, 0
    c = rng.standard_normal(c_shape).astype(np.float32)
    fw = ops.F32Weight(w, trans_b=True)
    check(fw.gemm(a, c, alpha=0.5, beta=2.0), a, w, c, 0.5, 2.0)
    if c.shape == (m, n):
        ad, yd = ops.DeviceBuffer.from_array(a), ops.DeviceBuffer.from_array(c)
        fw.gemm_dev(ad.ptr, m, yd.ptr, yd.ptr, c.shape, alpha=0.5, beta=2.0)
        check(yd.to_array((m, n), np.float32), a, w, c, 0.5, 2.0)
        ad.free()
        yd.free()
    fw.release()


def test_inf_and_nan_beside_small(ops):
    # As test_inf_and_nan, at a K of the pairs, with rows of zeros and of small
    # elements among them: 0 Inf is NaN, as the sum in fp32 gives it.
    rng = np.random.default_rng(9)
    a = rng.standard_normal((100, 300)).astype(np.float32)
    w = rng.standard_normal((90, 300)).astype(np.float32)
    a[50] = 0
    a[51, 7] = 1e30
    w[20] = 0
    v = w.copy()
    v[11, 2], v[64, 64] = np.inf, np.nan
    b = a.copy()
    b[3, 7], b[40, 100] = -np.inf, np.nan
    fw, fv = ops.F32Weight(w, trans_b=True), ops.F32Weight(v, trans_b=True)
    clean, y, z = fw.gemm(a), fw.gemm(b), fv.gemm(a)
    fw.release()
    fv.release()
    check(clean, a, w)
    rows, cols = np.setdiff1d(np.arange(100), [3, 40]), np.setdiff1d(np.arange(90), [11, 64])
    np.testing.assert_array_equal(y[rows], clean[rows])
    with np.errstate(invalid="ignore"):
        np.testing.assert_array_equal(y[3], w[:, 7] * np.float32(-np.inf))
        assert np.isnan(y[40]).all()
        np.testing.assert_array_equal(z[:, cols], clean[:, cols])
        np.testing.assert_array_equal(z[:, 11], a[:, 2] * np.float32(np.inf))
    assert np.isnan(z[:, 64]).all()


def test_without_images(ops):
    # A context with images disabled: no pairs, products of the operands as they
    # are, so that a permutation and a filter of one tap copy bit for bit.
    rng = np.random.default_rng(10)
    k = 320
    a = rng.standard_normal((70, k)).astype(np.float32)
    order = rng.permutation(k)
    w = np.eye(k, dtype=np.float32)[order]
    x = rng.standard_normal((2, 32, 9, 9)).astype(np.float32)
    v = np.zeros((32, 32, 3, 3), np.float32)
    v[np.arange(32), order[order < 32], 1, 1] = 1
    ctx = ops.default_context()
    ctx.set_prefill_images(False)
    try:
        fw = ops.F32Weight(w, trans_b=True, ctx=ctx)
        y = ops.op_conv(x, v, None, pads=[1] * 4)
    finally:
        ctx.set_prefill_images(True)
    assert fw.info()[2] == 4 * k * k
    np.testing.assert_array_equal(fw.gemm(a), a[:, order])
    np.testing.assert_array_equal(y, x[:, order[order < 32]])
    fw.release()
    fw = ops.F32Weight(w, trans_b=True, ctx=ctx)
    assert fw.info()[2] > 8 * k * k
    fw.release()
