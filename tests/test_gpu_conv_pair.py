"""fp32 Conv on fp16 digit pairs against float64, at the edges of its 16-channel
blocks, 64 x 64 tiles and padded windows, over 1-D to 3-D geometries, over wide
ranges within an image or a filter, with Inf and NaN, and without its workspace
(the fp32 MFMA kernel)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from onnx_runtime_dart_amd import ops as _ops
    return _ops


def conv64(x, w, stride, pads, dil):
    r = x.ndim - 2
    x = np.pad(x, [(0, 0), (0, 0)] + [(pads[d], pads[r + d]) for d in range(r)])
    out = [(x.shape[2 + d] - (w.shape[2 + d] - 1) * dil[d] - 1) // stride[d] + 1 for d in range(r)]
    y = 0.0
    for tap in np.ndindex(*w.shape[2:]):
        at = tuple(slice(tap[d] * dil[d], tap[d] * dil[d] + (out[d] - 1) * stride[d] + 1, stride[d])
                   for d in range(r))
        y = y + np.moveaxis(np.tensordot(x[(..., *at)], w[(..., *tap)], ((1,), (1,))), -1, 1)
    return y


def reference(x, w, b, stride, pads, dil):
    """(result, its sum of magnitudes) in float64; pads as ONNX lists them."""
    x, w = x.astype(np.float64), w.astype(np.float64)
    b = b.astype(np.float64).reshape((1, -1) + (1,) * (x.ndim - 2))
    return (conv64(x, w, stride, pads, dil) + b,
            conv64(np.abs(x), np.abs(w), stride, pads, dil) + np.abs(b))


def check(y, x, w, b, stride, pads, dil, redone=False):
    """Two digits leave 2^-23 of an operand, lo lo' 2^-22 of a product, what
    small elements lose 2^-21 of the sum, and each of the K / 16 additions (and
    the last few) 2^-23 of the sum.  Outputs computed on fp32 MFMA add K / 2
    times, each 2^-24."""
    want, size = reference(x, w, b, stride, pads, dil)
    k = np.prod(w.shape[1:])
    steps = -(-w.shape[1] // 16) * np.prod(w.shape[2:])
    assert k >= 256
    assert y.shape == want.shape
    assert (np.abs(y - want) <= (steps + 12 + k / 4 * redone) * 2.0**-23 * size).all()


CASES = [  # x, w, stride, pads, dilation
    ((2, 256, 9), (65, 256, 1), (1,), (0, 0), (1,)),
    ((3, 100, 40), (5, 100, 7), (3,), (2, 5), (2,)),
    ((2, 33, 11, 13), (70, 33, 3, 3), (1, 1), (1, 1, 1, 1), (1, 1)),
    ((1, 17, 9, 30), (63, 17, 4, 5), (2, 3), (0, 3, 2, 1), (1, 2)),
    ((5, 256, 8, 8), (64, 256, 1, 1), (2, 2), (0, 0, 0, 0), (1, 1)),
    ((1, 16, 3, 3), (1, 16, 5, 5), (1, 1), (2, 2, 2, 2), (1, 1)),
    ((2, 31, 5, 6, 7), (66, 31, 3, 2, 3), (2, 1, 1), (1, 0, 2, 1, 1, 0), (1, 2, 1)),
    ((9, 272, 7, 7), (130, 272, 3, 3), (1, 1), (1, 1, 1, 1), (1, 1)),
]


def draw(case, seed=0):
    rng = np.random.default_rng(seed)
    xs, ws = case[:2]
    return (rng.standard_normal(xs).astype(np.float32), rng.standard_normal(ws).astype(np.float32),
            rng.standard_normal(ws[0]).astype(np.float32))


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[0] + c[1])))
def test_geometries(ops, case):
    x, w, b = draw(case)
    # One image of another size: every image has its own exponent.
    x[0] *= 2.0**40
    y = ops.op_conv(x, w, b, strides=list(case[2]), pads=list(case[3]), dilations=list(case[4]))
    check(y, x, w, b, *case[2:])


def test_inf_and_nan(ops):
    # An Inf or NaN reaches the outputs whose window holds it; other images
    # and channels are those without it, and the rest of its image is redone
    # on fp32 products.
    case = CASES[7]
    x, w, b = draw(case, 1)
    args = dict(strides=list(case[2]), pads=list(case[3]), dilations=list(case[4]))
    clean = ops.op_conv(x, w, b, **args)
    z = x.copy()
    z[4, 100, 3, 2], z[7, 5, 6, 6] = np.inf, np.nan
    y = ops.op_conv(z, w, b, **args)
    others = [0, 1, 2, 3, 5, 6, 8]
    np.testing.assert_array_equal(y[others], clean[others])
    hit = np.zeros((7, 7), bool)
    hit[2:5, 1:4] = True
    np.testing.assert_array_equal(np.isinf(y[4]), np.broadcast_to(hit, y[4].shape))
    want, size = reference(x, w, b, *case[2:])
    assert (np.abs(y[4] - want[4]) <= 2448 * 2.0**-24 * size[4])[:, ~hit].all()
    np.testing.assert_array_equal(np.isnan(y[7]).any(0),
                                  np.logical_and.outer(np.arange(7) > 4, np.arange(7) > 4))
    v = w.copy()
    v[65, 0, 1, 1] = np.inf
    y = ops.op_conv(x, v, b, **args)
    rest = np.setdiff1d(np.arange(130), [65])
    np.testing.assert_array_equal(y[:, rest], clean[:, rest])
    np.testing.assert_array_equal(y[:, 65], np.sign(x[:, 0]) * np.float32(np.inf))


@pytest.mark.parametrize("x,w,stride", [
    ((8, 256, 33, 33), (40, 256, 1, 1), 3),    # 8.5 MiB, mostly skipped: on fp32 MFMA
    ((3, 1030, 33, 25), (40, 1030, 1, 1), 3),  # 9.7 MiB, longer chain: on digit pairs
    ((2, 256, 64, 65), (40, 256, 4, 4), 4)])
def test_large_strided_inputs(ops, x, w, stride):
    x, w, b = draw((x, w))
    y = ops.op_conv(x, w, b, strides=[stride] * 2)
    check(y, x, w, b, (stride,) * 2, (0,) * 4, (1, 1), redone=True)


@pytest.mark.parametrize("big", [1e6, 1e12, 1e20, -3.4028235e38])
@pytest.mark.parametrize("case", CASES[1:4] + CASES[7:], ids=lambda c: "x".join(map(str, c[0] + c[1])))
def test_large_value_in_a_corner(ops, case, big):
    # One value of an image (and one of a filter) far above the others: the
    # windows (channels) that do not hold it are as good as without it.
    x, w, b = (t / 10 for t in draw(case, 3))
    whole = x.copy()
    x[0, 0].flat[0] = big
    x[-1, -1].flat[-1] = big
    v = w.copy()
    v[len(v) // 2, 0].flat[0] = big
    args = dict(strides=list(case[2]), pads=list(case[3]), dilations=list(case[4]))
    check(ops.op_conv(x, w, b, **args), x, w, b, *case[2:], redone=True)
    check(ops.op_conv(whole, v, b, **args), whole, v, b, *case[2:], redone=True)


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[0] + c[1])))
def test_opposite_ranges(ops, case):
    # Channels over 2^80 in the input and the other way round in the filters; an
    # image and a filter of zeros.
    x, w, b = draw(case, 4)
    s = np.random.default_rng(5).integers(-40, 41, x.shape[1]).reshape((1, -1) + (1,) * (x.ndim - 2))
    x, w = (x * 2.0**s).astype(np.float32), (w * 2.0**-s).astype(np.float32)
    x[-1] *= len(x) == 1
    w[-1] *= len(w) == 1
    y = ops.op_conv(x, w, b, strides=list(case[2]), pads=list(case[3]), dilations=list(case[4]))
    check(y, x, w, b, *case[2:], redone=True)


def test_two_gib_of_output(ops):
    # Images that would fill a round's output to exactly 2^31 bytes.
    n, c, size, m = 64, 32, 64, 2048
    rng = np.random.default_rng(6)
    x = rng.standard_normal((n, c, size, size)).astype(np.float32)
    w = rng.standard_normal((m, c, 3, 3)).astype(np.float32)
    xd, wd = ops.DeviceBuffer.from_array(x), ops.DeviceBuffer.from_array(w)
    y = ops.DeviceBuffer(n * m * size * size * 4)
    assert y.nbytes == 1 << 31

    class Tail(ops.DeviceBuffer):
        def __init__(self, image, channel):
            self.ctx, self.ptr = y.ctx, y.ptr + (image * m + channel) * size * size * 4

        def free(self):
            pass

    nan = np.full((size, size), np.nan, np.float32)
    at = [(0, 0), (31, 1000), (62, m - 1), (63, 0), (63, m - 1)]
    for i, o in at:
        ops.check(ops.lib.mg_buffer_upload(y.ctx.handle, Tail(i, o).ptr, nan.ctypes.data, nan.nbytes))
    ops.conv_f32_dev(xd.ptr, x.shape, wd.ptr, w.shape, y.ptr, strides=[1, 1], pads=[1] * 4)
    for i, o in at:
        got = Tail(i, o).to_array((1, 1, size, size), np.float32)
        check(got, x[i:i + 1], w[o:o + 1], np.zeros(1, np.float32), (1, 1), (1, 1, 1, 1), (1, 1))
    for d in (xd, wd, y):
        d.free()


def test_without_workspace(ops):
    case = CASES[2]
    x, w, b = draw(case, 2)
    ctx = ops.default_context()
    bufs = [ops.DeviceBuffer.from_array(t) for t in (x, w, b)]
    y = ops.DeviceBuffer(2 * 70 * 11 * 13 * 4)
    ctx.set_control(None, max_bytes=4096)
    try:
        ops.conv_f32_dev(bufs[0].ptr, x.shape, bufs[1].ptr, w.shape, y.ptr, bufs[2].ptr,
                         strides=[1, 1], pads=[1] * 4, ctx=ctx)
    finally:
        ctx.set_control(None, max_bytes=-1)
    want, size = reference(x, w, b, *case[2:])
    assert (np.abs(y.to_array(want.shape, np.float32) - want) <= 297 * 2.0**-23 * size).all()
    for d in bufs + [y]:
        d.free()
