"""The one-pass decode step of GroupQueryAttention (device entry point) against
float64 over its key ranges, head sizes, group sizes and rotary forms; present
K / V bit for bit those of the host entry point."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from onnx_runtime_dart_amd import ops as _ops
    return _ops


def step(ops, q, k, v, pk, pv, cos, sin, heads, kv, half_rot, rotary, inter):
    b, _, hidden = q.shape
    d, past = hidden // heads, pk.shape[2]
    up = [ops.DeviceBuffer.from_array(t) if t.size else None for t in (q, k, v, pk, pv, cos, sin)]
    ptr = [u.ptr if u else 0 for u in up]
    shape = (b, kv, past + 1, d)
    y, ko, vo = ops.DeviceBuffer(q.nbytes), *(ops.DeviceBuffer(4 * int(np.prod(shape)))
                                              for _ in range(2))
    ops.group_query_attention_dev(ptr[0], ptr[1], ptr[2], b, 1, hidden, heads, kv, y.ptr, ko.ptr,
                                  vo.ptr, past_key_ptr=ptr[3], past_value_ptr=ptr[4],
                                  past_len=past, cos_ptr=ptr[5], sin_ptr=ptr[6],
                                  max_pos=past + 1, half_rot=half_rot, do_rotary=rotary,
                                  rotary_interleaved=inter)
    out = (y.to_array(q.shape, np.float32), ko.to_array(shape, np.float32),
           vo.to_array(shape, np.float32))
    for u in up + [y, ko, vo]:
        if u:
            u.free()
    return out


def rotate(x, cos, sin, inter):
    x, c, s = x.astype(np.float64), cos[-1].astype(np.float64), sin[-1].astype(np.float64)
    r = 2 * len(c)
    y = x.copy()
    a, b = (x[..., :r:2], x[..., 1:r:2]) if inter else (x[..., :r // 2], x[..., r // 2:r])
    lo, hi = a * c - b * s, b * c + a * s
    if inter:
        y[..., :r:2], y[..., 1:r:2] = lo, hi
    else:
        y[..., :r // 2], y[..., r // 2:r] = lo, hi
    return y


# heads, kv heads, head size, past, batch, rotated half, interleaved
CASES = [(1, 1, 64, 0, 1, 32, False), (4, 2, 64, 1, 3, 32, True), (6, 2, 64, 126, 1, 16, False),
         (8, 2, 64, 127, 2, 32, False), (14, 2, 64, 128, 1, 32, False), (16, 2, 64, 500, 1, 0, False),
         (18, 2, 64, 70, 1, 32, False), (8, 8, 128, 62, 2, 64, False), (4, 2, 128, 63, 1, 64, True),
         (28, 4, 128, 64, 1, 32, False), (32, 8, 64, 4096, 1, 32, False),
         (2, 1, 128, 30000, 1, 64, False), (64, 64, 64, 700, 16, 32, False),
         (3, 1, 32, 90, 1, 16, False)]


@pytest.mark.parametrize("case", CASES, ids=str)
def test_decode_step(ops, case):
    heads, kv, d, past, batch, half, inter = case
    rng = np.random.default_rng(heads + d + past)
    q, k, v = (rng.standard_normal((batch, 1, n * d)).astype(np.float32) for n in (heads, kv, kv))
    pk, pv = (rng.standard_normal((batch, kv, past, d)).astype(np.float32) for _ in range(2))
    angle = rng.uniform(0, 6, (past + 1, half))
    cos, sin = np.cos(angle).astype(np.float32), np.sin(angle).astype(np.float32)
    rotary = half > 0
    y, ko, vo = step(ops, q, k, v, pk, pv, cos, sin, heads, kv, half, rotary, inter)
    kr = rotate(k.reshape(batch, kv, 1, d), cos, sin, inter) if rotary else k.reshape(batch, kv, 1, d)
    np.testing.assert_array_equal(ko, np.concatenate([pk, kr.astype(np.float32)], 2))
    np.testing.assert_array_equal(vo, np.concatenate([pv, v.reshape(batch, kv, 1, d)], 2))
    qr = q.reshape(batch, kv, heads // kv, d)
    qr = (rotate(qr, cos, sin, inter) if rotary else qr).astype(np.float32).astype(np.float64)
    kf, vf = ko.astype(np.float64), vo.astype(np.float64)
    s = qr @ kf.transpose(0, 1, 3, 2) / np.sqrt(d)
    w = np.exp(s - s.max(-1, keepdims=True))
    want = (w / w.sum(-1, keepdims=True)) @ vf
    # A score is off by at most (d + 4) 2^-24 of its sum of magnitudes, a
    # weight by that share of itself (exp2 another 2^-22), the sums over keys
    # by 2^-24 a step of at most past + 1 in a chain.
    size = (np.abs(qr) @ np.abs(kf).transpose(0, 1, 3, 2)).max() / np.sqrt(d)
    eps = 2 * ((d + 4) * 2.0**-24 * size + 2.0**-22) + (past / 128 + 64) * 2.0**-24
    assert np.abs(y.reshape(want.shape) - want).max() <= eps * np.abs(vf).max()


def test_non_finite_keys(ops):
    # NaN in one head's cache stays with the heads that read it; a key of
    # -inf score has no weight.
    rng = np.random.default_rng(9)
    q, k, v = (rng.standard_normal((1, 1, n * 64)).astype(np.float32) for n in (8, 4, 4))
    pk, pv = (rng.standard_normal((1, 4, 300, 64)).astype(np.float32) for _ in range(2))
    args = (np.zeros((301, 0), np.float32), np.zeros((301, 0), np.float32), 8, 4, 0, False, False)
    clean = step(ops, q, k, v, pk, pv, *args)[0].reshape(4, 2, 64)
    pk[0, 1, 200, 3] = np.nan
    q[0, 0, 4 * 64], q[0, 0, 5 * 64] = 1.0, 1.0
    pk[0, 2, 7, 0] = -np.inf
    y = step(ops, q, k, v, pk, pv, *args)[0].reshape(4, 2, 64)
    np.testing.assert_array_equal(y[[0, 3]], clean[[0, 3]])
    assert np.isnan(y[1]).all() and np.isfinite(y[2]).all()
