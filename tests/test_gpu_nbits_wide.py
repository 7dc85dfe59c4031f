"""Prefill plans of the fp16 GEMM (blocks below 128): further K splits on grids
of few tiles, 64-column tiles where wide ones would leave CUs without work, the
forms of the activations' split, and the plan without further splits under a byte
budget and under capture; against the oracle on a subset of columns."""
import numpy as np
import pytest

import golden_io as G
import oracle

pytestmark = pytest.mark.gpu
TOL = 1e-3


@pytest.fixture(scope="module")
def ops():
    from onnx_runtime_dart_amd import ops as _ops
    return _ops


def weight(ops, rng, k, n, bs, ctx=None):
    nb = -(-k // bs)
    b = rng.integers(0, 256, (n, nb, bs // 2), dtype=np.uint8)
    s = rng.uniform(0.002, 0.02, (n, nb)).astype(np.float32)
    zp = rng.integers(0, 256, (n, (nb + 1) // 2), dtype=np.uint8)
    return (b, s, zp), ops.NBitsWeight(b, s, zp, k=k, n=n, block_size=bs, ctx=ctx)


def check(y, a, w, k, bs):
    n = len(w[0])
    cols = np.unique(np.concatenate([np.arange(0, n, max(1, n // 48)), np.arange(n - 3, n)]))
    ref = oracle.matmul_nbits(a, w[0][cols], w[1][cols], w[2][cols], k=k, n=len(cols),
                              block_size=bs)
    assert G.rms_error(y[:, cols], ref) <= TOL


@pytest.mark.parametrize("m,k,n,bs", [
    (301, 8192, 2048, 32),   # 96 tiles: 8 splits
    (17, 32 * 67, 130, 32),  # 3 tiles, 17 k groups: splits of uneven length
    (129, 640, 6144, 64),    # 192 tiles (three quarters of 256 CUs), 5 k groups: one split
    (129, 1024, 6145, 64),   # 194 tiles: above the line
    (301, 256, 16384, 32),   # 384 wide tiles: 768 narrow ones instead
    (256, 4128, 96, 32),     # few columns, 33 k groups
    (301, 1504, 3072, 32),   # 144 tiles, 12 k groups: 3 splits
    (301, 1408, 3072, 32),   # 11: one
    (140, 2016, 5500, 32),   # 172 tiles, 16 k groups: 4 splits
    (300, 2080, 2100, 64),   # 99 tiles, 17 k groups: 4 splits, the last one short
    (300, 4100, 2000, 32),   # 96 tiles, 33 k groups: 8 splits of 5 and fewer
    (70, 4128, 2600, 32),    # 41 tiles: 8 splits for 4
    (641, 4096, 1000, 32),   # 96 tiles in 6 rows of them: as without further splits
    (1025, 200, 65, 32),     # activations split with a wave a row
    (1023, 500, 65, 32), (1024, 512, 64, 32), (1024, 545, 64, 32)])
def test_plans(ops, m, k, n, bs):
    rng = np.random.default_rng(m + k + n)
    w, h = weight(ops, rng, k, n, bs)
    a = rng.standard_normal((m, k)).astype(np.float32)
    check(h(a), a, w, k, bs)
    h.release()


def test_plan_under_a_byte_budget(ops):
    # 12 MiB hold the activations' split and two partials (5 MB), not eight.
    rng = np.random.default_rng(7)
    m, k, n, bs = 301, 4096, 2048, 32
    w, h = weight(ops, rng, k, n, bs)
    a = rng.standard_normal((m, k)).astype(np.float32)
    ad, yd = ops.DeviceBuffer.from_array(a), ops.DeviceBuffer(m * n * 4)
    ctx = ops.default_context()
    for budget in (-1, 12 << 20):
        ctx.set_control(None, max_bytes=budget)
        try:
            h.run_dev(ad.ptr, m, yd.ptr)
        finally:
            ctx.set_control(None, max_bytes=-1)
        check(yd.to_array((m, n), np.float32), a, w, k, bs)
    for d in (ad, yd):
        d.free()
    h.release()


def test_host_call_under_a_byte_budget(ops):
    # The activations and results staged by the host entry point count against
    # the budget too: 7.4 MB beside 26 MB of the wide plan or 11 of the other.
    rng = np.random.default_rng(8)
    m, k, n, bs = 301, 4096, 2048, 32
    w, h = weight(ops, rng, k, n, bs)
    a = rng.standard_normal((m, k)).astype(np.float32)
    ctx = ops.default_context()
    ctx.set_control(None, max_bytes=27 << 20)
    try:
        y = h(a)
    finally:
        ctx.set_control(None, max_bytes=-1)
    check(y, a, w, k, bs)
    h.release()


def test_plan_under_capture(ops):
    # A capturing stream cannot grow the workspace: the plan keeps to the one
    # that an earlier call left (here under a byte budget), and replays give what
    # that call gave, also after the wide plan has run beside them.
    import ctypes as C
    from test_gpu_capture import Hip
    hip, ctx = Hip(), ops.Context()
    stream, graph, exe = C.c_void_p(), C.c_void_p(), C.c_void_p()
    hip.hipStreamCreate(C.byref(stream))
    ctx.set_stream(stream.value)
    rng = np.random.default_rng(9)
    m, k, n, bs = 301, 4096, 2048, 32
    w, h = weight(ops, rng, k, n, bs, ctx)
    a = rng.standard_normal((m, k)).astype(np.float32)
    ad, yd = ops.DeviceBuffer.from_array(a, ctx), ops.DeviceBuffer(m * n * 4, ctx)
    ctx.set_control(None, max_bytes=12 << 20)
    h.run_dev(ad.ptr, m, yd.ptr)
    ctx.set_control(None, max_bytes=-1)
    eager = yd.to_array((m, n), np.float32)
    check(eager, a, w, k, bs)
    hip.hipStreamBeginCapture(stream, 0)
    h.run_dev(ad.ptr, m, yd.ptr)
    hip.hipStreamEndCapture(stream, C.byref(graph))
    hip.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0))
    for _ in range(3):
        h.run_dev(ad.ptr, m, yd.ptr)
        check(yd.to_array((m, n), np.float32), a, w, k, bs)
        hip.hipGraphLaunch(exe, stream)
        np.testing.assert_array_equal(yd.to_array((m, n), np.float32), eager)
    hip.hipGraphExecDestroy(exe)
    hip.hipGraphDestroy(graph)
    for d in (ad, yd):
        d.free()
    h.release()
    ctx.close()
    hip.hipStreamDestroy(stream)
