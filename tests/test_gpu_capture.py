"""Ops with an optional workspace under HIP graph capture: replays give the
eager results, also after the workspace has grown past the captured one, and a
Gemm captured without any workspace runs the kernel that needs none.  The
workspace when the context changes streams."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from onnx_runtime_dart_amd import ops as _ops
    return _ops


class Hip:
    """The HIP runtime that the library itself has loaded."""

    def __init__(self):
        with open("/proc/self/maps") as f:
            path = next(line.split()[-1] for line in f if "libamdhip64" in line)
        self.lib = C.CDLL(path)

    def __getattr__(self, name):
        def call(*args):
            rc = getattr(self.lib, name)(*args)
            assert rc == 0, (name, rc)
        return call


SHAPES = dict(a=(100, 320), x=(2, 40, 9, 9), w=(24, 40, 3, 3), q=(1, 1, 256), k=(1, 1, 128),
              v=(1, 1, 128), pk=(1, 2, 300, 64), pv=(1, 2, 300, 64))
OUTPUTS = dict(gemm=(100, 70), conv=(2, 24, 9, 9), gqa=(1, 1, 256), ko=(1, 2, 301, 64),
               vo=(1, 2, 301, 64))


def run(ops, ctx, d, fw, gemm_only):
    # (a holds 100 rows of either K.)
    fw.gemm_dev(d["a"].ptr, 100, d["gemm"].ptr)
    if gemm_only:
        return
    ops.conv_f32_dev(d["x"].ptr, SHAPES["x"], d["w"].ptr, SHAPES["w"], d["conv"].ptr,
                     strides=[1, 1], pads=[1] * 4, ctx=ctx)
    ops.group_query_attention_dev(d["q"].ptr, d["k"].ptr, d["v"].ptr, 1, 1, 256, 4, 2,
                                  d["gqa"].ptr, d["ko"].ptr, d["vo"].ptr, past_key_ptr=d["pk"].ptr,
                                  past_value_ptr=d["pv"].ptr, past_len=300, ctx=ctx)


@pytest.mark.parametrize("k", [96, 320])  # without and with digit pairs
@pytest.mark.parametrize("warm", [True, False])
def test_graph_replays(ops, warm, k):
    rng = np.random.default_rng(1)
    ctx = ops.Context()
    hip = Hip()
    stream, graph, exe = C.c_void_p(), C.c_void_p(), C.c_void_p()
    hip.hipStreamCreate(C.byref(stream))
    ctx.set_stream(stream.value)
    fw = ops.F32Weight(rng.standard_normal((70, k)).astype(np.float32), trans_b=True, ctx=ctx)
    big = ops.F32Weight(rng.standard_normal((256, 1024)).astype(np.float32), trans_b=True, ctx=ctx)
    d = {key: ops.DeviceBuffer(4 * int(np.prod(s))) for key, s in {**SHAPES, **OUTPUTS}.items()}

    def fill(names):
        for key in names:
            s = SHAPES.get(key) or OUTPUTS[key]
            h = rng.standard_normal(s).astype(np.float32)
            hip.hipMemcpy(C.c_void_p(d[key].ptr), h.ctypes.data_as(C.c_void_p),
                          C.c_size_t(h.nbytes), 1)

    def results():
        hip.hipStreamSynchronize(stream)
        names = OUTPUTS if warm else ["gemm"]
        return {key: d[key].to_array(OUTPUTS[key], np.float32) for key in names}

    fill(SHAPES)
    if warm:
        run(ops, ctx, d, fw, False)
        hip.hipStreamSynchronize(stream)
    hip.hipStreamBeginCapture(stream, 0)
    run(ops, ctx, d, fw, not warm)
    hip.hipStreamEndCapture(stream, C.byref(graph))
    hip.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0))
    for step in (1, 2, 3):
        fill(list(SHAPES) + list(OUTPUTS))
        hip.hipGraphLaunch(exe, stream)
        got = results()
        fill(OUTPUTS)
        run(ops, ctx, d, fw, not warm)
        for key, want in results().items():
            if warm:
                np.testing.assert_array_equal(got[key], want)
            else:  # the graph holds the fp32 kernel: sums of k products, 2^-19 of ~100
                np.testing.assert_allclose(got[key], want, rtol=0, atol=1e-4)
        # A workspace larger than the graph's, other data in it.
        a, z = ops.DeviceBuffer(4096 * step * 4096), ops.DeviceBuffer(4096 * step * 1024)
        big.gemm_dev(a.ptr, 4096 * step, z.ptr)
        hip.hipStreamSynchronize(stream)
        a.free()
        z.free()
    hip.hipGraphExecDestroy(exe)
    hip.hipGraphDestroy(graph)
    for b in d.values():
        b.free()
    fw.release()
    big.release()
    ctx.close()
    hip.hipStreamDestroy(stream)


def test_any_captured_workspace_outlives_growth(ops):
    # A graph of an op that cannot do without its workspace (a decode GEMV split
    # over K); later calls need a larger one.
    rng = np.random.default_rng(3)
    hip = Hip()
    ctx = ops.Context()
    stream, graph, exe = C.c_void_p(), C.c_void_p(), C.c_void_p()
    hip.hipStreamCreate(C.byref(stream))
    ctx.set_stream(stream.value)
    k, n, bs = 8192, 2048, 32
    w = ops.NBitsWeight(rng.integers(0, 256, (n, k // bs, bs // 2), dtype=np.uint8),
                        rng.uniform(0.002, 0.02, (n, k // bs)).astype(np.float32), None, k=k, n=n,
                        block_size=bs, ctx=ctx)
    big = ops.F32Weight(rng.standard_normal((256, 1024)).astype(np.float32), trans_b=True, ctx=ctx)
    a = ops.DeviceBuffer.from_array(rng.standard_normal((1, k)).astype(np.float32), ctx)
    y = ops.DeviceBuffer(n * 4, ctx)
    w.run_dev(a.ptr, 1, y.ptr)
    want = y.to_array((n,), np.float32)
    hip.hipStreamBeginCapture(stream, 0)
    w.run_dev(a.ptr, 1, y.ptr)
    hip.hipStreamEndCapture(stream, C.byref(graph))
    hip.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0))
    zero = np.zeros(n, np.float32)
    for step in (1, 2, 3):
        rows = 4096 * step
        x, z = ops.DeviceBuffer(4096 * rows, ctx), ops.DeviceBuffer(1024 * rows, ctx)
        big.gemm_dev(x.ptr, rows, z.ptr)
        x.free()
        z.free()
        ops.check(ops.lib.mg_buffer_upload(ctx.handle, y.ptr, zero.ctypes.data, zero.nbytes))
        hip.hipGraphLaunch(exe, stream)
        np.testing.assert_array_equal(y.to_array((n,), np.float32), want)
    hip.hipGraphExecDestroy(exe)
    hip.hipGraphDestroy(graph)
    for b in (a, y):
        b.free()
    w.release()
    big.release()
    ctx.close()
    hip.hipStreamDestroy(stream)


@pytest.mark.parametrize("flags", [0, 1])  # blocking, non-blocking with the null stream
def test_stream_switch(ops, flags):
    # Calls pending on the null stream keep the workspace to themselves: the
    # switch to another stream, also one that is capturing, waits for them.
    rng = np.random.default_rng(2)
    hip = Hip()
    ctx = ops.Context()
    ctx.set_stream(0)
    m, k, n = 4096, 1536, 384
    w = ops.F32Weight(rng.standard_normal((n, k)).astype(np.float32), trans_b=True, ctx=ctx)
    a = [ops.DeviceBuffer.from_array(rng.standard_normal((m, k)).astype(np.float32), ctx)
         for _ in range(2)]
    y = [ops.DeviceBuffer(m * n * 4, ctx) for _ in range(8)]

    def result(b):
        return b.to_array((m, n), np.float32)

    w.gemm_dev(a[0].ptr, m, y[6].ptr)
    w.gemm_dev(a[1].ptr, m, y[7].ptr)
    want = [result(b) for b in y[6:]]
    stream, graph, exe = C.c_void_p(), C.c_void_p(), C.c_void_p()
    hip.hipStreamCreateWithFlags(C.byref(stream), flags)
    for b in y[:5]:
        w.gemm_dev(a[0].ptr, m, b.ptr)
    ctx.set_stream(stream.value)
    w.gemm_dev(a[1].ptr, m, y[5].ptr)
    np.testing.assert_array_equal(result(y[5]), want[1])
    ctx.set_stream(0)
    for b in y[:5]:
        np.testing.assert_array_equal(result(b), want[0])
        w.gemm_dev(a[0].ptr, m, b.ptr)
    hip.hipStreamBeginCapture(stream, 0)
    ctx.set_stream(stream.value)
    w.gemm_dev(a[1].ptr, m, y[5].ptr)
    hip.hipStreamEndCapture(stream, C.byref(graph))
    hip.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0))
    for _ in range(3):
        w.gemm_dev(a[0].ptr, m, y[5].ptr)
        hip.hipGraphLaunch(exe, stream)
        np.testing.assert_array_equal(result(y[5]), want[1])
    for b in y[:5]:
        np.testing.assert_array_equal(result(b), want[0])
    hip.hipGraphExecDestroy(exe)
    hip.hipGraphDestroy(graph)
    for b in a + y:
        b.free()
    w.release()
    ctx.close()
    hip.hipStreamDestroy(stream)
