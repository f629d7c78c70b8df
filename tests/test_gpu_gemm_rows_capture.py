"""Calls of a few rows under stream capture: they record nothing that the context may move later, and need no scratch that a capture
forbids to allocate."""
import ctypes as C

import numpy as np
import pytest

import oracle as o
from axonml_amd import quant as q
from tests.test_zz_no_alloc import _hip
from tests.util import gen_weight

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qtype,rows", [(o.Q4_K, 16), (o.Q4_0, 10), (o.Q6_K, 39)])
def test_few_rows_in_a_graph(qtype, rows):
    """On a context of its own, whose GEMM scratch has never been allocated; replayed three times, with calls between the replays that
    make that scratch grow."""
    ctx = q.Context(0)
    hip, lib = _hip(), ctx.lib
    rng = np.random.default_rng(rows)
    n, k = 512, 1024
    packed = o.quantize(qtype, gen_weight(rng, n, k))
    dw = q.DeviceWeight.upload(q.QuantizedTensor([n, k], qtype, packed), ctx)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    x_dev, y_dev = ctx.to_device(x), ctx.malloc(rows * n * 4)
    want = x.astype(np.float64) @ o.dequantize(qtype, packed, n * k).reshape(n, k).astype(np.float64).T
    for few in (8, rows % 8 or 8):  # first use of the kernels outside any capture
        ctx.check(lib.axq_gemv_f32(ctx.handle, dw.handle, x_dev, few, None, y_dev, 1))
    ctx.synchronize()
    stream, graph, gexec = C.c_void_p(), C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreateWithFlags(C.byref(stream), 1) == 0
    ctx.check(lib.axq_set_stream(ctx.handle, stream))
    try:
        assert hip.hipStreamBeginCapture(stream, 0) == 0
        st = lib.axq_gemv_f32(ctx.handle, dw.handle, x_dev, rows, None, y_dev, 1)
        assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
        ctx.check(st)
        assert hip.hipGraphInstantiate(C.byref(gexec), graph, None, None, 0) == 0
        for more in (rows, 50, 300):
            assert hip.hipGraphLaunch(gexec, stream) == 0
            ctx.synchronize()
            got = ctx.to_host(y_dev, (rows, n), np.float32)
            assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()  # some 2^-17: sums of 1024 products in f32
            q.quantized_matmul(rng.standard_normal((more, k)).astype(np.float32), q.QuantizedTensor([n, k], qtype, packed), None, ctx)
    finally:
        ctx.check(lib.axq_set_stream(ctx.handle, None))
        if gexec:
            hip.hipGraphExecDestroy(gexec)
        if graph:
            hip.hipGraphDestroy(graph)
        hip.hipStreamDestroy(stream)
