"""mk_topk in a captured graph, which keeps selecting right when the context's scratch has moved since the capture."""
import ctypes

import numpy as np
import pytest

import malkin_amd as mk_
from test_gpu_sampling import expected_topk

pytestmark = pytest.mark.gpu

RELAXED = 2  # hipStreamCaptureModeRelaxed


def test_graph_outlives_scratch():
    hip = ctypes.CDLL("libamdhip64.so")

    def hck(rc):
        assert rc == 0, rc

    ctx, L = mk_.Context(0), mk_.load()
    stream = ctypes.c_void_p(L.mk_stream(ctx.h))
    n, V, k = 3, 30000, 500
    dx, dv, di = ctx.alloc(n * V * 4), ctx.alloc(n * k * 4), ctx.alloc(n * k * 4)
    graph, run = ctypes.c_void_p(), ctypes.c_void_p()
    hck(hip.hipStreamBeginCapture(stream, RELAXED))
    mk_.check(L.mk_topk(ctx.h, dx.ptr, V, None, n, V, k, dv.ptr, di.ptr))
    hck(hip.hipStreamEndCapture(stream, ctypes.byref(graph)))
    hck(hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)))
    mk_.check(L.mk_reserve_scratch(ctx.h, 64 << 20))  # the old scratch is gone
    others = [ctx.to_device(np.full(1 << 18, 255, np.uint8)) for _ in range(16)]
    for i in range(4):
        x = np.random.default_rng(i).standard_normal((n, V)).astype(np.float32)
        dx.upload(x)
        print("replay", i, flush=True)
        hck(hip.hipGraphLaunch(run, stream))
        ctx.sync()
        got = di.download(np.int32).reshape(n, k)
        for r in range(n):
            assert np.array_equal(got[r], expected_topk(x[r], k)[1]), (i, r)
    assert all((b.download(np.uint8) == 255).all() for b in others)
    hck(hip.hipGraphExecDestroy(run))
    hck(hip.hipGraphDestroy(graph))
    for b in others + [dx, dv, di]:
        b.free()
    ctx.close()
