"""mk_topk in a captured graph, which keeps selecting right when the context's scratch has moved since the capture, and over
many rows, which are walked by one workgroup each instead of cut into slices."""
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


@pytest.mark.parametrize("V,k,n_rows", [(8193, 1, 70000), (8193, 1024, 32), (8193, 1024, 33), (9000, 40, 300),
                                        (65792, 1024, 256), (65792, 1024, 257), (1 << 18, 300, 257)])
def test_many_rows(mk, V, k, n_rows):
    """n_rows rows that are five logits rows over and over, around the count from which one workgroup walks a row."""
    rng = np.random.default_rng(V)
    x = rng.standard_normal((5, V)).astype(np.float32)
    rows = (np.arange(n_rows) * 3 % 5).astype(np.int32)
    dx, dr = mk.to_device(x), mk.to_device(rows)
    dv, di = mk.alloc(n_rows * k * 4), mk.alloc(n_rows * k * 4)
    print("topk many rows", V, k, n_rows, flush=True)
    mk_.check(mk_.load().mk_topk(mk.h, dx.ptr, V, dr.ptr, n_rows, V, k, dv.ptr, di.ptr))
    gv, gi = dv.download(np.uint32).reshape(n_rows, k), di.download(np.int32).reshape(n_rows, k)
    for r in range(5):
        ev, ei = expected_topk(x[r], k)
        assert (gi[rows == r] == ei).all() and (gv[rows == r] == ev.view(np.uint32)).all()
