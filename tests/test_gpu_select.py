"""mk_topk where its forms meet: rows that one workgroup takes alone (up to 8192 logits), rows cut into 64 slices, slices
of 4, 8, 12 or 16 logits a thread, slices walked in rounds (more than 4096 logits each), rows whose largest logits fall
into a few slices (which are then walked whole), and many rows, against numpy's stable order."""
import numpy as np
import pytest

import malkin_amd as mk_
from test_gpu_sampling import expected_topk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V,k,n_rows", [(8192, 1024, 2), (8193, 257, 2), (8193, 1024, 5), (32 * 1024 + 5, 1, 2),
                                        (65536, 40, 3), (65537, 700, 3), (131072, 40, 3), (131073, 999, 3),
                                        (196608, 40, 3), (196609, 500, 3),
                                        (64 * 4096, 300, 3), (64 * 4096 + 1, 300, 3), (64 * 4096 + 64, 1024, 3),
                                        (1 << 20, 1000, 3), (20000, 128, 70), (20000, 129, 3), (151936, 1024, 30)])
def test_topk_forms(mk, V, k, n_rows):
    rng = np.random.default_rng(V + k)
    x = rng.standard_normal((n_rows, V)).astype(np.float32)
    x[0] = np.round(x[0] * 2) / 2      # ties across slices
    if n_rows > 1:
        x[1] = -np.inf                 # every logit equal and the lowest
        x[1, V // 2] = np.float32(1.0)
    if n_rows > 2:
        x[2, np.arange(V) // 64 % 64 == 5] += 20.0  # the largest logits in one slice
    dx = mk.to_device(x)
    dv, di = mk.alloc(n_rows * k * 4), mk.alloc(n_rows * k * 4)
    print("topk forms", V, k, n_rows, flush=True)
    mk_.check(mk_.load().mk_topk(mk.h, dx.ptr, V, None, n_rows, V, k, dv.ptr, di.ptr))
    gv, gi = dv.download(np.float32).reshape(n_rows, k), di.download(np.int32).reshape(n_rows, k)
    for r in range(n_rows):
        ev, ei = expected_topk(x[r], k)
        assert np.array_equal(gi[r], ei), (V, k, r)
        assert np.array_equal(gv[r].view(np.uint32), ev.view(np.uint32)), (V, k, r)


@pytest.mark.parametrize("V,k", [(8193, 40), (8193, 1024), (20000, 256), (151936, 18), (151936, 1024), (1 << 19, 700)])
@pytest.mark.parametrize("n_full", [1, 3, 64])
def test_topk_full_slices(mk, V, k, n_full):
    """Rows whose largest logits fall into n_full of the 64 slices, with ties, distinct or all equal."""
    rng = np.random.default_rng(V + k + n_full)
    x = rng.standard_normal((3, V)).astype(np.float32)
    x[:, np.isin(np.arange(V) // 64 % 64, rng.permutation(64)[:n_full])] += 8.0
    x[1] = np.round(x[1])
    x[2] = 0.5
    dx, dv, di = mk.to_device(x), mk.alloc(3 * k * 4), mk.alloc(3 * k * 4)
    print("topk full slices", V, k, n_full, flush=True)
    mk_.check(mk_.load().mk_topk(mk.h, dx.ptr, V, None, 3, V, k, dv.ptr, di.ptr))
    gv, gi = dv.download(np.uint32).reshape(3, k), di.download(np.int32).reshape(3, k)
    for r in range(3):
        ev, ei = expected_topk(x[r], k)
        assert np.array_equal(gi[r], ei) and np.array_equal(gv[r], ev.view(np.uint32)), (V, k, n_full, r)
