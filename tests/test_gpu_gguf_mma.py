"""mk_matmul_gguf's forms, bit for bit against the CPU oracle's panel arithmetic: the 16-lanes-per-row kernel (1, 2 and up
to 4 tokens per pass, an odd last super-block, rows past the last workgroup), unaligned rows, which keep the byte-wise
kernel, and the int8 MFMA kernel of Q5_K batches (quarters of a 32-token tile skipped, partial row and token tiles, rings
of 6 and of 3 stages, refilled)."""
import numpy as np
import pytest

import malkin_amd as mk_
from oracle import bind
from test_gpu_rowpath import bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [bind.Q4_K, bind.Q5_K])
@pytest.mark.parametrize("rows,k,n,pad", [(17, 256, 1, 0), (72, 768, 2, 0), (40, 1280, 3, 0), (33, 512, 4, 16),
                                          (136, 512, 5, 0), (24, 1536, 8, 0), (264, 512, 9, 16), (129, 256, 16, 0),
                                          (130, 768, 17, 0), (33, 512, 33, 0), (4104, 256, 300, 0), (40, 512, 3, 4),
                                          (40, 512, 20, 4)])
def test_gguf_forms(mk, oracle, t, rows, k, n, pad):
    import make_golden
    rng = np.random.default_rng(t * 31 + rows + k + n)
    w = make_golden.random_rows(rng, t, rows, k)
    x = rng.uniform(-2, 2, (n, k)).astype(np.float32)
    x[:, ::97] *= 50
    x[rng.random((n, k)) < 0.2] = 0
    x[0, :64] = 0  # whole blocks of zeros
    xq = oracle.quantize_row_q8(x)
    exp = oracle.matmul(t, w, rows, k, xq.reshape(-1))
    wp = np.zeros((rows, w.shape[1] + pad), np.uint8)  # rows `pad` bytes apart
    wp[:, :w.shape[1]] = w
    dw, dq = mk.to_device(wp), mk.to_device(xq)
    y0 = rng.standard_normal((n, rows)).astype(np.float32)
    for acc in (0, 1):
        dy = mk.to_device(y0)
        print("gguf forms", t, rows, k, n, pad, acc, flush=True)
        mk_.check(mk_.load().mk_matmul_gguf(mk.h, t, dw.ptr, wp.shape[1], rows, k, dq.ptr, n, dy.ptr, rows, acc))
        got = dy.download(np.float32).reshape(n, rows)
        want = (y0 + exp) if acc else exp
        assert np.array_equal(bits(got), bits(want)), np.abs(got - want).max()


def check(mk, oracle, t, rows, k, n, pad):
    import make_golden
    rng = np.random.default_rng(t * 31 + rows + k + n)
    w = make_golden.random_rows(rng, t, rows, k)
    x = rng.uniform(-2, 2, (n, k)).astype(np.float32)
    x[:, ::97] *= 50
    x[-1, :64] = 0  # whole blocks of zeros
    xq = oracle.quantize_row_q8(x)
    wp = np.zeros((rows, w.shape[1] + pad), np.uint8)  # rows `pad` bytes apart
    wp[:, :w.shape[1]] = w
    y0 = rng.standard_normal((n, rows)).astype(np.float32)
    dw, dq, dy = mk.to_device(wp), mk.to_device(xq), mk.to_device(y0)
    print("gguf forms", t, rows, k, n, pad, flush=True)
    mk_.check(mk_.load().mk_matmul_gguf(mk.h, t, dw.ptr, wp.shape[1], rows, k, dq.ptr, n, dy.ptr, rows, 1))
    got, want = dy.download(np.float32).reshape(n, rows), y0 + oracle.matmul(t, w, rows, k, xq.reshape(-1))
    assert np.array_equal(bits(got), bits(want)), np.abs(got - want).max()


# Past 58 rows x groups of 4 tokens per CU (14848 on 256 CUs), by the tokens of a tile that are computed (8, 16, 32) and
# the ring: 6 stages up to one 128-row tile per CU, 3 past that. 1024 columns are 8 stages, 1280 are 10.
@pytest.mark.parametrize("rows,k,n,pad", [(14977, 1024, 4, 0), (7500, 1280, 8, 16), (5001, 1024, 9, 0),
                                          (3800, 1280, 16, 0), (1900, 1024, 32, 0), (1703, 1280, 33, 16),
                                          (33000, 1024, 5, 0), (33000, 1280, 12, 0), (33001, 1024, 17, 0),
                                          (4104, 1024, 300, 0)])
def test_q5_mfma_forms(mk, oracle, rows, k, n, pad):
    check(mk, oracle, bind.Q5_K, rows, k, n, pad)
