"""mk_matmul_rows for F32 / F16 / BF16 rows on the matrix cores, bit for bit against the CPU oracle, where the kernel's
forms and edges meet: few tokens (4 staged) on one and several workgroups per CU, 16 x 16, 16 x 32 and 32 x 32 tiles, each
over more stages than its ring holds, rows and tokens past the last tile, partial 64-column steps, k % 16 tails,
strided activations, and the unaligned rows that keep the lane-group kernel. Weights and activations hold signed zeros and denormals."""
import numpy as np
import pytest

import malkin_amd as mk_
from oracle import bind
from test_gpu_rowpath import bits, row_weights

pytestmark = pytest.mark.gpu

CASES = [(40, 16, 1), (40, 4100, 4), (4104, 80, 4), (4104, 80, 5), (24, 1032, 16), (56, 200, 33), (4000, 72, 50),
         (8200, 144, 97), (8193, 64, 128), (24, 36, 3), (24, 100, 20),
         # on 256 CUs the 4-token form past one tile per CU, 16 x 32 and 32 x 32 tiles, over 5 or 6 stages of their rings
         (4104, 1300, 4), (4000, 520, 50), (8200, 652, 97)]


@pytest.mark.parametrize("t", [bind.F32, bind.F16, bind.BF16])
@pytest.mark.parametrize("rows,k,n", CASES)
def test_rows_mfma_vs_oracle(mk, oracle, t, rows, k, n):
    rng = np.random.default_rng(t * 31 + rows + k + n)
    w = row_weights(rng, t, rows, k)
    h = w.view(np.uint32 if t == bind.F32 else np.uint16).reshape(rows, k)
    h[rng.random((rows, k)) < 0.02] = 0x80000000 if t == bind.F32 else 0x8000
    h[rng.random((rows, k)) < 0.02] = 3  # denormal
    x = rng.uniform(-2, 2, (n, k)).astype(np.float32)
    x[rng.random((n, k)) < 0.02] = -0.0
    x[rng.random((n, k)) < 0.02] = 1e-41
    xs = k + 4 - k % 4
    xp = np.full((n, xs), np.nan, np.float32)  # never read
    xp[:, :k] = x
    exp = oracle.matmul_rows(t, w, rows, k, x=x, xq=None, n=n)
    dw, dx = mk.to_device(w), mk.to_device(xp)
    y0 = rng.standard_normal((n, rows)).astype(np.float32)
    for acc in (0, 1):
        dy = mk.to_device(y0)
        print("rows mfma", t, rows, k, n, "accumulate", acc, flush=True)
        mk_.check(mk_.load().mk_matmul_rows(mk.h, t, dw.ptr, w.shape[1], rows, k, dx.ptr, xs, None, n, dy.ptr, rows, acc))
        got = dy.download(np.float32).reshape(n, rows)
        want = (y0 + exp) if acc else exp
        assert np.array_equal(bits(got), bits(want)), (t, rows, k, n, acc, np.abs(got - want).max())
