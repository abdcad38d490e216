"""Prompt-chunk attention on the fp32 matrix cores (head_dim 128, 16 tokens or more), bit for bit against the oracle's
attend_gqa: keys around its 16-key tiles and 64-key stages, G that does not divide 16, blocks of mixed sequences, the
longest rows its LDS holds (1856 keys), and just longer ones, which its form of 512-key chunks or the grouped kernel takes
(test_gpu_attn_mixed.py has that form's cases)."""
import ctypes

import numpy as np
import pytest

import malkin_amd as mk_
import test_gpu_kernels
from test_gpu_kernels import L
from test_gpu_kernels import test_attention_batch_vs_oracle as check_batch

pytestmark = pytest.mark.gpu

CASES = [  # D, H, KV, sequence per token, keys per token, n_ctx
    (128, 2, 2, [0] * 20, [t + 1 for t in range(20)], 32),
    (128, 6, 2, [0] * 16, [15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 66, 127, 128, 129], 129),
    (128, 7, 1, [0] * 9 + [1] * 9, [190 + t for t in range(9)] + [1 + t for t in range(9)], 200),
    (128, 12, 1, [t % 2 for t in range(16)], [1856 - 100 * t for t in range(16)], 1856),
    (128, 8, 8, [0] * 70, [1857 + t for t in range(70)], 1930),
    (128, 16, 8, [0] * 45 + [1] * 25, [2000 + t for t in range(45)] + [500 + 7 * t for t in range(25)], 2048),
]


@pytest.mark.parametrize("case", CASES, ids=[f"H{c[1]}KV{c[2]}keys{max(c[4])}" for c in CASES])
def test_attention_mma(mk, oracle, monkeypatch, case):
    monkeypatch.setattr(test_gpu_kernels, "ROWS_CASES", [case])
    check_batch(mk, oracle, 0)


@pytest.mark.parametrize("n,first", [(16, 200), (70, 1900)], ids=["whole", "chunks"])
def test_keys_of_other_rows(mk, n, first):
    """Token t has the keys below first + t; the key that an odd token adds has scales of infinity. The tokens before
    it, of which some share its workgroups (4 tokens each), keep their results to the bit."""
    D, H, KV, n_ctx = 128, 32, 8, first + n
    rng = np.random.default_rng(9)
    k8, v8 = (rng.integers(-127, 128, (1, KV, n_ctx, D), dtype=np.int8) for _ in range(2))
    ks, vs = (rng.uniform(0.001, 0.05, (1, KV, n_ctx)).astype(np.float32) for _ in range(2))
    q = rng.standard_normal((n, H * D)).astype(np.float32)
    nks = np.arange(first, first + n, dtype=np.int32)
    dk, dv, dq = mk.to_device(k8), mk.to_device(v8), mk.to_device(q)
    dseq, dnk, out = mk.to_device(np.zeros(n, np.int32)), mk.to_device(nks), mk.alloc(n * H * D * 4)

    def run():
        dks, dvs = mk.to_device(ks), mk.to_device(vs)
        kv = mk_.MkKvCache(dk.ptr, dv.ptr, dks.ptr, dvs.ptr, 1, 1, KV, D, n_ctx)
        mk_.check(L().mk_attention(mk.h, dq.ptr, H * D, out.ptr, H * D, n, H, ctypes.byref(kv), 0, dseq.ptr, dnk.ptr,
                                   None, None, int(nks[-1])))
        return out.download(np.float32).reshape(n, H * D).view(np.uint32)

    plain = run()
    cut = n // 2 | 1
    at = nks[cut] - 1
    ks[:, :, at] = vs[:, :, at] = np.inf
    got = run()
    assert np.array_equal(got[:cut], plain[:cut])
    assert not np.array_equal(got[cut:], plain[cut:])
