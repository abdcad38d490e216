"""mk_qk_norm_rope_kv at head_dim 128: the form with 16 lanes per head (16-byte aligned rows) against the one-wave form
that rows of an odd stride take, every q, k and cache byte, where heads do not fill a workgroup, with rows of zeros and of
infinities."""
import ctypes

import numpy as np
import pytest

import malkin_amd as mk_

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,H,KV", [(1, 1, 1), (1, 16, 8), (5, 7, 1), (17, 40, 8), (65, 32, 8)])
def test_qk_norm_rope_forms(mk, n, H, KV):
    D, n_ctx, n_seq = 128, 96, 2
    QKV, L = (H + 2 * KV) * D, mk_.load()
    rng = np.random.default_rng(n * H)
    x = (rng.standard_normal((n, QKV)) * 10.0 ** rng.integers(-3, 4, (n, 1))).astype(np.float32)
    x[n // 2, :D], x[n // 2, -D:] = 0.0, 0.0
    x[-1, H * D] = x[-1, -1] = np.inf
    norms = mk.to_device(rng.uniform(0.5, 1.5, 2 * D).astype(np.float32))
    ang = np.arange(n_ctx)[:, None] * 0.01 * (np.arange(D // 2) + 1)
    cos, sin = mk.to_device(np.cos(ang).astype(np.float32)), mk.to_device(np.sin(ang).astype(np.float32))
    pos = mk.to_device(rng.permutation(n_ctx)[:n].astype(np.int32))
    seq = mk.to_device((np.arange(n) % n_seq).astype(np.int32))
    print("qk_norm_rope", n, H, KV, flush=True)
    got = []
    for stride in (QKV, QKV + 1):
        rows = np.zeros((n, stride), np.float32)
        rows[:, :QKV] = x
        d = mk.to_device(rows)
        size = n_seq * KV * n_ctx
        kv8 = [mk.to_device(np.full(size * D, 7, np.int8)) for _ in range(2)]
        kvs = [mk.to_device(np.full(size, 3, np.float32)) for _ in range(2)]
        kv = mk_.MkKvCache(kv8[0].ptr, kv8[1].ptr, kvs[0].ptr, kvs[1].ptr, 1, n_seq, KV, D, n_ctx)
        mk_.check(L.mk_qk_norm_rope_kv(mk.h, d.ptr, d.offset(H * D * 4), d.offset((H + KV) * D * 4), stride, n, H,
                                       norms.ptr, norms.offset(D * 4), ctypes.c_float(1e-6), cos.ptr, sin.ptr, pos.ptr,
                                       seq.ptr, pos.ptr, ctypes.byref(kv), 0))
        got.append([d.download(np.float32).reshape(n, stride)[:, :QKV].copy().view(np.uint32)]
                   + [b.download(np.uint8) for b in kv8] + [b.download(np.uint32) for b in kvs])
    for a, b in zip(*got):
        assert np.array_equal(a, b)
