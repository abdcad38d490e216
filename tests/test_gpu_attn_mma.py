"""Prompt-chunk attention on the fp32 matrix cores (head_dim 128, 16 tokens or more), bit for bit against the oracle's
attend_gqa: keys around its 16-key tiles and 64-key stages, G that does not divide 16, blocks of mixed sequences, the
longest rows its LDS holds (1856 keys), and longer ones in 512-key chunks."""
import pytest

import test_gpu_kernels
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
