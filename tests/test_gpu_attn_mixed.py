"""Plain batches of several sequences on rows longer than attention_mma's LDS holds (head_dim 128, more than 1856 keys),
bit for bit against the oracle's attend_gqa: batches that the device sends to the matrix cores and batches that it leaves
to the grouped kernel (up to about 11500 keys) or k_attention_long; and a model's batches."""
import numpy as np
import pytest

import malkin_amd as mk_
import test_gpu_kernels
from test_gpu_kernels import test_attention_batch_vs_oracle as check_batch

pytestmark = pytest.mark.gpu


def batch(n, prompt, share, longest):
    """The first `prompt` tokens are sequence 1's, then each sequence has `share` tokens; every 5th token has about
    `longest` keys, the others a few."""
    seqs = [1 if t < prompt else 2 + (t - prompt) // share for t in range(n)]
    return seqs, [longest - t // 5 if t % 5 == 0 else 1 + 7 * t % 90 for t in range(n)]


CASES = [  # H, KV, tokens, tokens of sequence 1, tokens of each other one, longest row
    (8, 8, 80, 40, 1, 1900),     # grouped, whatever the sequences
    (8, 8, 130, 130, 1, 1900),   # matrix cores: one sequence, of a cache of several
    (8, 8, 130, 90, 1, 1900),    # grouped
    (32, 8, 70, 70, 1, 2000),    # matrix cores
    (24, 8, 73, 73, 1, 1900),    # matrix cores, blocks of 5 tokens
    (40, 8, 71, 71, 1, 1990),    # matrix cores, blocks of 3 tokens
    (16, 1, 520, 520, 1, 1870),  # matrix cores, blocks of one token
    (48, 8, 64, 20, 1, 1880),    # matrix cores, blocks of 2 tokens
    (64, 4, 33, 20, 1, 1880),    # matrix cores, blocks of one token
    (32, 8, 70, 33, 1, 2000),    # grouped
    (32, 8, 67, 0, 2, 3000),     # matrix cores, two sequences a block
    (32, 8, 70, 33, 1, 3000),    # grouped, a group's heads in workgroups of their own
    (16, 8, 70, 30, 3, 1857),    # grouped
    (40, 8, 71, 31, 2, 1990),    # grouped, all heads; blocks of 3 tokens
    (16, 8, 70, 60, 1, 11700),   # k_attention_long
    (16, 8, 70, 67, 1, 11700),   # matrix cores, a block of 4 sequences
]


@pytest.mark.parametrize("case", CASES, ids=["-".join(map(str, c)) for c in CASES])
def test_mixed_blocks(mk, oracle, monkeypatch, case):
    H, KV, n, prompt, share, longest = case
    seqs, keys = batch(n, prompt, share, longest)
    mk_.check(mk_.load().mk_reserve_scratch(mk.h, 8 << 20))
    monkeypatch.setattr(test_gpu_kernels, "ROWS_CASES", [(128, H, KV, seqs, keys, longest)])
    check_batch(mk, oracle, 0)


def test_model_batches(mk, synth_lib, tmp_path):
    """A model's batches past 1856 keys, whose sequences the host knows: 70 tokens of one sequence, then of 37, against the
    same tokens in batches of 10."""
    path = synth_lib.write_gguf(str(tmp_path / "m.gguf"), synth_lib.make_config(
        "tiny", synth_lib.Q8_0, seed=3, n_layer=1, n_head=16, n_head_kv=8, n_vocab=512))
    m = mk_.Model(mk, path, 2048, 40)
    toks = np.random.default_rng(4).integers(0, 512, 2100).astype(np.int32)
    for at in range(0, 1900, 190):
        m.forward(toks[at:at + 190], at)
    for seqs in ([0] * 70, [0] * 34 + list(range(1, 37))):
        pos = [1900 + t if s == 0 else 0 for t, s in enumerate(seqs)]
        rows = [(int(toks[t]), s, p, 1) for t, (s, p) in enumerate(zip(seqs, pos))]
        whole = m.forward_batch(mk_.batch(rows))
        parts = np.concatenate([m.forward_batch(mk_.batch(rows[i:i + 10])) for i in range(0, 70, 10)])
        assert np.array_equal(whole.view(np.uint32), parts.view(np.uint32))
    m.close()
