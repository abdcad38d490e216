"""Grouped attention (head_dim 128, trees) where the heads of a KV group are split over two, three or five workgroups,
also unevenly, bit for bit against the oracle's attend_gqa."""
import pytest

from test_gpu_kernels import _attention_vs_oracle, _tree

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,KV,depth", [(40, 8, 3), (40, 8, 6), (32, 8, 6), (24, 8, 7), (5, 1, 25)])
def test_attention_head_sets(mk, oracle, H, KV, depth):
    n, P = 2 * depth + 1, 300
    spec = (128, H, KV, [0] * n, [P] * n, P + n, _tree(P, depth))
    _attention_vs_oracle(mk, oracle, spec, 900 + H + depth, "grouped attention, %d of %d heads" % (H, KV), False)
