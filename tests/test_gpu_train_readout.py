"""The slot readout and its adjoint for bf16 calls at the edges of their tiles:
slot counts that are no multiple of 16 (or of 4), the fewest and the most of one
wave group, several blocks of 32 rows per workgroup with a last workgroup that
is not full, against float64 autograd through the CPU oracle (the bars of
test_gpu_backward)."""

import pytest
import torch

import test_gpu_backward as tb
from tolerance import metrics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,H,K,V,M", [
    (1, 40, 1, 32, 32, 4),      # the fewest slots, rows past T in the block
    (2, 70, 2, 32, 48, 6),      # pairs that end inside a lane's four slots
    (1, 130, 3, 64, 32, 98),
    (3, 1500, 4, 32, 32, 128),  # 144 blocks per head: 3 per workgroup (adjoint), 2 (forward)
    (1, 2200, 5, 32, 32, 34),   # 70 blocks per head, 2 per workgroup
])
def test_readout_edges_match_oracle_autograd(B, T, H, K, V, M):
    x, init, cot = tb._inputs(B, T, H, K, V, M, seed=T + M, dtype=torch.bfloat16, state=True)
    ref = tb._oracle_grads(x, init, cot, True, 64)
    got = tb._gpu_grads(x, init, cot, True, 64)
    for name, r in ref.items():
        m = metrics(got[name].float(), r)
        assert m["rrms"] < tb._bar(name, torch.bfloat16), f"{name}: {m}"
