"""The backward's chunk kernels where a chunk's output tiles are shared out over
several workgroups, in 64- and 128-wide tiles with remainders, against float64
autograd through the CPU oracle (the bars of test_gpu_backward)."""

import pytest
import torch

import test_gpu_backward as tb
from tolerance import metrics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,H,K,V,M,dtype", [
    (2, 1000, 3, 256, 256, 128, torch.bfloat16),  # 96 chunks: 128-wide tiles, three workgroups per chunk
    (2, 1000, 3, 256, 256, 128, torch.float32),
    (3, 700, 4, 192, 320, 96, torch.float32),     # ragged 128-wide tiles
    (2, 500, 2, 68, 36, 20, torch.float32),       # one 64-wide tile and a remainder
    (2, 330, 3, 150, 70, 32, torch.float32),      # rows that are no multiple of 4: 4-byte operand loads
])
def test_shared_out_chunks_match_oracle_autograd(B, T, H, K, V, M, dtype):
    x, init, cot = tb._inputs(B, T, H, K, V, M, seed=T + K, dtype=dtype, state=True)
    ref = tb._oracle_grads(x, init, cot, True, 64)
    got = tb._gpu_grads(x, init, cot, True, 64)
    for name, r in ref.items():
        m = metrics(got[name].float(), r)
        assert m["rrms"] < tb._bar(name, dtype), f"{name}: {m}"
