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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_readout_rows_of_other_sequences_stay_apart(dtype):
    """Per-row buffers of more than 2^31 bytes (43000 sequences of 128 rows, 100
    slots): a sequence of NaNs leaves every other one as it is."""
    from cyclic_flow_attention.ops import chunk_cyfa

    gen = torch.Generator(device="cuda").manual_seed(3)
    B, T, K, M = 43000, 100, 16, 100

    def rnd(*shape):
        return torch.randn(*shape, device="cuda", generator=gen)

    x = dict(q=rnd(B, T, 1, K).to(dtype), k=rnd(B, T, 1, K).to(dtype), v=rnd(B, T, 1, K).to(dtype),
             g=torch.nn.functional.logsigmoid(rnd(B, T, 1) + 3), delta=torch.sigmoid(rnd(B, T, 1)),
             beta=torch.sigmoid(rnd(B, T, 1)), readout=torch.eye(M - 1, device="cuda").expand(1, -1, -1).clone(),
             q_norm_weight=torch.ones(K, device="cuda"), k_norm_weight=torch.ones(K, device="cuda"))
    with torch.no_grad():
        o = chunk_cyfa(**x)[0]
        x["k"][-1100:] = float("nan")
        p = chunk_cyfa(**x)[0]
    assert o.isfinite().all().item() and torch.equal(p[:-1100], o[:-1100])


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
