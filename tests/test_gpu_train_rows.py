"""The backward's v, dO and dv rows: read and written in place where their rows
take 16-byte accesses, else through head-major copies. Both against float64
autograd through the CPU oracle (the bars of test_gpu_backward), and bit for
bit against each other."""

import pytest
import torch

import test_gpu_backward as tb
from tolerance import metrics

pytestmark = pytest.mark.gpu


def _misaligned(t):
    """t's values, contiguous, off the 16-byte grid."""
    base = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    out = base[1:].view(t.shape)
    return out.copy_(t)


# a chunk's last rows missing, heads side by side, V of one vector, of a
# partial tile and of no multiple of 4 (copies)
@pytest.mark.parametrize("B,T,H,K,V,M,dtype", [
    (2, 65, 3, 32, 4, 16, torch.bfloat16), (1, 127, 2, 64, 72, 32, torch.float32),
    (2, 1, 2, 16, 64, 8, torch.bfloat16), (1, 200, 2, 32, 70, 16, torch.bfloat16), (3, 90, 1, 32, 68, 6, torch.bfloat16)])
def test_value_rows_match_oracle_autograd(B, T, H, K, V, M, dtype):
    x, init, cot = tb._inputs(B, T, H, K, V, M, seed=T + V, dtype=dtype, state=True)
    ref = tb._oracle_grads(x, init, cot, True, 64)
    got = tb._gpu_grads(x, init, cot, True, 64)
    for name, r in ref.items():
        m = metrics(got[name].float(), r)
        assert m["rrms"] < tb._bar(name, dtype), f"{name}: {m}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_value_rows_in_place_and_copied_agree(dtype):
    from cyclic_flow_attention.ops import chunk_cyfa

    x, init, cot = tb._inputs(2, 150, 2, 64, 72, 32, seed=4, dtype=dtype, state=False)
    xg = {n: t.to("cuda").requires_grad_(True) for n, t in x.items()}
    o, _ = chunk_cyfa(**xg)
    do = cot["o"].to("cuda")
    placed = torch.autograd.grad(o, list(xg.values()), do, retain_graph=True)
    copied = torch.autograd.grad(o, list(xg.values()), _misaligned(do))
    for name, a, b in zip(xg, placed, copied):
        assert torch.equal(a, b), name
