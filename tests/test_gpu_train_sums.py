"""The training pass's serial sums (the clock and its cotangent, runs of tokens
per lane in batches of 16; the norm weights' partial rows, eight per lane at a
time) at runs and counts with remainders, against float64 autograd through the
CPU oracle (the bars of test_gpu_backward)."""

import pytest
import torch

import test_gpu_backward as tb
from tolerance import metrics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,H", [
    (2, 3, 1),      # runs of one token, most of them padding
    (1, 1100, 2),   # runs of 18: a batch and two tokens; padding in the last run
    (1, 2049, 17),  # runs of 33; 545 partial rows: a batch of eight per lane and a remainder
])
def test_serial_sums_match_oracle_autograd(B, T, H):
    x, init, cot = tb._inputs(B, T, H, 16, 16, 8, seed=T, dtype=torch.float32, state=True)
    ref = tb._oracle_grads(x, init, cot, True, 64)
    got = tb._gpu_grads(x, init, cot, True, 64)
    for name, r in ref.items():
        m = metrics(got[name].float(), r)
        assert m["rrms"] < tb._bar(name, torch.float32), f"{name}: {m}"


@pytest.fixture(scope="module")
def long_fp32_errors():
    """Relative errors against float64 of the fp32 gradients of 131072 token
    rows (16 blocks of 32 rows per readout workgroup, 2048 chunks): one pass, so
    the kernels' rounding alone, the same on every run."""
    x, init, cot = tb._inputs(4, 4096, 8, 16, 16, 8, seed=4, dtype=torch.float32, state=False)
    ref = tb._oracle_grads(x, init, cot, False, 64)
    got = tb._gpu_grads(x, init, cot, False, 64)
    return {name: metrics(got[name], r)["rrms"] for name, r in ref.items()}


# what fp32 FMA loops over the tokens and rows, in order, left on these inputs
# (measured), and half a percent
@pytest.mark.parametrize("name,loops", [("q", 3.796e-7), ("k", 4.013e-7), ("v", 3.034e-7),
                                        ("readout", 5.572e-7), ("g", 4.79e-7), ("beta", 3.254e-7),
                                        ("delta", 5.014e-6)])
def test_fp32_gradients_are_no_further_off_than_loops(long_fp32_errors, name, loops):
    assert long_fp32_errors[name] <= 1.005 * loops
