"""The attention layer calls modules that replace its own, or carry hooks, as it
documents them."""

import torch

from cyclic_flow_attention import CyclicFlowAttention
from cyclic_flow_attention.layers import cyfa


def test_replaced_or_hooked_output_norm_gets_the_scaled_input(monkeypatch):
    """o_norm(o (num_slots - 1), gate): a norm that takes no further argument
    fits in, and a hook sees the scaled input."""
    torch.manual_seed(0)
    layer = CyclicFlowAttention(hidden_size=32, num_heads=2, head_dim=16, num_slots=8)
    o = torch.randn(1, 5, 2, 16)
    monkeypatch.setattr(cyfa, "chunk_cyfa", lambda **_: (o, None))
    x = torch.randn(1, 5, 32)
    plain = layer(x)[0]
    seen = []
    hook = layer.o_norm.register_forward_pre_hook(lambda m, args: seen.append(args))
    hooked = layer(x)[0]
    hook.remove()
    (scaled, gate), = seen
    assert torch.equal(scaled, o * 7) and torch.equal(hooked, plain)

    class Norm(torch.nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner = inner

        def forward(self, x, gate):
            return self.inner(x, gate)

    layer.o_norm = Norm(layer.o_norm)
    assert torch.equal(layer(x)[0], plain)


def _replacements():
    """Modules of a layer's own classes that the fused masked path does not
    compute: (name, module of a layer of 32 columns, 2 heads)."""
    from torch import nn

    for name in ("q_proj", "k_proj", "v_proj", "o_proj"):
        yield name, nn.Linear(32, 32)
    yield "a_proj", nn.Linear(32, 2)
    for name in ("b_proj", "d_proj"):
        yield name, nn.Linear(32, 2, bias=False)
    yield "g_proj", nn.Sequential(nn.Linear(32, 16), nn.Linear(16, 32))
    for name in ("q_conv1d", "k_conv1d", "v_conv1d"):
        yield name, cyfa.ShortConvolution(32, 4, True)
        yield name, cyfa.ShortConvolution(32, 3)
        yield name, cyfa.ShortConvolution(16, 4)
    yield "k_proj", nn.Linear(32, 16, bias=False)


def test_only_layers_with_the_biases_and_sizes_of_the_fused_path_are_plain():
    def layer():
        return CyclicFlowAttention(hidden_size=32, num_heads=2, head_dim=16, num_slots=8)

    assert layer()._plain()
    for name, module in _replacements():
        changed = layer()
        setattr(changed, name, module)
        assert not changed._plain(), (name, module)
    unbiased = layer()  # g_proj[1]'s bias may be missing: the fused path takes that
    unbiased.g_proj[1].bias = None
    assert unbiased._plain()
