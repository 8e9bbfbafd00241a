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
