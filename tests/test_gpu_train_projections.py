"""The four projections of a training step as one function (q, k and v with
their short convolutions, and the gate) against float64 autograd of the same in
plain torch, and the layers that must not take it."""

import pytest
import torch

from cyclic_flow_attention import CyclicFlowAttention
from cyclic_flow_attention.layers.autograd import projections
from cyclic_flow_attention.layers.cyfa import general_projections

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _rel(a, b):
    return ((a.double().cpu() - b).norm() / b.norm().clamp_min(1e-30)).item()


def _values(D, widths, rank, Dv, W, bias, dtype, gen):
    def rnd(*shape, scale=1.0):
        return (scale * torch.randn(*shape, generator=gen)).to(dtype)

    proj = [rnd(n, D, scale=D ** -0.5) for n in (*widths, rank)]
    conv = [rnd(n, W, scale=W ** -0.5) for n in widths]
    cb = [rnd(n, scale=0.1) if bias else None for n in widths]
    return [*proj, rnd(Dv, rank, scale=rank ** -0.5), rnd(Dv, scale=0.1), *conv, *cb]


def _call(x, w):
    return projections(x, w[:4], w[4], w[5], w[6:9], w[9:12], general_projections)


# equal widths (one convolution launch over parts) and unequal ones, with and
# without biases, one token, remainders of the convolution's runs and blocks
@pytest.mark.parametrize("B,T,D,widths,rank,W,bias,dtype", [
    (1, 1, 8, (8, 8, 8), 8, 4, True, torch.float32), (2, 67, 64, (64, 64, 64), 24, 4, False, torch.bfloat16),
    (1, 130, 40, (264, 264, 264), 32, 3, True, torch.bfloat16), (2, 33, 72, (24, 24, 48), 16, 4, True, torch.float32),
    (3, 50, 128, (64, 64, 40), 40, 2, False, torch.bfloat16)])
def test_projection_gradients(B, T, D, widths, rank, W, bias, dtype):
    """bf16: the projections and their cotangents are rounded (at most 2^-8 of
    each value) before the convolution, the gate product and the sums, and the
    results again. fp32: sums of at most a few hundred terms, 64 roundings."""
    gen = torch.Generator().manual_seed(T + D)
    w = _values(D, widths, rank, widths[2], W, bias, dtype, gen)
    x = torch.randn(B, T, D, generator=gen).to(dtype)
    cots = [torch.randn(B, T, n, generator=gen).to(dtype) for n in (*widths, widths[2])]
    ref = [None if t is None else t.double().requires_grad_(True) for t in (x, *w)]
    ro = general_projections(*ref)
    rg = torch.autograd.grad(ro, [t for t in ref if t is not None], [c.double() for c in cots])
    got = [None if t is None else t.to(DEV).requires_grad_(True) for t in (x, *w)]
    leaves = [t for t in got if t is not None]
    out = _call(got[0], got[1:])
    cg = [c.to(DEV) for c in cots]
    g = torch.autograd.grad(out, leaves, cg, retain_graph=True)
    again = torch.autograd.grad(out, leaves, cg)
    bar = 2 * 2.0 ** -8 if dtype == torch.bfloat16 else 64 * 2.0 ** -24
    for a, r in zip(out, ro):
        assert a.shape == r.shape and _rel(a.detach(), r.detach()) <= bar
    for a, b, r, leaf in zip(g, again, rg, leaves):
        assert a.dtype == leaf.dtype and a.shape == r.shape and torch.equal(a, b)
        assert _rel(a, r) <= bar
    # a recorded backward, and one for a part of the inputs
    rec = torch.autograd.grad(_call(got[0], got[1:]), leaves, cg, create_graph=True)
    assert rec[0].requires_grad and all(_rel(a.detach(), r) <= 2 * bar for a, r in zip(rec, rg))
    frozen = [None if t is None else t.detach() for t in got[1:]]
    gx, = torch.autograd.grad(_call(got[0], frozen), got[0], cg)
    assert torch.equal(gx, g[0])
    wk = frozen[1].requires_grad_(True)
    gk, = torch.autograd.grad(_call(got[0].detach(), frozen), wk, cg)
    assert torch.equal(gk, g[2])


def test_layer_takes_projections_only_when_plain():
    torch.manual_seed(0)
    layer = CyclicFlowAttention(hidden_size=64, num_heads=2, head_dim=32, num_slots=16).to(DEV)
    x = torch.randn(2, 40, 64, device=DEV)

    def names(y):
        seen, todo = set(), [y.grad_fn]
        while todo:
            f = todo.pop()
            if f is not None and f not in seen:
                seen.add(f)
                todo += [n for n, _ in f.next_functions]
        return {f.name() for f in seen}

    def grads(y):
        return torch.autograd.grad(y.pow(2).sum(), list(layer.parameters()))

    y = layer(x)[0]
    assert "ProjectionsBackward" in names(y)
    ref = grads(y)
    calls = []
    for m in (layer.k_conv1d, layer.g_proj, layer.v_proj):
        hook = m.register_forward_hook(lambda *_: calls.append(1))
        z = layer(x)[0]
        hook.remove()
        assert "ProjectionsBackward" not in names(z)
        # fp32 sums in another order; the gradients pass several hundred terms
        assert _rel(z.detach(), y.detach().double().cpu()) <= 1e-5
        for a, r in zip(grads(z), ref):
            assert _rel(a, r.double().cpu()) <= 1e-4
    assert len(calls) == 3
    for kwargs in (dict(use_cache=True), dict(attention_mask=torch.ones(2, 40, device=DEV))):
        z, cache = layer(x, **kwargs)
        assert "ProjectionsBackward" not in names(z)
    layer.q_proj = torch.nn.Linear(64, 64, bias=True, device=DEV)
    assert "ProjectionsBackward" not in names(layer(x)[0])
