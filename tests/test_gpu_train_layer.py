"""The layer-side HIP kernels of a training step against float64 autograd of
the same operation in plain torch, and the calls that must not take them."""

import pytest
import torch
import torch.nn.functional as F

from cyclic_flow_attention.layers.cyfa import ShortConvolution

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _rel(a, b):
    return ((a.double().cpu() - b).norm() / b.norm().clamp_min(1e-30)).item()


def _bar(dtype):
    """bf16 results are rounded once from an fp32 sum: each value within half
    an ulp, at most 2^-8 of itself (8 significant bits), so the 2-norm is too; fp32 sums of up to a few
    hundred terms, added pairwise or in runs of 16, stay within 16 roundings."""
    return 2.0 ** -8 if dtype == torch.bfloat16 else 16 * 2.0 ** -24


def _conv64(x, w, bias, cache):
    W = w.shape[-1]
    h = F.pad(x, (0, 0, W - 1, 0)) if cache is None else torch.cat([cache, x], 1)
    y = F.conv1d(h.transpose(1, 2), w, bias, groups=x.shape[-1]).transpose(1, 2)
    return y


# one token, runs of 16 and workgroups of 64 tokens with remainders, channel
# blocks of 256 with remainders, every width
@pytest.mark.parametrize("B,T,D,W,bias,cache,dtype", [
    (1, 1, 8, 4, True, True, torch.bfloat16), (2, 2, 24, 4, False, False, torch.float32),
    (3, 17, 256, 4, True, False, torch.bfloat16), (1, 64, 264, 3, False, True, torch.float32),
    (2, 65, 1024, 4, False, False, torch.bfloat16), (1, 700, 512, 2, True, True, torch.bfloat16),
    (2, 333, 768, 4, True, True, torch.float32), (1, 5000, 72, 4, False, False, torch.bfloat16)])
def test_short_conv_training_gradients(B, T, D, W, bias, cache, dtype):
    gen = torch.Generator().manual_seed(B * 1000 + T + D)
    conv = ShortConvolution(D, W, bias)
    with torch.no_grad():
        for p in conv.parameters():
            p.copy_(0.5 * torch.randn(p.shape, generator=gen))
    conv = conv.to(dtype)
    x = torch.randn(B, T, D, generator=gen).to(dtype)
    c = torch.randn(B, W - 1, D, generator=gen).to(dtype) if cache else None
    dy = torch.randn(B, T, D, generator=gen).to(dtype)
    ref = [None if t is None else t.detach().double().requires_grad_(True) for t in (x, conv.weight, conv.bias, c)]
    ry = _conv64(*ref)
    rg = torch.autograd.grad(ry, [t for t in ref if t is not None], dy.double())
    conv = conv.to(DEV)
    xg = x.to(DEV).requires_grad_(True)
    cg = None if c is None else c.to(DEV).requires_grad_(True)
    leaves = [xg, conv.weight] + ([conv.bias] if bias else []) + ([cg] if cache else [])
    y, _ = conv(xg, cg)
    assert y.grad_fn.name() == "ShortConvBackward"
    g = torch.autograd.grad(y, leaves, dy.to(DEV), retain_graph=True)
    again = torch.autograd.grad(y, leaves, dy.to(DEV))
    assert _rel(y.detach(), ry.detach()) <= _bar(dtype)
    for a, b, r in zip(g, again, rg):
        assert a.dtype == dtype and a.shape == r.shape
        assert torch.equal(a, b)
        assert _rel(a, r) <= _bar(dtype)


def test_short_conv_training_views_second_derivatives_and_transforms():
    """A misaligned, strided x; a second derivative (through the torch path);
    vmap and forward-mode calls keep the torch path."""
    gen = torch.Generator().manual_seed(3)
    conv = ShortConvolution(16, 4).to(DEV)
    base = torch.randn(2, 40, 33, generator=gen).to(DEV)
    x = base[:, ::2, 1:17].detach().requires_grad_(True)
    ref = x.detach().double().cpu().requires_grad_(True)
    w64 = conv.weight.detach().double().cpu()
    y, _ = conv(x)
    ry = _conv64(ref, w64, None, None)
    gx, = torch.autograd.grad(y.pow(3).sum(), x, create_graph=True)
    rx, = torch.autograd.grad(ry.pow(3).sum(), ref, create_graph=True)
    gg, = torch.autograd.grad(gx.pow(2).sum(), x)
    rr, = torch.autograd.grad(rx.pow(2).sum(), ref)
    assert _rel(gx.detach(), rx.detach()) < 1e-5 and _rel(gg, rr) < 1e-5
    xs = torch.randn(3, 2, 20, 16, generator=gen).to(DEV)
    out = torch.func.vmap(lambda t: conv(t)[0])(xs)
    assert _rel(out.detach(), torch.stack([_conv64(t.double().cpu(), w64, None, None) for t in xs])) < 1e-6
    _, tangent = torch.func.jvp(lambda t: conv(t)[0], (xs[0],), (xs[1],))
    assert _rel(tangent.detach(), _conv64(xs[1].double().cpu(), w64, None, None)) < 1e-6
