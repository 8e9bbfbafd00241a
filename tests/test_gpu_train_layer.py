"""The layer-side HIP kernels of a training step against float64 autograd of
the same operation in plain torch, and the calls that must not take them."""

import pytest
import torch
import torch.nn.functional as F

from cyclic_flow_attention import _native
from cyclic_flow_attention.layers.cyfa import RMSNorm, ShortConvolution

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
    cots = torch.randn(3, 2, 20, 16, generator=gen).to(DEV)
    y, _ = conv(x)
    batched, = torch.autograd.grad(y, x, cots, is_grads_batched=True, retain_graph=True)
    for c, b in zip(cots, batched):
        assert _rel(b, torch.autograd.grad(y, x, c, retain_graph=True)[0].double().cpu()) < 1e-5
    xs = torch.randn(3, 2, 20, 16, generator=gen).to(DEV)
    out = torch.func.vmap(lambda t: conv(t)[0])(xs)
    assert _rel(out.detach(), torch.stack([_conv64(t.double().cpu(), w64, None, None) for t in xs])) < 1e-6
    _, tangent = torch.func.jvp(lambda t: conv(t)[0], (xs[0],), (xs[1],))
    assert _rel(tangent.detach(), _conv64(xs[1].double().cpu(), w64, None, None)) < 1e-6


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_short_conv_of_single_tokens_of_a_time_major_tensor(dtype):
    """x [B, 1, D], a view of [1, B, D] whose stride over the one token spans
    the whole tensor, and the same of the cache [B, 1, D]."""
    gen = torch.Generator().manual_seed(11)
    for W in (2, 4):
        conv = ShortConvolution(24, W, True)
        with torch.no_grad():
            for p in conv.parameters():
                p.copy_(0.5 * torch.randn(p.shape, generator=gen))
        conv = conv.to(dtype)
        base = torch.randn(1, 5, 24, generator=gen).to(dtype)
        cbase = torch.randn(W - 1, 5, 24, generator=gen).to(dtype)
        dy = torch.randn(5, 1, 24, generator=gen).to(dtype)
        ref = [t.detach().double().requires_grad_(True) for t in (base, conv.weight, conv.bias, cbase)]
        ry = _conv64(ref[0].transpose(0, 1), *ref[1:3], ref[3].transpose(0, 1))
        rg = torch.autograd.grad(ry, ref, dy.double())
        conv = conv.to(DEV)
        leaves = [base.to(DEV).requires_grad_(True), conv.weight, conv.bias, cbase.to(DEV).requires_grad_(True)]
        x, cache = leaves[0].transpose(0, 1), leaves[3].transpose(0, 1)
        y, _ = conv(x, cache)
        assert y.grad_fn.name() == "ShortConvBackward" and _rel(y.detach(), ry.detach()) <= _bar(dtype)
        for a, r in zip(torch.autograd.grad(y, leaves, dy.to(DEV)), rg):
            assert _rel(a, r) <= _bar(dtype)
        with torch.no_grad():
            assert _rel(conv(x, cache)[0], ry.detach()) <= _bar(dtype)


@pytest.mark.parametrize("T,dtype", [(1, torch.float32), (13, torch.bfloat16), (21, torch.float32), (66, torch.bfloat16)])
def test_short_conv_gradients_with_an_infinite_last_token(T, dtype):
    """The last row of x meets one tap only: the others' gradients are finite."""
    gen = torch.Generator().manual_seed(T)
    conv = ShortConvolution(16, 4, True).to(dtype).to(DEV)
    x, dy = torch.randn(2, T, 16, generator=gen).to(dtype), torch.randn(2, T, 16, generator=gen).to(dtype)
    x[:, -1] = float("inf")
    h = F.pad(x.double(), (0, 0, 3, 0))
    ref = torch.stack([(dy.double() * h[:, w:w + T]).sum((0, 1)) for w in range(4)], -1)
    y, _ = conv(x.to(DEV).requires_grad_(True))
    gw, gb = torch.autograd.grad(y, [conv.weight, conv.bias], dy.to(DEV))
    assert _rel(gw[:, 0, :3], ref[:, :3]) <= _bar(dtype) and _rel(gb, dy.double().sum((0, 1))) <= _bar(dtype)
    assert torch.equal(gw[:, 0, 3].double().cpu().isfinite(), ref[:, 3].isfinite())


def test_traced_training_calls_record_the_torch_operations():
    """A graph traced from one input gives another input's result."""
    from torch.fx.experimental.proxy_tensor import make_fx

    torch.manual_seed(0)
    conv, norm = ShortConvolution(16, 4).to(DEV), RMSNorm(16, 1e-6).to(DEV)
    x, x2 = torch.randn(2, 20, 16, device=DEV), torch.randn(2, 20, 16, device=DEV)

    def call(t):
        return norm(conv(t)[0])

    graph = make_fx(call)(x)
    assert _rel(graph(x2).detach(), call(x2).detach().double().cpu()) <= 1e-5


def _norm64(x, w, gate, prescale):
    x = x * prescale
    y = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * w
    return y if gate is None else y * torch.sigmoid(gate)


# one row, remainders of a workgroup's 4 and 32 rows, every number of column
# blocks with remainders, with and without the gate and the prescale
@pytest.mark.parametrize("rows,D,gate,prescale,dtype", [
    (1, 4, False, 1.0, torch.float32), (33, 256, True, 127.0, torch.bfloat16), (70, 256, True, 127.0, torch.float32),
    (37, 300, True, 1.0, torch.bfloat16), (64, 1024, False, 1.0, torch.bfloat16), (5, 1536, False, 1.0, torch.float32),
    (2000, 256, True, 127.0, torch.bfloat16), (31, 2048, True, 3.0, torch.bfloat16)])
def test_rms_norm_training_gradients(rows, D, gate, prescale, dtype):
    """For bf16, x prescale is itself rounded (at most 2^-8 of each value), which
    moves the result and the gradients by as much again: two roundings. The
    weight's gradient is an fp32 sum of such terms."""
    gen = torch.Generator().manual_seed(rows + D)
    norm = RMSNorm(D, 1e-6)
    with torch.no_grad():
        norm.weight.copy_(1 + 0.2 * torch.randn(D, generator=gen))
    x = torch.randn(rows, D, generator=gen).to(dtype)
    g = torch.randn(rows, D, generator=gen).to(dtype) if gate else None
    dy = torch.randn(rows, D, generator=gen).to(dtype)
    ref = [None if t is None else t.detach().double().requires_grad_(True) for t in (x, norm.weight, g)]
    ry = _norm64(*ref, prescale)
    rg = torch.autograd.grad(ry, [t for t in ref if t is not None], dy.double())
    norm = norm.to(DEV)
    xg = x.to(DEV).requires_grad_(True)
    gg = None if g is None else g.to(DEV).requires_grad_(True)
    leaves = [xg, norm.weight] + ([gg] if gate else [])
    y = norm(xg, gg, prescale=prescale)
    assert y.grad_fn.name() == "GatedNormBackward"
    got = torch.autograd.grad(y, leaves, dy.to(DEV), retain_graph=True)
    again = torch.autograd.grad(y, leaves, dy.to(DEV))
    bar = 2 * _bar(dtype)
    assert _rel(y.detach(), ry.detach()) <= bar
    for a, b, r, leaf in zip(got, again, rg, leaves):
        assert a.dtype == leaf.dtype and a.shape == r.shape
        assert torch.equal(a, b)
        assert _rel(a, r) <= bar
    # a recorded backward (second derivatives) gives the same first ones
    rec = torch.autograd.grad(norm(xg, gg, prescale=prescale), leaves, dy.to(DEV), create_graph=True)
    for a, r in zip(rec, rg):
        assert a.requires_grad and _rel(a.detach(), r) <= 2 * bar


# rows that leave a place of the last pair of rows empty, and eps that adds nothing
@pytest.mark.parametrize("rows,D", [(1, 256), (3, 1024), (33, 256), (33, 1024), (7, 2048)])
@pytest.mark.parametrize("eps", [0.0, 1e-46])
def test_rms_norm_gradients_without_eps(rows, D, eps):
    gen = torch.Generator().manual_seed(rows + D)
    norm = RMSNorm(D, eps).to(DEV)
    x, g, dy = (torch.randn(rows, D, generator=gen) for _ in range(3))
    ref = [t.detach().double().cpu().requires_grad_(True) for t in (x, norm.weight, g)]
    r = ref[0] * torch.rsqrt(ref[0].pow(2).mean(-1, keepdim=True)) * ref[1] * torch.sigmoid(ref[2])
    rg = torch.autograd.grad(r, ref, dy.double())
    xg, gg = x.to(DEV).requires_grad_(True), g.to(DEV).requires_grad_(True)
    y = norm(xg, gg)
    assert y.grad_fn.name() == "GatedNormBackward"
    for a, b in zip(torch.autograd.grad(y, [xg, norm.weight, gg], dy.to(DEV)), rg):
        assert _rel(a, b) <= 2 * _bar(torch.float32)


def test_rms_norm_of_more_rows_than_a_launch_takes(monkeypatch):
    norm = RMSNorm(64, 1e-6).to(DEV)
    x = torch.randn(5, 7, 64, device=DEV, requires_grad=True)
    y = norm(x)
    monkeypatch.setattr(_native, "NORM_TRAIN_MAX_ROWS", 34)
    z = norm(x)
    assert y.grad_fn.name() == "GatedNormBackward" != z.grad_fn.name()
    assert _rel(z.detach(), y.detach().double().cpu()) <= 1e-6


def test_rms_norm_takes_misaligned_rows():
    norm = RMSNorm(1024, 1e-6).to(DEV)
    x = torch.randn(3 * 1024 + 1, device=DEV).bfloat16()[1:].view(3, 1024)  # rows off the 16-byte grid
    with torch.no_grad():
        assert torch.equal(norm(x), norm(x.clone()))


def _gates64(x, wa, wb, bb, wd, bd, dt_bias, A_log, dtype):
    def rounded(t):  # the projection's rounding, passed straight through by the gradient
        return t + (t.detach().to(dtype).double() - t.detach())

    a, b, d = rounded(x @ wa.mT), rounded(x @ wb.mT + bb), rounded(x.detach() @ wd.mT + bd)
    return -A_log.exp() * F.softplus(a + dt_bias), torch.sigmoid(b), torch.sigmoid(d)


# one row, remainders of 16, 32 and 64 rows, one and two column tiles of the
# projection, both register widths, K with remainders of a step and of 256
@pytest.mark.parametrize("rows,K,H,dtype", [(1, 8, 1, torch.float32), (17, 256, 4, torch.bfloat16),
                                            (65, 1000, 6, torch.float32), (100, 40, 5, torch.bfloat16),
                                            (333, 2048, 8, torch.bfloat16), (3000, 1024, 4, torch.bfloat16),
                                            (70, 264, 3, torch.float32),
                                            (32768 + 41, 264, 2, torch.bfloat16)])  # 128 rows per workgroup
def test_gates_training_gradients(rows, K, H, dtype):
    """bf16: the projections' cotangents are rounded (2^-8 of each) before the
    sums, and the results are rounded again; a projection on a rounding edge may
    go either way, for few values. fp32: dot products and column sums of up to
    3000 terms, whose roundings add up as their square root, 64 of them at most."""
    from cyclic_flow_attention.layers.autograd import gates
    from cyclic_flow_attention.layers.cyfa import general_gates

    gen = torch.Generator().manual_seed(rows + K)

    def rnd(*shape):
        return torch.randn(*shape, generator=gen)

    x = rnd(rows, K).to(dtype)
    ws = [(rnd(H, K) * K ** -0.5).to(dtype) for _ in range(3)]
    bb, bd = (0.1 * rnd(H)).to(dtype), (0.1 * rnd(H)).to(dtype)
    vals = (x, ws[0], ws[1], bb, ws[2], bd, rnd(H) - 2, rnd(H))
    cots = [rnd(rows, H) for _ in range(3)]
    ref = [t.double().requires_grad_(True) for t in vals]
    ro = _gates64(*ref, dtype)
    rg = torch.autograd.grad(ro, ref, [c.double() for c in cots])
    got = [t.to(DEV).requires_grad_(True) for t in vals]
    out = gates(*got, general_gates)
    cg = [c.to(DEV) for c in cots]
    g = torch.autograd.grad(out, got, cg, retain_graph=True)
    again = torch.autograd.grad(out, got, cg)
    bar = 2 * 2.0 ** -8 if dtype == torch.bfloat16 else 64 * 2.0 ** -24
    for a, r in zip(out, ro):
        assert _rel(a.detach(), r.detach()) <= bar
    for a, b, r, leaf in zip(g, again, rg, vals):
        assert a.dtype == leaf.dtype and a.shape == r.shape
        assert torch.equal(a, b)
        assert _rel(a, r) <= bar
    rec = torch.autograd.grad(gates(*got, general_gates), got, cg, create_graph=True)
    assert all(a.requires_grad and _rel(a.detach(), r) <= 2 * bar for a, r in zip(rec, rg))


def test_layer_keeps_wrapped_gate_projections():
    """A hook on a gate projection is called, and a subclass's forward runs."""
    from cyclic_flow_attention import CyclicFlowAttention

    torch.manual_seed(0)
    layer = CyclicFlowAttention(hidden_size=256, num_heads=1).to(DEV)
    x = torch.randn(1, 70, 256, device=DEV, requires_grad=True)
    y, _ = layer(x)
    calls = []
    handle = layer.d_proj.register_forward_hook(lambda *a: calls.append(1))
    y2, _ = layer(x)
    handle.remove()
    assert calls and _rel(y2.detach(), y.detach().double().cpu()) < 1e-5
