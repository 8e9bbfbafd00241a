"""Autograd functions of the layer-side operations, for training on the GPU.

Each runs its forward and its adjoint as HIP kernels behind the C ABI in place
of the chain of torch operations of the module's general path, with the same
result up to rounding and the gradients of that path. A backward pass that is
itself recorded (``create_graph=True``) goes through the general path, so
higher derivatives stay available.
"""

import torch
from torch.autograd import forward_ad

from .. import _native


def hip_autograd_ok(*tensors):
    """Whether a call that records gradients may take these functions: plain
    tensors of one GPU, and nothing that has to see the torch operations
    themselves (torch.func transforms, forward-mode derivatives, tracing or
    compiling, dispatch modes, which make_fx and operation counters are, autocast)."""
    given = [t for t in tensors if t is not None]
    if not all(type(t) in (torch.Tensor, torch.nn.Parameter) and t.is_cuda for t in given):
        return False
    if any(t.device != given[0].device for t in given):
        return False
    return (torch.is_grad_enabled() and not torch.is_autocast_enabled("cuda")
            and torch._C._functorch.peek_interpreter_stack() is None and forward_ad._current_level < 0
            and not torch.compiler.is_compiling() and not torch.jit.is_tracing()
            and torch._C._len_torch_dispatch_stack() == 0)


def _through_torch(*cotangents):
    """Whether a backward pass has to run in torch operations: one that is
    itself recorded, or batched over several cotangents (vmap)."""
    return (torch.is_grad_enabled() or torch._C._functorch.peek_interpreter_stack() is not None
            or any(torch._C._functorch.is_legacy_batchedtensor(t) for t in cotangents))


def _torch_grads(fn, inputs, needed, dy):
    """Gradients of fn(*inputs) by autograd, themselves recorded when this
    backward pass is."""
    recorded = torch.is_grad_enabled()
    with torch.enable_grad():
        wanted = [t for t, n in zip(inputs, needed) if n]
        grads = iter(torch.autograd.grad(fn(*inputs), wanted, dy, create_graph=recorded, allow_unused=True))
    return tuple(next(grads) if n else None for n in needed)


def short_conv(x, weight, bias, cache, general):
    """The causal depthwise convolution (layers/cyfa.py:138-233) with its HIP
    adjoint: x [B, T, D], weight [D, W], bias [D] or None, cache [B, W-1, D] or
    None, all of one dtype (bf16 or fp32). ``general``: the same in torch
    operations."""
    cache = None if cache is None else _native.aligned_rows(cache)
    return ShortConv.apply(_native.aligned_rows(x), weight.contiguous(), bias, cache, general)


class ShortConv(torch.autograd.Function):
    """short_conv's function; every input contiguous."""

    @staticmethod
    def forward(ctx, x, weight, bias, cache, general):
        ctx.save_for_backward(x, weight, bias, cache)
        ctx.general = general
        return _native.short_conv(x, weight, bias, cache)[0]

    @staticmethod
    def backward(ctx, dy):
        x, weight, bias, cache = ctx.saved_tensors
        needed = ctx.needs_input_grad[:4]
        if _through_torch(dy):
            return _torch_grads(ctx.general, (x, weight, bias, cache), needed, dy) + (None,)
        grads = _native.short_conv_grad(x, weight, cache, _native.aligned_rows(dy), needed)
        return (*grads, None)


def rms_norm(x, weight, gate, eps, prescale, general):
    """norm(x prescale) [* sigmoid(gate)] (layers/cyfa.py:62-135) with its HIP
    adjoint: x and gate [..., D] bf16 or fp32 of one dtype, weight fp32 [D].
    ``general``: the same of (x, weight, gate) in torch operations."""
    gate = None if gate is None else _native.aligned_rows(gate)
    return GatedNorm.apply(_native.aligned_rows(x), _native.aligned_rows(weight), gate, eps, prescale, general)


class GatedNorm(torch.autograd.Function):
    """rms_norm's function; every input contiguous."""

    @staticmethod
    def forward(ctx, x, weight, gate, eps, prescale, general):
        ctx.save_for_backward(x, weight, gate)
        ctx.args = (eps, prescale)
        ctx.general = general
        return _native.norm_train(x, weight, gate, eps, prescale)

    @staticmethod
    def backward(ctx, dy):
        x, weight, gate = ctx.saved_tensors
        needed = ctx.needs_input_grad[:3]
        if _through_torch(dy):
            return _torch_grads(ctx.general, (x, weight, gate), needed, dy) + (None,) * 3
        return (*_native.norm_grad(x, weight, gate, *ctx.args, _native.aligned_rows(dy), needed), None, None, None)


def gates(x, wa, wb, bb, wd, bd, dt_bias, A_log, general):
    """The gates (g, beta, delta) fp32 [..., H] of x [..., K] (layers/cyfa.py:
    323-326) with their HIP adjoint: the weights [H, K] and biases [H] of x's
    dtype (bf16 or fp32), dt_bias and A_log fp32 [H]. The clock branch (wd, bd)
    sends no gradient into x. ``general``: the same in torch operations."""
    wa, wb, wd = (_native.aligned_rows(w) for w in (wa, wb, wd))
    flat = _native.aligned_rows(x.reshape(-1, x.shape[-1]))
    bb, bd, dt_bias, A_log = (t.contiguous() for t in (bb, bd, dt_bias, A_log))
    out = Gates.apply(flat, wa, wb, bb, wd, bd, dt_bias, A_log, general)
    return tuple(t.reshape(x.shape[:-1] + t.shape[-1:]) for t in out)


class Gates(torch.autograd.Function):
    """gates' function; every input contiguous, x [rows, K]."""

    @staticmethod
    def forward(ctx, x, wa, wb, bb, wd, bd, dt_bias, A_log, general):
        g, beta, delta, abd = _native.gates_train(x, wa, wb, bb, wd, bd, dt_bias, A_log)
        ctx.save_for_backward(x, wa, wb, bb, wd, bd, dt_bias, A_log, abd)
        ctx.general = general
        return g, beta, delta

    @staticmethod
    def backward(ctx, dg, dbeta, ddelta):
        *inputs, abd = ctx.saved_tensors
        x, wa, wb, _, wd, _, dt_bias, A_log = inputs
        needed = ctx.needs_input_grad[:8]
        if _through_torch(dg, dbeta, ddelta):
            return _torch_grads(ctx.general, inputs, needed, (dg, dbeta, ddelta)) + (None,)
        grads = _native.gates_grad(x, wa, wb, wd, dt_bias, A_log, abd, dg.contiguous(), dbeta.contiguous(),
                                   ddelta.contiguous(), needed[0])
        return tuple(t if n else None for t, n in zip(grads, needed)) + (None,)


def projections(x, proj, gate, gate_bias, conv, conv_bias, general):
    """(q, k, v, gate) [B, T, .] of x [B, T, D]: x against the weights
    ``proj`` = (wq, wk, wv, wg), the short convolutions ``conv`` (weights
    [., W] of one W, with ``conv_bias`` three biases or Nones) of the first
    three, and the product of the fourth with ``gate`` plus gate_bias. One dtype
    (bf16 or fp32). ``general``: the same in torch operations."""
    return Projections.apply(_native.aligned_rows(x), *proj, gate, gate_bias, *conv, *conv_bias, general)


class Projections(torch.autograd.Function):
    """projections' function. The four projections are one product against
    their weights side by side, and so are their adjoints: the cotangents
    gather in one [rows, N] buffer (the convolutions' adjoint and the gate
    product write their columns of it), from which one product each gives the
    cotangents of x and of the four weights. As modules of their own, q, k, v
    and the gate took five matrix products forward and ten backward besides
    three sums of x's cotangents, and three launches of each convolution
    kernel. A training step of 2 x 1500 tokens at 1024 wide is bound by the
    host's work for its launches on MI355X: 1547 us, and 1302 us so, with
    90 us less on the GPU."""

    @staticmethod
    def forward(ctx, x, wq, wk, wv, wg, w2, b2, cq, ck, cv, bq, bk, bv, general):
        ctx.general = general
        widths = [w.shape[0] for w in (wq, wk, wv)]
        n = sum(widths)
        y = torch.mm(x.reshape(-1, x.shape[-1]), torch.cat((wq, wk, wv, wg)).t())
        ctx.save_for_backward(x, wq, wk, wv, wg, w2, b2, cq, ck, cv, bq, bk, bv, y)
        y3 = y.view(*x.shape[:2], y.shape[-1])
        if widths[0] == widths[1] == widths[2]:
            bias = None if bq is None else torch.cat((bq, bk, bv))
            qkv = _native.short_conv(y3[..., :n], torch.cat((cq, ck, cv)), bias, split=widths[0])
        else:
            parts = y3[..., :n].split(widths, -1)
            qkv = [_native.short_conv(p, c, b)[0] for p, c, b in zip(parts, (cq, ck, cv), (bq, bk, bv))]
        gate = torch.nn.functional.linear(y[:, n:], w2, b2)
        return (*qkv, gate.view(*x.shape[:2], gate.shape[-1]))

    @staticmethod
    def backward(ctx, dq, dk, dv, dgate):
        *inputs, y = ctx.saved_tensors
        needed = ctx.needs_input_grad[:13]
        if _through_torch(dq, dk, dv, dgate):
            return _torch_grads(ctx.general, inputs, needed, (dq, dk, dv, dgate)) + (None,)
        x, wq, wk, wv, wg, w2, _, cq, ck, cv = inputs[:10]
        widths = [w.shape[0] for w in (wq, wk, wv)]
        n = sum(widths)
        rows = x.reshape(-1, x.shape[-1])
        y3 = y.view(*x.shape[:2], y.shape[-1])
        dqkv = [_native.aligned_rows(t) for t in (dq, dk, dv)]
        dgate = dgate.reshape(-1, dgate.shape[-1])
        dy = torch.empty_like(y)
        dy3 = dy.view_as(y3)
        conv = (False, any(needed[7:10]), any(needed[10:13]), False)
        if widths[0] == widths[1] == widths[2]:
            _, dc, db, _ = _native.short_conv_grad(y3[..., :n], torch.cat((cq, ck, cv)), None, dqkv, conv, dy3[..., :n])
            dconv = (None,) * 3 if dc is None else dc.split(widths)
            dbias = (None,) * 3 if db is None else db.split(widths)
        else:
            ys, ds = y3[..., :n].split(widths, -1), dy3[..., :n].split(widths, -1)
            grads = [_native.short_conv_grad(a, c.contiguous(), None, g, conv, d) for a, c, g, d in zip(ys, (cq, ck, cv), dqkv, ds)]
            dconv, dbias = [g[1] for g in grads], [g[2] for g in grads]
        torch.mm(dgate, w2, out=dy[:, n:])
        dw = torch.mm(dy.t(), rows).split(widths + [wg.shape[0]]) if any(needed[1:5]) else (None,) * 4
        grads = (torch.mm(dy, torch.cat((wq, wk, wv, wg))).view(x.shape) if needed[0] else None, *dw,
                 torch.mm(dgate.t(), y[:, n:]) if needed[5] else None, dgate.sum(0) if needed[6] else None,
                 *dconv, *dbias)
        return tuple(g if want else None for g, want in zip(grads, needed)) + (None,)
