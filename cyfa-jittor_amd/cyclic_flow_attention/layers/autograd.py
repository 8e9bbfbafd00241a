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
    compiling, autocast)."""
    given = [t for t in tensors if t is not None]
    if not all(type(t) in (torch.Tensor, torch.nn.Parameter) and t.is_cuda for t in given):
        return False
    if any(t.device != given[0].device for t in given):
        return False
    return (torch.is_grad_enabled() and not torch.is_autocast_enabled("cuda")
            and torch._C._functorch.peek_interpreter_stack() is None and forward_ad._current_level < 0
            and not torch.compiler.is_compiling() and not torch.jit.is_tracing())


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
