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


def rows_16(x):
    """x itself where it is contiguous and 16-byte aligned, else a copy that is
    (made before a function's ``apply``, so that it is part of the graph)."""
    x = x.contiguous()
    return x.clone() if x.data_ptr() % 16 else x


def _recorded_grads(fn, inputs, needed, dy):
    """Gradients of fn(*inputs), recorded for further derivatives."""
    with torch.enable_grad():
        wanted = [t for t, n in zip(inputs, needed) if n]
        grads = iter(torch.autograd.grad(fn(*inputs), wanted, dy, create_graph=True, allow_unused=True))
    return tuple(next(grads) if n else None for n in needed)


def short_conv(x, weight, bias, cache, general):
    """The causal depthwise convolution (layers/cyfa.py:138-233) with its HIP
    adjoint: x [B, T, D], weight [D, W], bias [D] or None, cache [B, W-1, D] or
    None, all of one dtype (bf16 or fp32). ``general``: the same in torch
    operations."""
    return ShortConv.apply(rows_16(x), weight.contiguous(), bias, None if cache is None else rows_16(cache), general)


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
        if torch.is_grad_enabled():
            return _recorded_grads(ctx.general, (x, weight, bias, cache), needed, dy) + (None,)
        grads = _native.short_conv_grad(x, weight, cache, rows_16(dy), needed)
        return (*grads, None)


def rms_norm(x, weight, gate, eps, prescale, general):
    """norm(x prescale) [* sigmoid(gate)] (layers/cyfa.py:62-135) with its HIP
    adjoint: x and gate [..., D] bf16 or fp32 of one dtype, weight fp32 [D].
    ``general``: the same of (x, weight, gate) in torch operations."""
    return GatedNorm.apply(rows_16(x), rows_16(weight), None if gate is None else rows_16(gate), eps, prescale, general)


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
        if torch.is_grad_enabled():
            return _recorded_grads(ctx.general, (x, weight, gate), needed, dy) + (None,) * 3
        return (*_native.norm_grad(x, weight, gate, *ctx.args, rows_16(dy), needed), None, None, None)
