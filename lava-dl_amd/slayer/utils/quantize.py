"""Straight-through parameter quantiser (utils/quantize.py:18-94 in the reference)."""
from enum import IntEnum, unique

import numpy as np
import torch
from torch.autograd import forward_ad

from .. import _native as N


@unique
class MODE(IntEnum):
    ROUND = 0
    FLOOR = 1


# Plain numbers: not tensors or arrays, whose elements differ, may be trained, or lie on the GPU.
_NUMBER = (int, float, np.integer, np.floating)
_FLOAT32_MAX = torch.finfo(torch.float32).max
_STEP_MIN, _STEP_MAX = 2.0 ** -126, 2.0 ** 126                      # steps whose reciprocal is a float32 number too


class _StraightThrough(torch.autograd.Function):
    """Snap to a grid of ``step`` in the forward pass, identity in the backward pass."""

    @staticmethod
    def forward(ctx, input, step, use_floor):
        if isinstance(step, _NUMBER) and step == 1:                          # what follows, without the two products by one
            return torch.floor(input) if use_floor else torch.round(input)
        scaled = input / step
        return (torch.floor(scaled) if use_floor else torch.round(scaled)) * step

    @staticmethod
    def backward(ctx, grad_output):
        return grad_output, None, None


def quantize(input, step=1, mode=MODE.ROUND):
    """Quantise ``input`` to multiples of ``step`` (round or floor); gradients pass through."""
    if mode not in (MODE.ROUND, MODE.FLOOR):
        raise ValueError(f'{mode=} is not recognized.')
    if not (torch.is_grad_enabled() and input.requires_grad):      # nothing to pass a gradient to
        snap = torch.floor if mode == MODE.FLOOR else torch.round
        return snap(input) if isinstance(step, _NUMBER) and step == 1 else snap(input / step) * step
    return _StraightThrough.apply(input, step, mode == MODE.FLOOR)


class _Limited(torch.autograd.Function):
    """limit() in one launch each way (slayer_quantize)."""

    @staticmethod
    def forward(ctx, input, step, lo, hi, scale):
        inside = torch.empty(input.shape, dtype=torch.bool, device=input.device)
        ctx.save_for_backward(inside)
        ctx.scale = scale
        return _launch(input, step, lo, hi, scale, inside)

    @staticmethod
    def backward(ctx, grad_output):
        inside, = ctx.saved_tensors
        if torch.is_grad_enabled() or not takes_kernel(grad_output, contiguous=False):      # create_graph=True, batched gradients
            return torch.where(inside, grad_output * ctx.scale, 0.0), None, None, None, None
        grad_output = grad_output.contiguous()
        grad = torch.empty_like(grad_output)
        with N.device_guard(grad.device):
            N.check(N.lib().slayer_quantize_bwd(N.ptr(grad), N.ptr(grad_output), N.ptr(inside), ctx.scale, grad.numel(),
                                                N.stream_handle()))
        return grad, None, None, None, None


def _launch(input, step, lo, hi, scale, inside):
    out = torch.empty_like(input)
    with N.device_guard(out.device):
        N.check(N.lib().slayer_quantize(N.ptr(out), N.ptr(inside), N.ptr(input), step, lo, hi, scale, out.numel(),
                                        N.stream_handle()))
    return out


def takes_kernel(input, contiguous=True):
    """float32 weights on the GPU as they lie in memory, and nobody who wants to see the single operations: tracing,
    compilation, dispatch modes (make_fx), function transforms (those of ``is_grads_batched`` too, whose tensors have no
    memory of their own), forward-mode differentiation."""
    return (type(input) in (torch.Tensor, torch.nn.Parameter) and input.is_cuda and input.dtype == torch.float32
            and not torch.jit.is_tracing() and not torch.compiler.is_compiling()
            and torch._C._len_torch_dispatch_stack() == 0
            and torch._C._functorch.peek_interpreter_stack() is None and forward_ad._current_level < 0
            and not torch._C._functorch.is_legacy_batchedtensor(input)
            and (not contiguous or input.is_contiguous()))


def _fits_kernel(step, lo, hi, scale):
    """Plain numbers inside the range of float32."""
    return (isinstance(step, _NUMBER) and isinstance(lo, _NUMBER) and isinstance(hi, _NUMBER) and isinstance(scale, _NUMBER)
            and _STEP_MIN <= abs(step) <= _STEP_MAX and -_FLOAT32_MAX <= lo <= _FLOAT32_MAX
            and -_FLOAT32_MAX <= hi <= _FLOAT32_MAX and -_FLOAT32_MAX <= scale <= _FLOAT32_MAX)


def limit(input, step, lo, hi, scale=1):
    """``quantize(input, step).clamp(lo, hi) * scale``.  A step, a limit or a scale may be a tensor (one per channel, or one that is
    trained); those take the operators."""
    if not (takes_kernel(input) and _fits_kernel(step, lo, hi, scale)):
        q = quantize(input, step=step).clamp(lo, hi)
        return q if isinstance(scale, _NUMBER) and scale == 1 else q * scale
    if torch.is_grad_enabled() and input.requires_grad:
        return _Limited.apply(input, float(step), float(lo), float(hi), float(scale))
    return _launch(input, float(step), float(lo), float(hi), float(scale), None)


def quantize_hook_fx(x, scale=1 << 6, num_bits=8, descale=False):
    """Synapse pre-hook quantiser (utils/quantize.py:84-115 in the reference): even multiples of
    1 / scale, limited to the signed ``num_bits`` weight range; ``descale`` returns integers."""
    lo = -2 * (1 << num_bits) / scale
    hi = 2 * ((1 << num_bits) - 1) / scale
    return limit(x, 2 / scale, lo, hi, scale if descale else 1)
