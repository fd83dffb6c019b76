"""Dropout: drop-in for ``TritonHub/Layers/dropout.py`` of the reference -- the ``dropout`` autograd Function
(dropout.py:95-111) and the ``Dropout`` module (:113-119).

The mask is the reference's: element i of the flattened tensor is dropped when Triton's ``tl.rand(seed, i) < p``
(dropout.py:20-21), and the HIP kernel evaluates the same Philox-4x32-10 stream.  The seed is drawn as the reference
draws it, ``random.randint(0, 2**16)`` from Python's ``random`` module once per forward call (dropout.py:98), so a
program that seeds ``random`` sees the same masks with either library.
"""
import random

import torch

from .. import _native
from .._autograd import PYTHON, native_apply
from ..Activations._launch import _call


def _dropout_apply(t: torch.Tensor, p, seed, training, what: str) -> torch.Tensor:
    """Forward and backward are the same function of their tensor (dropout.py:25-50, :69-94)."""
    if not t.is_cuda:
        _native.require_gpu(t)
    if t.stride(-1) != 1:
        t = t.contiguous()
    assert t.stride(-1) == 1 or t.numel() == 0, 'expect input to be row-major'     # (empty: any strides)
    if (p == 0.0) or (not training):
        return t
    if p == 1.0:
        return torch.zeros_like(t, memory_format=torch.contiguous_format)
    flat = t.reshape(-1)                      # a copy when the tensor is not contiguous, as in the reference
    out = torch.empty_like(flat, memory_format=torch.contiguous_format)
    assert out.shape == flat.shape, 'expect output shape to be the same as input shape'
    assert out.stride(-1) == 1, 'expect output to be row-major'
    if flat.numel() > 0:
        _call(t.device, 'thn_dropout', flat.data_ptr(), out.data_ptr(), flat.numel(), 0, float(p), int(seed),
              _native.dtype_code(t.dtype))
    return out.reshape(t.shape)


# From this many elements on a dropout that will be differentiated keeps its decisions instead of drawing them again in the
# backward.  Below it the kernels take less time than the host needs for the extra tensor.
KEEP_FROM = 1 << 22


class dropout(torch.autograd.Function):
    """forward(ctx, input, p, training) -> output; keeps (p, seed, training) on ctx.  The forward of a large input also keeps
    there which elements were dropped (``mask``, one byte per 16 bytes of input) if a backward can follow, which reads them and
    gives them back; every other backward, a second one among them, regenerates the mask from the seed.  The two give the
    same bits.  The mask is no saved tensor, as the seed is none, so a graph can be walked again without retain_graph; under
    saved-tensor hooks, which would not see it, and so in a non-reentrant checkpoint, none is kept."""

    apply = native_apply(PYTHON)

    @staticmethod
    def forward(ctx, input, p, training):
        seed = random.randint(0, 2**16)
        ctx.p = p
        ctx.seed = seed
        ctx.training = training
        ctx.mask = None
        # needs_input_grad says that the input requires a gradient, also where gradients are off (no_grad, inference mode, the
        # first forward of a reentrant checkpoint): only a node with somewhere to pass a gradient on to has a backward
        keep = ctx.needs_input_grad[0] and input.numel() >= KEEP_FROM and len(ctx.next_functions) > 0
        done = _native.host().dropout_fwd(input, p, seed, keep) if training else None
        if done is None:
            return _dropout_apply(input, p, seed, training, 'input')
        output, ctx.mask = done
        if keep:
            ctx.captured = torch.cuda.is_current_stream_capturing()
        return output

    @staticmethod
    def backward(ctx, d_out):
        if ctx.training:
            mask, ctx.mask = ctx.mask, None          # given back as saved tensors are; another backward draws the same bits
            if mask is not None and ctx.captured != torch.cuda.is_current_stream_capturing():
                mask = None          # a captured backward would read it on every replay, long after it has been freed
            if mask is not None:
                d_out = d_out.contiguous()           # an expanded gradient, say (the general way copies it too)
            grad = _native.host().dropout_bwd(d_out, ctx.p, ctx.seed, mask)
            if grad is not None:
                return grad, None, None
        grad = _dropout_apply(d_out, ctx.p, ctx.seed, ctx.training, 'gradient')
        return grad, None, None


class Dropout(torch.nn.Module):
    """Dropout(p=0.5): zeroes each element with probability p while training and scales the rest by 1 / (1 - p)."""

    def __init__(self, p=0.5):
        super().__init__()
        self.p = p
        self.dropout_fn = dropout.apply

    def forward(self, x):
        return self.dropout_fn(x, self.p, self.training)
