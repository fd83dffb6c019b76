"""The autograd Functions without Python frames for ordinary tensors (csrc/thn_host.cpp, "The autograd Functions").

A Function is written as usual, with ``forward`` and ``backward`` in Python, which make every form of call.  An ``apply``
of this module's in its class body adds the native way::

    class silu(torch.autograd.Function):
        apply = native_apply(ACT, _native.ACT_SILU)

The node in the graph is the one that torch makes of the Function either way: same context class, same saved tensors,
attributes and hooks.  Transforms (functorch), keyword arguments and subclasses of a Function go through
``torch.autograd.Function.apply`` as ever.
"""
import torch

from . import _native

LAYERNORM, RMSNORM, SOFTMAX, ACT, PNORM, NORMALIZE, PYTHON = range(7)       # enum Kind in csrc/thn_host.cpp


class ReadContext:
    """A Function's context whose saved tensors have been read already, for the Python backward to go on with."""
    __slots__ = ("ctx", "saved_tensors")

    def __init__(self, ctx, saved_tensors):
        self.ctx, self.saved_tensors = ctx, saved_tensors

    def __getattr__(self, name):
        return getattr(self.ctx, name)


class native_apply:
    """``kind`` and ``code``: which operator; ``params``: the names under which the context keeps the arguments behind the tensors;
    ``flag``: an activation code follows (norms), the output is saved (activations).  The class attribute is replaced when it is
    first read, so that importing the package loads no library; where the library is missing, the Python forward says so."""

    def __init__(self, kind, code=0, params=(), flag=False):
        self.spec = (kind, code, tuple(params), flag)

    def __set_name__(self, owner, name):
        self.owner = owner

    def __get__(self, instance, cls=None):
        cls = type(instance) if cls is None else cls
        owner = self.owner
        general = super(owner, owner).apply
        try:
            made = _native.host().autograd_function(owner, general, *self.spec)
        except (RuntimeError, AttributeError):
            made = None
        if made is None:
            return super(owner, cls).apply
        capsule, forward, backward, apply = made
        namespace = {'__module__': owner.__module__, '__qualname__': owner.__qualname__, '__doc__': owner.__doc__, 'apply': general}
        if self.spec[0] != PYTHON:
            namespace['forward'] = staticmethod(forward)
        quick = type(owner)(owner.__name__, (owner,), namespace)
        quick._backward_cls = owner._backward_cls          # one class of nodes, whichever way they were made
        owner._backward_cls.apply = backward
        from .Normalization import _launch
        _native.host().autograd_function_ready(capsule, super(torch.autograd.Function, quick).apply, _launch.__dict__, ReadContext)
        owner.apply = classmethod(apply)
        return getattr(cls, 'apply')
