"""Every autograd Function that is made natively (csrc/thn_host.cpp) against the same Function with its Python forward and backward.  A
subclass of a Function has torch's own apply and the Python methods, so it is the other side: the two must agree in every bit, saved
tensor, attribute and error."""
import importlib
import random

import pytest
import torch

from TritonHub import _native

pytestmark = pytest.mark.gpu

W, B = object(), object()                                                   # places of a weight and a bias


def function(module, name):
    return getattr(importlib.import_module(module), name)


ACTS, NORMS, OPS = "TritonHub.Activations.", "TritonHub.Normalization.", "TritonHub.Ops."
CASES = {
    "layernorm": (NORMS + "layernorm", "layernorm", (W, B, 1e-5)), "layernorm no bias": (NORMS + "layernorm", "layernorm", (W, None, 1e-5)),
    "rmsnorm": (NORMS + "rmsnorm", "rmsnorm", (W, 1e-5)), "layernorm + gelu": (NORMS + "fused", "layernorm_act", (W, B, 1e-5, _native.ACT_GELU)),
    "rmsnorm + silu": (NORMS + "fused", "rmsnorm_act", (W, 1e-5, _native.ACT_SILU)), "softmax": (ACTS + "softmax", "softmax", ()),
    "logsoftmax": (ACTS + "logsoftmax", "logsoftmax", ()), "softmin": (ACTS + "softmin", "softmin", ()), "softmin of": (ACTS + "softmin", "_softmin_of", ()),
    "gelu": (ACTS + "gelu", "gelu", ("none",)), "gelu tanh": (ACTS + "gelu", "gelu", ("tanh",)), "silu": (ACTS + "silu", "silu", ()),
    "relu": (ACTS + "relu", "relu", ()), "relu6": (ACTS + "relu6", "relu6", ()), "leaky relu": (ACTS + "leaky_relu", "leakyrelu", (0.2,)),
    "sigmoid": (ACTS + "sigmoid", "sigmoid", ()), "tanh": (ACTS + "tanh", "tanh", ()), "mish": (ACTS + "mish", "mish", ()),
    "softplus": (ACTS + "softplus", "softplus", (2.0, 5.0)), "threshold": (ACTS + "threshold", "threshold_fn", (0.1, -3.0)),
    "norm": (OPS + "norm", "Norm", ()), "norm 3": (OPS + "norm", "Norm", (3, 1e-4)), "normalize": (OPS + "normalize", "Normalize", (2,)),
    "normalize 1": (OPS + "normalize", "Normalize", (1, 1e-3)), "dropout": ("TritonHub.Layers.dropout", "dropout", (0.4, True)),
}


def make_input(form):
    torch.manual_seed(7)
    x = torch.randn(3, 10, 68, device="cuda")
    if form == "bf16": x = x.bfloat16()
    if form == "f64": x = x.double()
    if form == "int": x = x.to(torch.int32)
    if form == "strided": x = x.transpose(0, 1)
    if form == "empty": x = x[:, :0]
    if form == "4d": x = x.view(3, 2, 5, 68)
    return x


def observed(apply, args, form, grads):
    """Everything that a caller can see of one forward and backward; an error as its type and text."""
    random.seed(5)
    x = make_input(form)
    x = x.requires_grad_(grads and x.is_floating_point())
    w, b = (torch.linspace(-1, 2, 68, device="cuda", dtype=x.dtype if x.is_floating_point() else torch.float32).requires_grad_(grads) for _ in range(2))
    try:
        arguments = [x, *[w if a is W else b if a is B else a for a in args]]
        y = apply(*arguments)
        seen = [y, y.requires_grad, y.stride()]
        if y.grad_fn is not None:
            node = y.grad_fn
            seen += [len(node.saved_tensors), *node.saved_tensors, node.needs_input_grad, sorted((k, repr(v)) for k, v in vars(node).items())]
            dy = torch.linspace(-1, 1, y.numel(), device="cuda").to(y.dtype).view(y.shape)
            inputs = [a for a in arguments if isinstance(a, torch.Tensor)]
            seen += torch.autograd.grad(y, inputs, dy, retain_graph=True)
            seen += torch.autograd.grad(y, inputs, dy.transpose(0, -1).contiguous().transpose(0, -1))         # not contiguous
            try:
                torch.autograd.grad(y, inputs, dy)
            except RuntimeError as error:
                seen.append(str(error)[:80])
        return seen
    except Exception as error:
        return [type(error).__name__, str(error)]


@pytest.mark.parametrize("name", CASES)
def test_the_same_as_in_python(name):
    module, cls, args = CASES[name]
    native = function(module, cls)
    general = type(native)(native.__name__, (native,), {})
    for form in ("f32", "bf16", "f64", "strided", "empty", "4d", "int"):
        for grads in (True, False):
            print(f"{name} {form} grads={grads}", flush=True)
            got, want = observed(native.apply, args, form, grads), observed(general.apply, args, form, grads)
            assert len(got) == len(want), (form, grads, got, want)
            for i, (a, b) in enumerate(zip(got, want)):
                if isinstance(b, torch.Tensor):
                    assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride() and torch.equal(a, b), (form, grads, i)
                else:
                    assert a == b, (form, grads, i, a, b)


@pytest.mark.parametrize("name", CASES)
def test_without_a_graph(name):
    """No gradient can follow: no context is made."""
    module, cls, args = CASES[name]
    native = function(module, cls)
    general = type(native)(native.__name__, (native,), {})
    for mode in (torch.no_grad, torch.inference_mode):
        with mode():
            got, want = observed(native.apply, args, "bf16", True), observed(general.apply, args, "bf16", True)
        assert torch.equal(got[0], want[0]) and got[1:] == want[1:] and got[0].is_inference() == want[0].is_inference(), mode


def test_the_cache_policy_is_read_at_each_call(monkeypatch):
    from TritonHub.Normalization import _launch
    seen = []
    for policy in ("auto", "keep", "stream"):
        monkeypatch.setattr(_launch, "_cache_policy", policy)
        seen.append(observed(function(NORMS + "layernorm", "layernorm").apply, (W, B, 1e-5), "bf16", True))
    for other in seen[1:]:
        assert all(torch.equal(a, b) for a, b in zip(seen[0], other) if isinstance(a, torch.Tensor))


@pytest.mark.parametrize("form", ["f32", "strided"])
@pytest.mark.parametrize("name", CASES)
def test_saved_tensors_are_read_once(name, form):
    """A non-reentrant checkpoint's hooks refuse a second reading, whichever way the backward of this input goes."""
    from torch.utils.checkpoint import checkpoint
    module, cls, args = CASES[name]
    apply = function(module, cls).apply
    print(f"{name} {form}", flush=True)
    w, b = (torch.linspace(-1, 2, 68, device="cuda") for _ in range(2))
    arguments = [w if a is W else b if a is B else a for a in args]
    gradients = []
    for run in (lambda t: apply(t, *arguments), lambda t: checkpoint(lambda u: apply(u, *arguments), t, use_reentrant=False)):
        random.seed(5)
        x = make_input(form).requires_grad_(True)
        y = run(x)
        random.seed(5)
        gradients += torch.autograd.grad(y, x, torch.linspace(-1, 1, y.numel(), device="cuda").view(y.shape))
    assert torch.equal(*gradients)
    read = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: read.append(t) or t):
        random.seed(5)
        y = apply(make_input(form).requires_grad_(True), *arguments)
    held = sum(t is not None for t in y.grad_fn.saved_tensors)
    read.clear()
    y.backward(torch.ones_like(y))
    assert len(read) == held
