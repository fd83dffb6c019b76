"""The native host module (TritonHub/_host.so) against the Python wrappers' general way: the same bits for every form of call
that it takes, and None for what it leaves to them."""
import types

import pytest
import torch

from TritonHub import _native
from TritonHub.Activations import _launch as act_launch
from TritonHub.Layers import Dropout
from TritonHub.Layers import dropout as dropout_layer
from TritonHub.Normalization import _launch as norm_launch


class _General:
    """Stands in for the host module: everything goes the general way."""

    def __getattr__(self, name):
        return lambda *args: None


def test_host_tensors_and_wrong_argument_counts():
    host, x = _native.host(), torch.randn(4, 8)
    assert host.norm_fwd(x, None, None, 1e-5, True, -1, 0) is None
    assert host.norm_bwd(x, x, None, None, None, x, False, -1, True, True) is None
    assert host.softmax_fwd(x, 0) is None and host.softmax_bwd(x, x, 0) is None
    assert host.act_fwd(x, 0, 0.0, 0.0) is None and host.act_bwd(x, x, 0, 0.0, 0.0) is None
    assert host.softmax_fwd(None, 0) is None and host.softmax_fwd("x", 0) is None
    for name, count in (("norm_fwd", 7), ("norm_bwd", 10), ("softmax_fwd", 2), ("softmax_bwd", 3), ("act_fwd", 4), ("act_bwd", 5)):
        with pytest.raises(TypeError):
            getattr(host, name)(*[x] * (count - 1))


def test_dropout_refusals():
    host, x = _native.host(), torch.randn(4, 8)
    assert host.dropout_fwd(x, 0.5, 1, True) is None and host.dropout_bwd(x, 0.5, 1, None) is None
    for count in (3, 5):
        for name in ("dropout_fwd", "dropout_bwd"):
            with pytest.raises(TypeError):
                getattr(host, name)(*[x] * count)


@pytest.fixture
def dropout_calls(monkeypatch):
    """Dropout over a host module that only notes what it is asked for, for tensors of four elements and more; the "mask" is
    the tensor 7."""
    calls = types.SimpleNamespace(keep=[], masks=[], gradients=[], capturing=False)

    class Host:
        def dropout_fwd(self, x, p, seed, keep):
            calls.keep.append(keep)
            return x.clone(), torch.tensor(7) if keep else None

        def dropout_bwd(self, g, p, seed, mask):
            calls.masks.append(mask)
            calls.gradients.append(g)
            return g.clone()

    monkeypatch.setattr(_native, "host", lambda: Host())
    monkeypatch.setattr(dropout_layer, "KEEP_FROM", 4)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: calls.capturing)
    return calls


def test_dropout_keeps_decisions_only_for_a_backward(dropout_calls):
    """Not under no_grad or in inference mode, nor in the first forward of a reentrant checkpoint, whatever the input says."""
    from torch.utils.checkpoint import checkpoint
    module, x = Dropout(0.5), torch.ones(4, requires_grad=True)
    with torch.no_grad():
        assert module(x).grad_fn is None
    with torch.inference_mode():
        module(x)
    module(x.detach())
    module(x[:3])
    assert dropout_calls.keep == [False] * 4
    assert module(x).grad_fn.mask is not None and module(x * 2).grad_fn.mask is not None
    assert dropout_calls.keep[4:] == [True, True]
    checkpoint(lambda t: module(t) * t, x, use_reentrant=True).sum().backward()
    assert dropout_calls.keep[6:] == [False, True] and len(dropout_calls.masks) == 1 and dropout_calls.masks[0] is not None


def test_dropout_gives_its_decisions_back(dropout_calls):
    """The first backward reads them and lets them go, although the graph (here through y) lives on; the second draws."""
    x = torch.ones(4, requires_grad=True)
    y = Dropout(0.5)(x)
    assert y.grad_fn.mask is not None
    y.backward(torch.ones(4))
    assert y.grad_fn.mask is None
    y.backward(torch.ones(4))
    assert [m is None for m in dropout_calls.masks] == [False, True]


def test_dropout_reads_its_decisions_for_any_gradient(dropout_calls):
    """The expanded gradient of a sum and a strided one meet the mask as a contiguous copy; without a mask they are passed on."""
    for backward in (lambda y: y.sum().backward(), lambda y: y.backward(torch.ones(4, 2)[:, 0])):
        backward(Dropout(0.5)(torch.ones(4, requires_grad=True)))
        assert dropout_calls.masks[-1] is not None and dropout_calls.gradients[-1].is_contiguous()
    Dropout(0.5)(torch.ones(3, requires_grad=True)).sum().backward()
    assert dropout_calls.masks[-1] is None and not dropout_calls.gradients[-1].is_contiguous()


@pytest.mark.parametrize("forward_captured", [False, True])
@pytest.mark.parametrize("backward_captured", [False, True])
def test_dropout_decisions_do_not_cross_the_border_of_a_graph(dropout_calls, forward_captured, backward_captured):
    """A backward captured after an eager forward draws: the decisions of that forward are gone when the graph is replayed.
    Captured both, they live in the graph's memory."""
    dropout_calls.capturing = forward_captured
    y = Dropout(0.5)(torch.ones(4, requires_grad=True))
    dropout_calls.capturing = backward_captured
    y.backward(torch.ones(4))
    assert (dropout_calls.masks[-1] is not None) == (forward_captured == backward_captured)


def _same(a, b):
    if a is None or b is None:
        return a is None and b is None
    return a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride() and torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16, torch.float64])
@pytest.mark.parametrize("shape", [(1,), (7,), (3, 1, 5), (2, 100, 128), (65, 4098)])
def test_same_bits_as_the_general_way(shape, dtype, monkeypatch):
    host, n = _native.host(), shape[-1]
    g = torch.Generator(device="cuda").manual_seed(n)
    x, dy = (torch.randn(*shape, device="cuda", generator=g).to(dtype) for _ in range(2))
    w, b = (torch.randn(n, device="cuda", generator=g).to(dtype) for _ in range(2))
    w32 = w.float()

    def norms(act):
        for layernorm in (True, False):
            for weight, bias in ((w, b), (w, None), (None, None), (w32, None), (None, b), (w32, b)):
                if bias is not None and not layernorm:
                    continue
                y, mean, rstd = norm_launch.norm_fwd(x, weight, bias, 1e-5, layernorm, act)
                yield from (y, mean, rstd)
                for need_dw, need_db in ((True, True), (False, True), (True, False), (False, False)):
                    yield from norm_launch.norm_bwd(x, dy, weight, bias, mean, rstd, layernorm, act, need_dw, need_db)

    def everything():
        yield from norms(-1)
        yield from norms(_native.ACT_SILU)
        for kind in (_native.SOFTMAX, _native.SOFTMIN, _native.LOGSOFTMAX):
            y = act_launch.softmax_fwd(x, kind)
            yield from (y, act_launch.softmax_bwd(y, dy, kind))
        for act, p0, p1 in ((_native.ACT_GELU, 0.0, 0.0), (_native.ACT_LEAKY_RELU, 0.1, 0.0), (_native.ACT_THRESHOLD, 0.2, -1)):
            yield from (act_launch.act_fwd(x, act, p0, p1), act_launch.act_bwd(x, dy, act, p0, p1))

    here = list(everything())
    monkeypatch.setattr(_native, "host", lambda: _General())
    general = list(everything())
    assert len(here) == len(general) and all(_same(a, c) for a, c in zip(here, general))
    # what it takes, and what it leaves to the wrappers
    assert host.norm_fwd(x, w, b, 1e-5, True, -1, 0) is not None and host.softmax_fwd(x, 0) is not None
    assert host.norm_fwd(x, w32, b, 1e-5, True, -1, 0) is None or dtype == torch.float32
    rstd = torch.ones(x.numel() // n, device="cuda")
    assert host.norm_bwd(x, dy.double() if dtype != torch.float64 else dy.float(), w, None, None, rstd, False, -1, True, True) is None
    assert host.norm_bwd(x, dy, w, None, None, rstd.double(), False, -1, True, True) is None
    assert host.norm_fwd(x, torch.ones(n + 1, device="cuda", dtype=dtype), None, 1e-5, True, -1, 0) is None
    assert host.softmax_fwd(x[..., :0], 0) is None and host.softmax_fwd(x.expand(2, *shape), 0) is None
    assert host.softmax_fwd(torch.ones(4, 4, device="cuda", dtype=torch.int32), 0) is None
    assert host.softmax_bwd(x, dy.reshape(-1, 1), 0) is None or n == 1
    with pytest.raises(RuntimeError, match="libthnorm"):
        host.softmax_fwd(x, 9)


@pytest.mark.gpu
def test_dropout_results_have_contiguous_strides(monkeypatch):
    """Also where a dimension of one element of the input or the gradient has a stride of its own, as the general way does."""
    def strides():
        x, dy = (torch.randn(2, 1, 3, 8, device="cuda").as_strided((2, 1, 3, 8), (24, 7, 8, 1)) for _ in range(2))
        y = Dropout(0.5)(x.requires_grad_(True))
        return y.stride(), torch.autograd.grad(y, x, dy)[0].stride()

    here = strides()
    monkeypatch.setattr(_native, "host", lambda: _General())
    assert here == strides() == ((24, 24, 8, 1),) * 2


@pytest.mark.gpu
def test_dropout_forms_left_to_the_wrapper():
    """A mask of another size, type or place, a probability or a seed that is no plain number, rows apart."""
    host, n = _native.host(), 1 << 13          # two pieces of 1024 vectors in float32, one in 16 bits
    x = torch.randn(n, device="cuda")
    out, mask = host.dropout_fwd(x, 0.5, 1, True)
    assert host.dropout_bwd(x, 0.5, 1, mask) is not None and host.dropout_bwd(x, 0.5, 1, None) is not None
    for other in (mask[:-1], torch.cat((mask, mask)), mask.float(), mask.cpu(), mask.repeat(2)[::2], "mask"):
        assert host.dropout_bwd(x, 0.5, 1, other) is None
    assert host.dropout_bwd(x.bfloat16(), 0.5, 1, mask) is None          # half the pieces: half the mask
    for p, seed in ((0.0, 1), (1.0, 1), (1.0 - 1e-12, 1), (float("nan"), 1), ("0.5", 1), (0.5, 1.0), (0.5, 1 << 70)):
        assert host.dropout_fwd(x, p, seed, False) is None and host.dropout_bwd(x, p, seed, None) is None, (p, seed)
    for t in (x[::2], x[:0], x.int()):
        assert host.dropout_fwd(t, 0.5, 1, False) is None and host.dropout_bwd(t, 0.5, 1, None) is None


@pytest.mark.gpu
@pytest.mark.parametrize("side_stream", [False, True])
@pytest.mark.parametrize("dtype,param", [(torch.float16, torch.bfloat16), (torch.bfloat16, torch.float16), (torch.float32, torch.float64)])
def test_other_parameter_types_streams_and_gradients(dtype, param, side_stream, monkeypatch):
    """Parameters of another type than the input, the calls on a stream of their own with work in front of them, gradients
    that are not contiguous (which the wrappers take): the same bits as the general way."""
    rows, n = 300, 1000
    g = torch.Generator(device="cuda").manual_seed(n)
    x, dy = (torch.randn(rows, n, device="cuda", generator=g).to(dtype) for _ in range(2))
    w, b = (torch.randn(n, device="cuda", generator=g).to(param) for _ in range(2))
    gradients = (dy, dy.t().contiguous().t(), torch.stack((dy, dy), -1)[..., 0], dy[:1].expand(rows, n))
    assert _native.host().norm_fwd(x, w, b, 1e-5, True, -1, 0) is not None

    def everything():
        for layernorm, bias in ((True, b), (False, None)):
            y, mean, rstd = norm_launch.norm_fwd(x, w, bias, 1e-5, layernorm)
            yield from (y, mean, rstd)
            for grad in gradients:
                yield from norm_launch.norm_bwd(x, grad, w, bias, mean, rstd, layernorm)
        y = act_launch.softmax_fwd(x, _native.SOFTMAX)
        yield y
        for grad in gradients:
            yield act_launch.softmax_bwd(y, grad, _native.SOFTMAX)
            yield act_launch.act_bwd(x, grad, _native.ACT_GELU)

    def on_a_stream():
        stream = torch.cuda.Stream() if side_stream else torch.cuda.current_stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            busy = torch.ones(1 << 24, device="cuda")
            for _ in range(4):
                busy = busy * 1.5
            results = list(everything())
        stream.synchronize()
        return results

    here = on_a_stream()
    monkeypatch.setattr(_native, "host", lambda: _General())
    general = on_a_stream()
    assert len(here) == len(general) and all(_same(a, c) for a, c in zip(here, general))
