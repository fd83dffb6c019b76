"""The GeLU epilogues that go by a table (thn_gelu_table.h), at every node and every edge between two of its intervals, beyond its ends and
at values that are not finite.  A weight of 0 makes the pre-activation the bias itself, so a column holds one argument: the
output is GeLU of it and, with an upstream gradient of 1, dB is rows * GeLU'(b)."""
import numpy as np
import pytest
import torch
from scipy.special import log_ndtr

from test_fused_parity_gpu import announce, make, run_and_compare
from TritonHub.Normalization.fused import LayerNormActivation

pytestmark = pytest.mark.gpu
ULP = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 2.0 ** -23}            # spacing over value, at most
LEAST = {torch.bfloat16: 2.0 ** -133, torch.float16: 2.0 ** -24, torch.float32: 2.0 ** -149}       # the smallest subnormal


def arguments(n, dtype):
    """n values from -15 to 7 in steps of at most 1/64, as the type holds them, in an order that mixes them."""
    values = (torch.arange(n, dtype=torch.float64) * 22.0 / (n - 1) - 15.0) if n > 1409 else torch.arange(n, dtype=torch.float64) / 64 - 15.0
    return values[torch.randperm(n, generator=torch.Generator().manual_seed(n))].to(dtype)


def at_bias(b, rows, dtype):
    n = b.numel()
    module = LayerNormActivation(n, "gelu", device="cuda", dtype=dtype)
    with torch.no_grad():
        module.weight.zero_()
        module.bias.copy_(b)
    x = torch.randn(rows, n, generator=torch.Generator().manual_seed(1)).to(dtype).cuda().requires_grad_(True)
    y = module(x)
    y.backward(torch.ones_like(y))
    return y.detach(), module.bias.grad


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n", [1408, 1409, 4096, 8200, 16384])
def test_every_interval(n, dtype):
    rows = 64
    announce(f"GeLU table {dtype} {rows} x {n}")
    b = arguments(n, dtype)
    y, db = at_bias(b, rows, dtype)
    z = b.double().numpy()
    cdf, pdf = np.exp(log_ndtr(z)), np.exp(-0.5 * z * z) / np.sqrt(2.0 * np.pi)
    assert bool((y == y[0]).all())
    # the cubics: 3.1e-10*z^4 of their own (below -12 outputs are 1e-31 and less), and three roundings of at most the size of the result: the
    # constant coefficient, the product with the distance and the sum.  float32 forwards and 1024-thread backwards off the 128-bit path
    # go by the polynomial.
    fit = 3.0 * 2.0 ** -24 + 3.2e-10 * z ** 4
    outputs = ((y[0], z * cdf, np.abs(z) * cdf), (db / rows, cdf + z * pdf, cdf + np.abs(z) * pdf))
    for got, want, size in outputs if dtype != torch.float32 else outputs[1:]:
        error = np.abs(got.double().cpu().numpy() - want)
        bound = size * (fit + 0.5 * ULP[dtype]) + LEAST[dtype] + 1e-30
        assert (error <= bound).all(), (float((error / bound).max()), z[np.argmax(error / bound)])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n", [1024, 1111, 2047])
def test_values_beyond_the_ends(n, dtype):
    announce(f"GeLU table beyond its ends {dtype} {n}")
    most = torch.finfo(dtype).max
    special = [float("nan"), float("inf"), -float("inf"), most, -most, 0.0, -0.0, 6.0, -14.0, 20.0, -20.0]
    b = torch.zeros(n, dtype=dtype)
    b[:len(special)] = torch.tensor(special, dtype=torch.float64).to(dtype)
    y, db = at_bias(b, 8, dtype)
    want = [float("nan"), float("inf"), float("nan"), most, 0.0, 0.0, 0.0, 6.0, 0.0, 20.0, 0.0]
    assert torch.allclose(y[0, :len(want)].double().cpu(), torch.tensor(want, dtype=torch.float64), atol=1e-30, equal_nan=True)
    # the reference's x*phi(x) is inf*0 at the infinities
    slopes = [float("nan"), float("nan"), float("nan"), 8.0, 0.0, 4.0, 4.0, 8.0, 0.0, 8.0, 0.0]
    assert torch.allclose(db[:len(want)].double().cpu(), torch.tensor(slopes, dtype=torch.float64), rtol=1e-6, atol=1e-30, equal_nan=True)
    assert bool((y[:, len(want):] == 0).all()) and bool((db[len(want):] == 4).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,n", [(700, 40), (600, 250), (600, 256), (300, 1024), (90, 4099), (40, 12301), (40, 16384), (20, 17001), (20, 32768)])
def test_wide_pre_activations(rows, n, dtype):
    if n * torch.empty(0, dtype=dtype).element_size() > 65536:
        pytest.skip("wider than 64 KiB")
    announce(f"GeLU table, wide pre-activations {dtype} {rows} x {n}")
    x, dy, w, b = make((rows, n), dtype, seed=n)
    wide = 1 if dtype == torch.float32 else 6          # the float32 bar, 1e-5, is that of pre-activations of a few units
    run_and_compare("ln", "gelu", x, dy, w * wide, b * wide, 1e-5, f"ln+gelu {rows} x {n}")
    run_and_compare("rms", "gelu", x, dy, w * wide, None, 1e-5, f"rms+gelu {rows} x {n}")
