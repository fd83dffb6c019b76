"""Softmax family over few rows of more than 64 KiB, cut into slices of one workgroup each (thn_softmax_sliced.h): against the oracle
at the edges of slices and rows, the rows and columns around them, and the rule that chooses these kernels."""
import pytest
import torch

from oracle import softmax_oracle as so
from test_output_guards_gpu import PADS, check_guards, padded
from test_softmax_parity_gpu import CODE, KINDS, MODULE, announce, make, run_and_compare
from TritonHub import _native
from TritonHub.Activations import _launch
from TritonHub.Normalization._launch import query_launch

pytestmark = pytest.mark.gpu
DTYPES = [torch.float32, torch.bfloat16, torch.float16]
SLICE = 2048                     # 16-byte vectors


def vec_of(dtype):
    return 16 // torch.empty((), dtype=dtype).element_size()


@pytest.fixture
def sliced():
    lib = _native.lib()
    for which in (2, 3):
        assert lib.thn_norm_set_launch_override(which, 4, 512, 0, 0) == 0
    yield
    for which in (2, 3):
        lib.thn_norm_set_launch_override(which, 0, 0, 0, 0)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("kind", KINDS)
def test_edges_of_slices_and_rows(kind, dtype, sliced):
    """Rows of whole slices and a vector more, of every number of elements behind the last vector, whose starts go through the
    offsets from a 16-byte boundary (an odd width), and the widest ones."""
    vec, log = vec_of(dtype), kind == "logsoftmax"
    for rows, n in ((3, 4096 * vec + 1), (vec + 1, 3 * SLICE * vec - 1), (2, 3 * SLICE * vec), (2, 3 * SLICE * vec + vec), (vec + 1, 3 * SLICE * vec + vec + vec // 2 + 1),
                    (1, 64 * SLICE * vec), (2, 64 * SLICE * vec - 1), (70, 4096 * vec + vec - 1)):
        slices = -(-(n // vec) // SLICE)
        for which in (2, 3):
            assert query_launch(which, log, rows, n, dtype)[:4] == (4, 512, 512, rows * slices), n
        announce(f"slices {kind} {dtype} {rows} x {n}")
        x, dy = make((rows, n), dtype, seed=n, scale=3.0)
        run_and_compare(kind, x, dy, f"{kind} {rows} x {n}")
    assert query_launch(2, log, 2, 64 * SLICE * vec + vec, dtype)[1] != 512             # a lane of a wave per slice, no more


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("kind", ["softmax", "logsoftmax"])
def test_slices_without_a_finite_value(kind, dtype, sliced):
    """-inf in whole slices and in everything but one edge element, rows of -inf alone, a NaN or +inf in one slice: what the kernels with
    a workgroup per row give, and no other row is touched."""
    n = 3 * SLICE * vec_of(dtype) + 5
    x = torch.randn(8, n, device="cuda").to(dtype)
    x[0, :n // 2] = float("-inf")
    x[1, :n - 1] = float("-inf")
    x[2, 1:] = float("-inf")
    x[3] = float("-inf")
    x[4, n // 2] = float("nan")
    x[5, n - 1] = float("inf")
    x[6, :] = 3.0
    y = MODULE[kind]()(x)
    ref = (torch.softmax if kind == "softmax" else torch.log_softmax)(x.double(), -1)
    assert bool(torch.isnan(y[3:6]).all())
    keep = torch.tensor([0, 1, 2, 6, 7], device="cuda")
    got, want = y[keep].double(), ref[keep]
    assert bool((torch.isinf(got) == torch.isinf(want)).all())
    finite = ~torch.isinf(want)
    eps = torch.finfo(dtype).eps                # one rounding to storage, float32 arithmetic in front of it
    bound = eps * want[finite].abs() + 2e-6 * (1 + want[finite].abs() if kind == "logsoftmax" else want[finite].abs()) + torch.finfo(dtype).tiny * (2 * eps)
    assert bool(((got[finite] - want[finite]).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("pad", PADS)
def test_slices_keep_to_their_rows(pad, dtype, sliced):
    """The records of the slices lie in the output while it is made: none is left behind, none lands in the padding of the rows; and the
    padding of the inputs, which is NaN, is not read."""
    vec = vec_of(dtype)
    n, m = 3 * SLICE * vec + vec - 1, 5
    announce(f"output guards, slices N={n} pad={pad} {dtype}")
    lib, st, code, pitch = _native.lib(), torch.cuda.current_stream().cuda_stream, _native.dtype_code(dtype), n + pad
    g = torch.Generator(device="cuda").manual_seed(n + pad)

    def source(values):
        buf, ptr, lead = padded(m, n, pad, dtype)
        buf.fill_(float("nan"))
        buf[lead:lead + m * pitch].view(m, pitch)[:, :n] = values
        return buf, ptr

    x = (0.3 + torch.randn(m, n, device="cuda", generator=g)).to(dtype)
    dy = torch.randn(m, n, device="cuda", generator=g).to(dtype)
    for kind in (_native.SOFTMAX, _native.LOGSOFTMAX):
        xbuf, xptr = source(x)
        ybuf, yptr, lead = padded(m, n, pad, dtype)
        assert lib.thn_softmax_fwd(xptr, pitch, yptr, pitch, m, n, kind, code, st) == 0
        y = check_guards(ybuf, m, n, pad, lead, f"softmax forward kind {kind}")
        ref = (torch.softmax if kind == _native.SOFTMAX else torch.log_softmax)(x.float(), -1)
        assert torch.allclose(y, ref.cpu(), rtol=1e-2 if dtype == torch.bfloat16 else 1e-5, atol=1e-6)
        ysbuf, ysptr = source(ref.to(dtype))
        dybuf, dyptr = source(dy)
        dxbuf, dxptr, lead = padded(m, n, pad, dtype)
        assert lib.thn_softmax_bwd(ysptr, pitch, dyptr, pitch, dxptr, pitch, m, n, kind, code, st) == 0
        dx = check_guards(dxbuf, m, n, pad, lead, f"softmax backward kind {kind}")
        saved, up = ref.to(dtype).double(), dy.double()
        want = saved * (up - (saved * up).sum(-1, keepdim=True)) if kind == _native.SOFTMAX else up - saved.exp() * up.sum(-1, keepdim=True)
        assert torch.allclose(dx.double(), want.cpu(), rtol=1e-2 if dtype == torch.bfloat16 else 1e-4, atol=1e-6)


def test_which_rows_are_sliced():
    """The edges of the rule (softmax_slicing in thn_api.hip), and streams out of step, which go to the walking kernels."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    bf16, f32 = torch.bfloat16, torch.float32
    half = (cus - 1) // 2
    for which, log, n, dtype, rows, want in (
            (2, 0, 65536, bf16, half, True), (2, 0, 65536, bf16, half + 1, False), (2, 0, 65535, bf16, half, False), (2, 1, 32768, f32, 1, True),
            (2, 1, 32767, f32, 1, False), (3, 1, 65536, bf16, half, True), (3, 0, 65536, bf16, cus // 4, True), (3, 0, 65536, bf16, cus // 4 + 1, False),
            (2, 0, 24576 * 8 + 7, bf16, half + 1, False), (2, 0, 24577 * 8, bf16, cus + cus // 2, True), (2, 0, 24577 * 8, bf16, cus + cus // 2 + 1, False),
            (3, 0, 24577 * 4, f32, cus + cus // 2, True), (3, 1, 24577 * 4, f32, cus + cus // 2 + 1, False),
            (2, 0, 7680 * 8, bf16, cus + 1, True), (2, 0, 7680 * 8, bf16, cus + cus // 5 + 1, False), (2, 0, 7681 * 8, bf16, cus + 1, False),
            (3, 0, 5120 * 8, bf16, cus + 1, False), (2, 0, 24577 * 8, torch.float64, 3, False)):
        shape = query_launch(which, log, rows, n, dtype)
        assert (shape[1] == 512) == want, (which, log, n, dtype, rows, shape)
    n = 128256
    x, dy = (t.cuda() for t in make((3, n), bf16, seed=2, scale=3.0))
    apart = torch.empty(x.numel() + 1, dtype=bf16, device="cuda")[1:].view_as(x)
    for kind in KINDS:
        y0, y1 = _launch.softmax_fwd(apart.copy_(x), CODE[kind]), _launch.softmax_fwd(x, CODE[kind])
        assert torch.allclose(y0.double(), y1.double(), rtol=2 ** -6, atol=1e-6)
        assert torch.allclose(y1.double().cpu(), torch.from_numpy(so.FWD[kind](x.double().cpu().numpy())), rtol=2 ** -7, atol=1e-6)
        d0, d1 = _launch.softmax_bwd(y1, apart.copy_(dy), CODE[kind]), _launch.softmax_bwd(y1, dy, CODE[kind])
        assert torch.allclose(d0.double(), d1.double(), rtol=2 ** -6, atol=1e-6)
