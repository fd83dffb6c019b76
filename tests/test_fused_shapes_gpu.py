"""Norm kernels with an activation epilogue: every launch shape off the 128-bit path, and the rules that choose shapes and workgroups
per compute unit (plan_launch in thn_api.hip) at their edges."""
import os
import re

import pytest
import torch

from conftest import ROOT
from test_fused_parity_gpu import announce, fused_shapes, make, run_and_compare
from TritonHub import _native
from TritonHub.Normalization._launch import query_launch

pytestmark = pytest.mark.gpu


def off_path_shapes():
    text = open(os.path.join(ROOT, "triton-hub_amd", "csrc", "thn_fused_dispatch.h")).read()
    body = re.search(r"#define THN_FUSED_BWD_SHAPES_OFF_PATH\(X\)(.*)\n", text).group(1)
    fwd, bwd = fused_shapes()
    return fwd, bwd + [(int(k), int(t), int(b)) for k, t, b in re.findall(r"X\((\d+), (\d+), (\d+)\)", body)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_every_launch_shape_off_the_128_bit_path(dtype):
    """Full rows but for one element (an overlapped window of which one column counts), and rows that leave a third of the slots idle."""
    lib, vec = _native.lib(), 16 // torch.empty(0, dtype=dtype).element_size()
    try:
        for which, shapes in zip((9, 10), off_path_shapes()):
            for k, tpr, block in shapes:
                for n in (k * tpr * vec - 1, (k * tpr - tpr // 3) * vec + 1):
                    if n * (16 // vec) > 65536:
                        continue
                    m = 2 * (block // tpr) + 1
                    announce(f"fused shape off the path family={which} K={k} TPR={tpr} block={block} N={n} M={m} {dtype}")
                    assert lib.thn_norm_set_launch_override(which, k, tpr, block, 0) == 0
                    assert query_launch(which, True, m, n, dtype)[:3] == (k, tpr, block)
                    x, dy, w, b = make((m, n), dtype, seed=k * 100 + tpr)
                    run_and_compare("ln", "gelu", x, dy, w, b, 1e-5, f"ln shape {k},{tpr},{block}")
                    run_and_compare("rms", "silu", x, dy, w, None, 1e-5, f"rms shape {k},{tpr},{block}")
                    assert lib.thn_norm_set_launch_override(which, 0, 0, 0, 0) == 0
    finally:
        lib.thn_norm_set_launch_override(9, 0, 0, 0, 0)
        lib.thn_norm_set_launch_override(10, 0, 0, 0, 0)


@pytest.mark.parametrize("dtype,rows,n", [(torch.bfloat16, 12288, 264), (torch.bfloat16, 12288, 320), (torch.float16, 6144, 640), (torch.bfloat16, 3072, 1281),
                                          (torch.float16, 1536, 2560), (torch.bfloat16, 768, 5120), (torch.float32, 8192, 384), (torch.float32, 1536, 1025),
                                          (torch.bfloat16, 16384, 384), (torch.float16, 300, 1601), (torch.bfloat16, 300, 12301)])
def test_many_rows_in_the_shapes_of_their_own(rows, n, dtype):
    announce(f"fused {dtype} {rows} x {n}")
    x, dy, w, b = make((rows, n), dtype, seed=n)
    run_and_compare("ln", "gelu", x, dy, w, b, 1e-5, f"ln+gelu {rows} x {n}")
    run_and_compare("ln", "silu", x, dy, w, b, 1e-5, f"ln+silu {rows} x {n}")
    run_and_compare("rms", "silu", x, dy, w, None, 1e-5, f"rms+silu {rows} x {n}")


def test_which_shapes_and_how_many_workgroups():
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    bf16, f32 = torch.bfloat16, torch.float32
    ln, gelu, silu, tanh = 1, 2 * _native.ACT_GELU, 2 * _native.ACT_SILU, 2 * _native.ACT_GELU_TANH
    for which, flavour, rows, n, dtype, shape in (
            # 5 x t from 1.5 workgroup steps per compute unit on, 33 to 40, 65 to 80 ... vectors
            (9, ln + gelu, 48 * cus, 320, bf16, (5, 8, 256)), (9, ln + gelu, 48 * cus - 1, 320, bf16, (3, 16, 256)), (9, ln + gelu, 24 * cus - 1, 320, bf16, (4, 16, 256)),
            (9, ln + gelu, 48 * cus, 328, bf16, (3, 16, 256)),
            (9, ln + gelu, 48 * cus, 256, bf16, (4, 8, 256)), (9, ln + gelu, 24 * cus, 640, bf16, (5, 16, 256)), (9, silu, 24 * cus, 640, bf16, (3, 32, 256)),
            (9, silu, 12 * cus, 1280, bf16, (5, 32, 256)), (9, gelu, 6 * cus, 2561, bf16, (3, 128, 256)), (9, gelu, 6 * cus, 2553, bf16, (5, 64, 256)),
            (9, ln + gelu, 3 * cus, 5120, bf16, (5, 128, 256)), (9, ln + gelu, 3 * cus - 1, 5120, bf16, (3, 256, 256)), (9, ln + gelu, 48 * cus, 160, f32, (4, 16, 256)),
            (9, gelu, 12 * cus, 513, f32, (5, 32, 256)), (9, gelu, 16, 1027, bf16, (4, 64, 256)),
            # 3 x 16 and 3 x 32 backward
            (10, ln + gelu, 64 * cus, 384, bf16, (3, 16, 256)), (10, ln + gelu, 64 * cus - 1, 384, bf16, (2, 32, 256)), (10, silu, 32 * cus, 768, f32, (3, 64, 256)),
            (10, silu, 32 * cus, 768, bf16, (3, 32, 256)), (10, silu, 16, 690, bf16, (3, 32, 256)),
            # off the path
            (10, ln + silu, 4096, 1601, bf16, (4, 64, 256)), (10, ln + gelu, 4096, 1601, bf16, (2, 128, 512)), (10, silu, 4096, 1601, bf16, (2, 128, 512)),
            (10, silu, 4096, 12301, bf16, (4, 512, 512)), (10, ln + silu, 4096, 12301, bf16, (2, 1024, 1024)), (10, tanh, 4096, 4099, bf16, (4, 256, 256)),
            (10, gelu, 4096, 4099, bf16, (3, 256, 512)), (10, silu, 4096, 5, bf16, (4, 8, 256))):
        assert query_launch(which, flavour, rows, n, dtype)[:3] == shape, (which, flavour, rows, n, dtype)
    for flavour, rows, n, dtype, groups in ((silu, 256 * cus, 256, bf16, 4), (silu, 255 * cus, 256, bf16, 2), (silu, 64 * cus - 1, 256, bf16, 1), (ln + silu, 64 * cus, 1536, bf16, 2),
                                            (silu, 64 * cus, 1536, bf16, 1), (silu, 64 * cus, 1280, bf16, 2), (silu, 256 * cus, 128, f32, 1), (silu, 256 * cus, 108, f32, 2),
                                            (gelu, 64 * cus, 2048, bf16, 1), (ln + gelu, 64 * cus, 1024, f32, 1)):
        grid = query_launch(10, flavour, rows, n, dtype)[3]
        assert (groups - 1) * cus < grid <= groups * cus, (flavour, rows, n, dtype, grid)
