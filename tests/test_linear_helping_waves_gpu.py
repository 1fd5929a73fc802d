"""Linear layers of five to sixteen short rows in one launch, where more waves quantise than share K: the bits of the two launches."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K", [(512, 128), (264, 512), (1024, 1024), (4096, 768), (7168, 2048), (24576, 1536), (16384, 1024), (32768, 512)])
@pytest.mark.parametrize("M", [2, 4, 6, 8, 13, 16])
@pytest.mark.parametrize("row_scales", [False, True])
@pytest.mark.parametrize("dtype,bias", [(torch.bfloat16, False), (torch.float16, True)])
def test_equals_quantise_then_multiply(dev, M, N, K, row_scales, dtype, bias):
    from sglang_amd.ops import fp8_scaled_mm, sgl_per_token_quant_fp8
    from sglang_amd.quantization.fp8_kernel import sglang_per_token_group_quant_fp8, w8a8_block_fp8_matmul
    from sglang_amd.quantization.fp8_utils import apply_fp8_linear, dispatch_w8a8_block_fp8_linear

    g = torch.Generator(device=dev).manual_seed(M + N + K)
    w = torch.randn(N, K, generator=g, device=dev).mul_(100).clamp_(-448, 448).to(torch.float8_e4m3fn)
    b = torch.randn(N, generator=g, device=dev).to(dtype) if bias else None
    ws = (torch.rand(N, 1, generator=g, device=dev) if row_scales else torch.rand(-(-N // 128), K // 128, generator=g, device=dev)) * 1e-3 + 1e-4
    print(f"one launch M={M} N={N} K={K} row_scales={row_scales} {dtype}", flush=True)
    for kind in ("plain", "zeros", "nan"):
        x = torch.randn(M, K, generator=g, device=dev).to(dtype)
        x[-1, -1] = 50.0  # the maximum of the last row in its last group
        if kind != "plain":
            x[M // 2] = 0 if kind == "zeros" else float("nan")
        if row_scales:
            out = apply_fp8_linear(x, w.t(), ws, bias=b, use_per_token_if_dynamic=True)
            q, s = torch.empty(M, K, device=dev, dtype=torch.float8_e4m3fn), torch.empty(M, 1, device=dev, dtype=torch.float32)
            sgl_per_token_quant_fp8(x, q, s)
            ref = fp8_scaled_mm(q, w.t(), s, ws, dtype, b)
        else:
            out = dispatch_w8a8_block_fp8_linear()(x, w, [128, 128], ws, bias=b)
            q, s = sglang_per_token_group_quant_fp8(x, 128, column_major_scales=True)
            ref = w8a8_block_fp8_matmul(q, w, s, ws, [128, 128], output_dtype=dtype)
            ref = ref + b if bias else ref
        assert torch.equal(out.isnan(), ref.isnan())
        assert torch.equal(out.nan_to_num(), ref.nan_to_num())


MORE_ROWS = """
import torch
from sglang_amd.quantization.fp8_kernel import sglang_per_token_group_quant_fp8, w8a8_block_fp8_matmul
from sglang_amd.quantization.fp8_utils import dispatch_w8a8_block_fp8_linear
g = torch.Generator(device="cuda").manual_seed(1)
for M in (16, 17, 32):
    x = torch.randn(M, 512, generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randn(1024, 512, generator=g, device="cuda").mul_(100).clamp_(-448, 448).to(torch.float8_e4m3fn)
    ws = torch.rand(8, 4, generator=g, device="cuda") * 1e-3 + 1e-4
    print("rows", M, flush=True)
    out = dispatch_w8a8_block_fp8_linear()(x, w, [128, 128], ws)
    q, s = sglang_per_token_group_quant_fp8(x, 128, column_major_scales=True)
    assert torch.equal(out, w8a8_block_fp8_matmul(q, w, s, ws, [128, 128], output_dtype=torch.bfloat16)), M
"""


def test_a_limit_past_the_tile_is_the_tile(dev):
    """SGLAMD_LINEAR_FUSE_ROWS above the sixteen rows that a workgroup holds (read once per process)."""
    import os
    import subprocess
    import sys

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", MORE_ROWS], env=dict(os.environ, SGLAMD_LINEAR_FUSE_ROWS="64"), cwd=root, timeout=100,
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
