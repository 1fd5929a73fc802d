"""A block-scaled linear layer of a few rows quantises them in the GEMM's workgroups: the bits of the two launches it stands
for, over widths and depths that change the tile, the waves that share K and the passes over the rows, and at the number of
rows and the depth where it goes back to two launches."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K", [(64, 128), (1024, 256), (7168, 16384), (7168, 18432), (2112, 7168), (24576, 1536), (576, 4096),
                                 (36864, 640), (4160, 2432)])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("dtype,bias", [(torch.bfloat16, False), (torch.float16, True)])
def test_equals_quantise_then_multiply(dev, M, N, K, dtype, bias):
    from sglang_amd.quantization.fp8_kernel import sglang_per_token_group_quant_fp8, w8a8_block_fp8_matmul
    from sglang_amd.quantization.fp8_utils import dispatch_w8a8_block_fp8_linear

    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device=dev).to(dtype)
    x[:, :128] = 0  # a group of zeros: its scale is the smallest one
    if K > 256:
        x[-1, 200] = float("inf")
        x[0, 300] = float("nan")
    w = torch.randn(N, K, generator=g, device=dev).mul_(100).clamp_(-448, 448).to(torch.float8_e4m3fn)
    ws = torch.rand(-(-N // 128), K // 128, generator=g, device=dev) * 1e-3 + 1e-4
    b = torch.randn(N, generator=g, device=dev).to(dtype) if bias else None
    print(f"one launch M={M} N={N} K={K} {dtype} bias={bias}", flush=True)
    out = dispatch_w8a8_block_fp8_linear()(x, w, [128, 128], ws, bias=b)
    q, s = sglang_per_token_group_quant_fp8(x, 128, column_major_scales=True)
    ref = w8a8_block_fp8_matmul(q, w, s, ws, [128, 128], output_dtype=dtype)
    if bias:
        ref = ref + b
    assert torch.equal(out.isnan(), ref.isnan())
    assert torch.equal(out.nan_to_num(), ref.nan_to_num())
    # a second call on other rows: nothing of the first stays
    x2 = torch.randn(M, K, generator=g, device=dev).to(dtype)
    q, s = sglang_per_token_group_quant_fp8(x2, 128, column_major_scales=True)
    ref = w8a8_block_fp8_matmul(q, w, s, ws, [128, 128], output_dtype=dtype)
    assert torch.equal(dispatch_w8a8_block_fp8_linear()(x2, w, [128, 128], ws, bias=b), ref + b if bias else ref)


@pytest.mark.parametrize("N,K", [(64, 128), (1024, 256), (7168, 16384), (7168, 18432), (2112, 7168), (24576, 1536), (576, 4096),
                                 (36864, 640), (4160, 2432), (264, 2064)])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("dtype,bias", [(torch.bfloat16, False), (torch.float16, True)])
def test_per_channel_equals_quantise_then_multiply(dev, M, N, K, dtype, bias):
    """The row's maximum spans all of its groups, several waves and passes; rows of zeros have the scale zero."""
    from sglang_amd.ops import fp8_scaled_mm, sgl_per_token_quant_fp8
    from sglang_amd.quantization.fp8_utils import apply_fp8_linear

    g = torch.Generator(device=dev).manual_seed(M + N + K)
    w = torch.randn(N, K, generator=g, device=dev).mul_(100).clamp_(-448, 448).to(torch.float8_e4m3fn)
    ws = torch.rand(N, 1, generator=g, device=dev) * 1e-3 + 1e-4
    b = torch.randn(N, generator=g, device=dev).to(dtype) if bias else None
    for kind in ("plain", "zeros", "nan", "inf"):
        x = torch.randn(M, K, generator=g, device=dev).to(dtype)
        x[-1, -1] = 50.0  # the maximum of a row in its last group
        if kind == "zeros":
            x[0] = 0
        elif kind == "nan":
            x[M // 2, K // 2] = float("nan")
        elif kind == "inf":
            x[M // 2, 3] = float("inf")
        print(f"one launch, row scales, M={M} N={N} K={K} {dtype} {kind}", flush=True)
        out = apply_fp8_linear(x, w.t(), ws, bias=b, use_per_token_if_dynamic=True)
        q = torch.empty(M, K, device=dev, dtype=torch.float8_e4m3fn)
        s = torch.empty(M, 1, device=dev, dtype=torch.float32)
        sgl_per_token_quant_fp8(x, q, s)
        ref = fp8_scaled_mm(q, w.t(), s, ws, dtype, b)
        assert torch.equal(out.isnan(), ref.isnan())
        assert torch.equal(out.nan_to_num(), ref.nan_to_num())
