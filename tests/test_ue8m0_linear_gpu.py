"""The linear layer with packed UE8M0 weight scales in one call: against the same layer in its separate steps, at the
edges of the launch that quantises the activations and expands the weight scales together."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(1, 128, 128), (3, 192, 640), (33, 576, 1024), (130, 1000, 512), (5, 64, 4608)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_one_call_equals_its_steps(dev, M, N, K, dtype):
    from sglang_amd.quantization.fp8_kernel import sglang_per_token_group_quant_fp8, w8a8_block_fp8_matmul
    from sglang_amd.quantization.fp8_utils import deepgemm_w8a8_block_fp8_linear_with_fallback

    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device=dev).to(dtype)
    w = (torch.randn(N, K, generator=g, device=dev) * 100).clamp(-448, 448).to(torch.float8_e4m3fn)
    words = -(-(K // 128) // 4)
    e = torch.randint(112, 118, (-(-N // 128), words * 4), generator=g, device=dev, dtype=torch.uint8)
    ws = e.view(torch.int32).repeat_interleave(128, dim=0)[:N].contiguous()
    bias = torch.randn(N, generator=g, device=dev).to(dtype)
    out = deepgemm_w8a8_block_fp8_linear_with_fallback(x, w, [128, 128], ws, bias=bias)
    q, s = sglang_per_token_group_quant_fp8(x, 128, column_major_scales=True, scale_tma_aligned=True, scale_ue8m0=True)
    want = w8a8_block_fp8_matmul(q, w, s, ws, [128, 128], output_dtype=dtype) + bias
    assert out.shape == (M, N) and torch.equal(out, want)
