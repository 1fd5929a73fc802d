"""Block-scaled FP8 linears with a bias: added inside the GEMM's epilogue, the bits of out.add_(bias) behind it, on every
kernel the GEMM may run."""
import pytest
import torch

pytestmark = pytest.mark.gpu

STREAMING, TILE64, TILE128, TILE256, PERSISTENT256, POW2, TILE192, STRIP = 1, 2, 3, 4, 5, 7, 9, 10  # SGLAMD_KERNEL_* of include/sglamd.h


@pytest.mark.parametrize("M,N,K,kernel", [
    (1, 1000, 1024, STREAMING),
    (24, 776, 2048, STREAMING),
    (40, 512, 1024, STREAMING),
    (40, 512, 12288, TILE64),           # K split: the bias in the reduction
    (40, 512, 7168, STRIP),             # ... of strips
    (48, 24640, 512, TILE64),           # ragged last column tile
    (40, 36864, 5120, STRIP),
    (24, 40000, 2560, STRIP),           # one row tile
    (128, 33026, 512, TILE128),         # N not a multiple of 4
    (300, 24577, 1280, TILE192),        # N odd
    (1000, 14340, 512, TILE256),
    (512, 36864, 512, TILE256),         # cut in two along N
    (2500, 8392, 512, PERSISTENT256),   # last column tile of 200: a patch that starts inside the last 32 columns
    (2600, 8968, 640, TILE128),         # odd number of K blocks
    (65800, 24, 512, PERSISTENT256),    # fewer columns than the patch that the epilogue reads the bias in
])
@pytest.mark.parametrize("ue8m0", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_bias_in_the_epilogue(dev, M, N, K, kernel, ue8m0, dtype):
    from sglang_amd import _C
    from sglang_amd._lib import lib

    print(f"bias M={M} N={N} K={K} ue8m0={ue8m0} {dtype}", flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).to(dtype).to(dev)
    w = (torch.randn(N, K, generator=g) * 100).clamp(-448, 448).to(torch.float8_e4m3fn).to(dev)
    nb, kb = -(-N // 128), K // 128
    if ue8m0:
        codes = torch.randint(110, 118, (N, -(-kb // 4) * 4), generator=g, dtype=torch.uint8)
        codes = codes[torch.arange(N) // 128 * 128]  # one scale per 128 rows
        ws = codes.view(torch.int32).t().contiguous().t().to(dev)
    else:
        ws = (torch.rand(nb, kb, generator=g) * 1e-3 + 1e-4).to(dev)
    for off in (0, 1):  # the second time a view one element into its storage
        bias = (torch.randn(N + off, generator=g) * 3).to(dtype).to(dev)[off:]
        plain = _C.block_linear(x, w, ws, None)
        ran = lib.sglamd_last_gemm_kernel()
        out = _C.block_linear(x, w, ws, bias)
        assert ran == (POW2 if ue8m0 and kernel == PERSISTENT256 else kernel), f"ran kernel {ran}"
        assert lib.sglamd_last_gemm_kernel() == ran, "another kernel with the bias"
        assert plain.abs().max() > 1 and not torch.equal(out, plain)
        want = plain.float().to(dtype).add_(bias)
        assert torch.equal(out, want)
