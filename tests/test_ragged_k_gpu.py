"""Row-scaled GEMMs whose K is not a multiple of 128, on the tile kernel: the last K block holds one to seven 16-byte
pieces of a row, and what lies behind them in memory (here: NaN codes) must not be read into the sums."""
import pytest
import torch

from oracle import gemm as og
from tests.util import assert_gemm_close

pytestmark = pytest.mark.gpu

GENERIC, TILES = 6, (2, 3, 4)  # SGLAMD_KERNEL_* of include/sglamd.h


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("M,N,K", [
    (65, 264, 528),       # one piece in the last block, ragged column tile
    (100, 33024, 752),    # seven pieces, 128-row tiles in one slice
    (130, 520, 4112),     # K split over workgroups, the last slice ends in one piece
    (300, 1000, 2096),    # split, ragged rows
    (1000, 14336, 592),   # 256-row tiles
    (40, 20480, 1040),    # 33..64 rows
    (200, 520, 4208),     # K split, seven pieces in the last slice
    (100, 520, 400),      # short K stays with the generic kernel
])
def test_ragged_k(dev, int8, M, N, K):
    import sglang_amd as sa
    from sglang_amd._lib import lib

    g = torch.Generator().manual_seed(M + N + K)
    pad = -K % 128 + 128
    if int8:
        a, b = (torch.randint(-127, 128, s, generator=g, dtype=torch.int8) for s in ((M, K + pad), (N, K + pad)))
    else:
        a, b = ((torch.randn(s, generator=g) * 50).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
                for s in ((M, K + pad), (N, K + pad)))
        a[:, K:], b[:, K:] = 0x7F, 0x7F
        a, b = a.view(torch.float8_e4m3fn), b.view(torch.float8_e4m3fn)
    s_a, s_b = torch.rand(M, 1, generator=g) * 1e-2, torch.rand(N, 1, generator=g) * 1e-2
    bias = torch.randn(N, generator=g).to(torch.bfloat16)
    mm, ref_mm = (sa.int8_scaled_mm, og.int8_scaled_mm) if int8 else (sa.fp8_scaled_mm, og.fp8_scaled_mm)
    out = mm(a.to(dev)[:, :K], b.to(dev)[:, :K].t(), s_a.to(dev), s_b.to(dev), torch.bfloat16, bias.to(dev))
    ran = lib.sglamd_last_gemm_kernel()
    assert ran == GENERIC if K < 512 else ran in TILES, f"ran kernel {ran}"
    raw = lambda t: t.numpy() if int8 else t.view(torch.uint8).numpy()  # noqa: E731
    ref = ref_mm(raw(a[:, :K].contiguous()), raw(b[:, :K].contiguous()), s_a.numpy().reshape(-1),
                 s_b.numpy().reshape(-1), out_dtype=torch.bfloat16, bias=bias)
    assert_gemm_close(out, ref.float(), f"ragged rows M={M} N={N} K={K}")
