"""Dense GEMMs in 192-row tiles, at the edges of the tiles, against the oracle."""
import pytest
import torch

from tests.test_strip_gpu import MODES, _check, _run

pytestmark = pytest.mark.gpu

TILE192 = 9  # SGLAMD_KERNEL_* of include/sglamd.h


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("M,N,K,pitch", [
    (300, 24577, 1280, 0),     # the last column tile of one column
    (385, 16390, 1152, 128),   # one row in the last row tile; an odd number of K blocks
    (384, 24576, 1280, 0),
    (577, 30724, 1152, 0),     # two rounds
    (383, 7172, 12288, 0),     # K split
    (385, 16390, 1168, 16),    # row modes: one piece in the last K block
    (530, 6000, 12400, 0),     # ... seven, in the last slice
])
def test_tiles_of_192_rows(dev, mode, M, N, K, pitch):
    from sglang_amd._lib import lib

    if K % 128 and mode.startswith("block"):
        pytest.skip("block scales cover whole K blocks")
    print(f"192-row tiles {mode} M={M} N={N} K={K} pitch +{pitch}", flush=True)
    out, ref = _run(dev, mode, M, N, K, torch.bfloat16, False, pitch, col_scales=M % 2 == 0)
    assert lib.sglamd_last_gemm_kernel() == TILE192, f"kernel {lib.sglamd_last_gemm_kernel()}"
    _check(out, ref, f"192-row tiles {mode} M={M} N={N} K={K}")


@pytest.mark.parametrize("mode", MODES)  # (a bias with block scales: tests/test_block_bias_gpu.py)
@pytest.mark.parametrize("M,N,K", [(300, 24577, 1280), (383, 7172, 12288)])
def test_tiles_of_192_rows_half_and_bias(dev, mode, M, N, K):
    from sglang_amd._lib import lib

    print(f"192-row tiles, half, {mode} M={M} N={N} K={K}", flush=True)
    out, ref = _run(dev, mode, M, N, K, torch.float16, True, 0, False)
    assert lib.sglamd_last_gemm_kernel() == TILE192, f"kernel {lib.sglamd_last_gemm_kernel()}"
    _check(out, ref, f"192-row tiles {mode} M={M} N={N} K={K} half, bias")
