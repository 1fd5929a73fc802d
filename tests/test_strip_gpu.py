"""Dense GEMMs of 17 to 1024 rows off the tile kernels: the strip kernel (weights in tiles of 32 to 160 rows, loading and multiplying
waves) and the streaming kernel walking several row tiles, at the edges of their tiles, against the oracle."""
import numpy as np
import pytest
import torch

from oracle import gemm as og
from tests.util import assert_gemm_close

pytestmark = pytest.mark.gpu

MODES = ["block_fp8", "block_int8", "row_fp8", "row_int8"]


def _codes(shape, int8, g):
    if int8:
        return torch.randint(-128, 128, shape, generator=g, dtype=torch.int32).to(torch.int8)
    c = torch.randint(0, 256, shape, generator=g, dtype=torch.int32).to(torch.uint8)
    return torch.where((c & 0x7F) == 0x7F, c & 0x80, c)


def _run(dev, mode, M, N, K, dtype, bias, pitch, col_scales):
    """(output, reference); operands are views into rows of K + pitch bytes, the bytes past K NaN codes, and with a pitch the output
    one into longer rows too."""
    from sglang_amd._lib import lib

    int8 = mode.endswith("int8")
    g = torch.Generator().manual_seed(M * 7 + N + K)
    a, b = _codes((M, K), int8, g), _codes((N, K), int8, g)

    def put(t):
        wide = torch.full((t.shape[0], K + pitch), 0x7F, dtype=t.dtype)
        wide[:, :K] = t
        wide = wide.to(dev)
        return (wide if int8 else wide.view(torch.float8_e4m3fn))[:, :K]

    ad, bd, an, bn = put(a), put(b), a.numpy(), b.numpy()
    bi = torch.randn(N, generator=g).to(dtype) if bias else None
    # through the C ABI, which takes any pitch and any N
    need = lib.sglamd_gemm_workspace_bytes(M, N, K)
    scratch, ldc = torch.empty(max(need, 16), dtype=torch.uint8, device=dev), N + (13 if pitch else 0)
    rows = torch.full((M, ldc), 7.0, dtype=dtype, device=dev)
    out = rows[:, :N]
    tag, stream = 2 if dtype == torch.bfloat16 else 1, torch.cuda.current_stream().cuda_stream
    if mode.startswith("block"):
        xs = (torch.rand(M, K // 128, generator=g) * 1e-2 + 1e-3)
        ws = (torch.rand(-(-N // 128), K // 128, generator=g) * 1e-2 + 1e-3)
        xs_d = xs.to(dev).t().contiguous().t() if col_scales else xs.to(dev)
        fn, ref_mm = ((lib.sglamd_int8_blockwise_scaled_mm, og.block_int8_matmul) if int8
                      else (lib.sglamd_fp8_blockwise_scaled_mm, og.block_fp8_matmul))
        ws_d = ws.to(dev)
        rc = fn(ad.data_ptr(), ad.stride(0), bd.data_ptr(), bd.stride(0), xs_d.data_ptr(), xs_d.stride(0), xs_d.stride(1),
                ws_d.data_ptr(), ws_d.stride(0), ws_d.stride(1), out.data_ptr(), ldc, tag, M, N, K, scratch.data_ptr(), need, stream)
        assert rc == 0 and bool((rows[:, N:] == 7.0).all())
        return out, ref_mm(an, bn, xs.numpy(), ws.numpy(), return_fp32=True)
    s_a, s_b = torch.rand(M, generator=g) * 1e-2 + 1e-3, torch.rand(N, generator=g) * 1e-2 + 1e-3
    fn, ref_mm = ((lib.sglamd_int8_scaled_mm, og.int8_scaled_mm) if int8 else (lib.sglamd_fp8_scaled_mm, og.fp8_scaled_mm))
    sa_d, sb_d, bi_d = s_a.to(dev), s_b.to(dev), None if bi is None else bi.to(dev)
    rc = fn(ad.data_ptr(), ad.stride(0), bd.data_ptr(), bd.stride(0), sa_d.data_ptr(), sb_d.data_ptr(), 0 if bi is None else bi_d.data_ptr(),
            out.data_ptr(), ldc, tag, M, N, K, scratch.data_ptr(), need, stream)
    assert rc == 0 and bool((rows[:, N:] == 7.0).all())
    return out, ref_mm(an, bn, s_a.numpy(), s_b.numpy(), out_dtype=dtype, bias=bi).float()


def _check(out, ref, what):
    assert_gemm_close(out, ref, what)
    o, r = out.float().cpu(), torch.as_tensor(np.asarray(ref)).float()
    for dim, name in ((1, "row"), (0, "column")):
        each = (o - r).norm(dim=dim) / r.norm(dim=dim).clamp_min(1e-30)
        assert float(each.max()) <= 1e-2, f"{what}: {name} {int(each.argmax())} rel-L2 {float(each.max()):.3e}"


# rows either side of the row tiles' edges; weight rows that end inside a strip, half a strip and a scale block; tiles that straddle
# scale blocks; several items per workgroup; K split, and K blocks that do not divide by the slices
@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("M,N,K,pitch", [
    (17, 40009, 2560, 0),       # one row tile: five strips
    (31, 65540, 2048, 128),     # ... four, two tiles a workgroup
    (24, 24570, 4224, 0),       # ... three
    (32, 28672, 3584, 0),
    (33, 30016, 4096, 0),
    (64, 30024, 4096, 128),     # five strips, the last tile ragged
    (65, 28681, 4096, 0),       # N odd: single stores
    (96, 30720, 2688, 256),
    (97, 28672, 3200, 0),
    (128, 33010, 3072, 0),
    (128, 65540, 2560, 0),      # two tiles a workgroup
    (48, 9000, 6400, 0),        # K split
    (64, 7176, 9088, 128),      # ... 71 blocks
    (128, 7172, 10752, 0),
])
def test_strip_kernel(dev, mode, M, N, K, pitch):
    from sglang_amd._lib import lib

    print(f"strip {mode} M={M} N={N} K={K} pitch +{pitch}", flush=True)
    out, ref = _run(dev, mode, M, N, K, torch.bfloat16, False, pitch, col_scales=M % 2 == 0)
    shape = lib.sglamd_last_strip_shape()
    assert shape >> 24 == -(-M // 32) and lib.sglamd_last_gemm_kernel() == 10, f"not the strip kernel: {shape:#x}"
    assert lib.sglamd_last_streaming_shape() == 0
    assert (shape >> 16 & 0xFF) > 1 or N > 10000, "meant to split K"
    _check(out, ref, f"strip {mode} M={M} N={N} K={K}")


# the shortest K of each depth with three and more tiles a workgroup, where the weight scales of a tile are requested while the
# one before is multiplied; a block less, and block scales stay with the streaming kernel
@pytest.mark.parametrize("mode", ["block_fp8", "block_int8"])
@pytest.mark.parametrize("M,N,K,strips", [
    (17, 195416, 512, True),    # five stages
    (23, 209576, 512, True),
    (31, 127568, 896, True),    # six
    (33, 200008, 512, True),    # three
    (80, 200008, 512, True),
    (100, 200008, 768, True),
    (32, 261376, 384, False),
    (17, 398592, 256, False),
    (24, 790016, 128, False),
])
def test_few_k_blocks_and_many_tiles(dev, mode, M, N, K, strips):
    from sglang_amd._lib import lib

    print(f"short K {mode} M={M} N={N} K={K}", flush=True)
    out, ref = _run(dev, mode, M, N, K, torch.bfloat16, False, 0, col_scales=True)
    shape = lib.sglamd_last_strip_shape()
    assert (shape != 0) == strips and (not strips or -(-N // (shape & 0xFFFF)) > 512), f"{shape:#x}"
    _check(out, ref, f"short K {mode} M={M} N={N} K={K}")


@pytest.mark.parametrize("mode", MODES)  # (the block modes without a bias: tests/test_block_bias_gpu.py)
@pytest.mark.parametrize("M,N,K", [(65, 28681, 4096), (100, 9000, 9600), (30, 40009, 2560)])
def test_strip_kernel_half_and_bias(dev, mode, M, N, K):
    from sglang_amd._lib import lib

    out, ref = _run(dev, mode, M, N, K, torch.float16, True, 0, False)
    assert lib.sglamd_last_strip_shape(), "not the strip kernel"
    _check(out, ref, f"strip {mode} M={M} N={N} K={K} half, bias")


# the same bits for a row wherever it sits, for a bias added by the kernel or behind it, and from run to run
@pytest.mark.parametrize("M,N,K", [(128, 33010, 3072), (64, 7176, 9088), (200, 600, 1664), (72, 2050, 2048)])
def test_rows_and_bias(dev, M, N, K):
    from sglang_amd import _C
    from sglang_amd._lib import lib

    g = torch.Generator().manual_seed(M + N)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).to(dev)
    w = (torch.randn(N, K, generator=g) * 100).clamp(-448, 448).to(torch.float8_e4m3fn).to(dev)
    ws = (torch.rand(-(-N // 128), K // 128, generator=g) * 1e-3 + 1e-4).to(dev)
    bias = torch.randn(N, generator=g).to(torch.bfloat16).to(dev)
    out = _C.block_linear(x, w, ws, None)
    strip, kernel = lib.sglamd_last_strip_shape(), lib.sglamd_last_gemm_kernel()
    assert strip if N > 7000 else kernel == 1, f"kernel {kernel}, strip {strip:#x}"
    assert torch.equal(out, _C.block_linear(x, w, ws, None))
    perm = torch.randperm(M, generator=g).to(dev)
    assert torch.equal(_C.block_linear(x[perm].contiguous(), w, ws, None), out[perm])
    assert torch.equal(_C.block_linear(x, w, ws, bias), out.clone().add_(bias))
    assert (lib.sglamd_last_strip_shape(), lib.sglamd_last_gemm_kernel()) == (strip, kernel), "another kernel with the bias"


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("M,N,K", [
    (65, 1000, 8192),     # row tiles of 32, the last of one row
    (72, 2050, 2048),
    (130, 512, 8192),
    (200, 600, 1664),
    (320, 512, 512),
    (150, 1152, 2176),    # an odd number of K blocks
    (40, 576, 6144),
])
def test_streaming_kernel_over_row_tiles(dev, mode, M, N, K):
    from sglang_amd._lib import lib

    out, ref = _run(dev, mode, M, N, K, torch.bfloat16, False, 0, col_scales=True)
    assert lib.sglamd_last_gemm_kernel() == 1 and lib.sglamd_last_strip_shape() == 0
    _check(out, ref, f"row tiles {mode} M={M} N={N} K={K}")


# a K that does not fill its last block: one piece, seven, K split; rows that are views
@pytest.mark.parametrize("mode", ["row_fp8", "row_int8"])
@pytest.mark.parametrize("M,N,K,pitch,kernel", [
    (18, 24580, 4112, 16, "strip"),
    (33, 30016, 4112, 0, "strip"),
    (80, 23800, 5984, 16, "strip"),
    (128, 28673, 3184, 128, "strip"),
    (48, 9000, 6416, 0, "strip"),       # K split
    (100, 9000, 8816, 16, "strip"),
    (96, 512, 1424, 0, 2),              # row tiles of 32 rows, 64, 16
    (110, 2160, 2672, 16, 4),
    (200, 584, 1264, 0, 4),
    (50, 968, 4928, 0, 1),
    (20, 600, 1936, 16, 1),
])
def test_ragged_k(dev, mode, M, N, K, pitch, kernel):
    from sglang_amd._lib import lib

    print(f"ragged {mode} M={M} N={N} K={K} pitch +{pitch}", flush=True)
    out, ref = _run(dev, mode, M, N, K, torch.bfloat16, True, pitch, col_scales=False)
    if kernel == "strip":
        assert lib.sglamd_last_strip_shape(), "not the strip kernel"
    else:
        assert lib.sglamd_last_gemm_kernel() == 1 and lib.sglamd_last_streaming_shape() >> 16 == kernel
    _check(out, ref, f"ragged {mode} M={M} N={N} K={K}")


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("M,N,K", [(17, 704, 4736), (31, 1152, 896), (32, 768, 7936), (33, 512, 1408), (64, 640, 4736)])
def test_row_tiles_of_16(dev, mode, M, N, K):
    from sglang_amd._lib import lib

    out, ref = _run(dev, mode, M, N, K, torch.bfloat16, False, 0, col_scales=False)
    assert lib.sglamd_last_gemm_kernel() == 1 and lib.sglamd_last_streaming_shape() >> 16 == 1 and not lib.sglamd_last_strip_shape()
    _check(out, ref, f"row tiles of 16 {mode} M={M} N={N} K={K}")


def test_without_workspace_the_strip_kernel_does_not_split(dev):
    """A call that has no room for the slabs runs what it ran before."""
    from sglang_amd._lib import lib

    M, N, K = 48, 9000, 6400
    g = torch.Generator().manual_seed(1)
    a, b = (_codes(s, False, g) for s in ((M, K), (N, K)))
    ad, bd = a.to(dev), b.to(dev)
    s_a, s_b = torch.rand(M, generator=g), torch.rand(N, generator=g)
    sad, sbd, out = s_a.to(dev), s_b.to(dev), torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    need = lib.sglamd_gemm_workspace_bytes(M, N, K)
    assert need > 0
    ws = torch.empty(need, dtype=torch.uint8, device=dev)
    ref = og.fp8_scaled_mm(a.numpy(), b.numpy(), s_a.numpy(), s_b.numpy(), out_dtype=torch.bfloat16).float()
    stream = torch.cuda.current_stream().cuda_stream
    for bytes_, strip in ((need, True), (0, False)):
        rc = lib.sglamd_fp8_scaled_mm(ad.data_ptr(), K, bd.data_ptr(), K, sad.data_ptr(), sbd.data_ptr(), 0, out.data_ptr(), N, 2, M, N, K,
                                      ws.data_ptr() if bytes_ else 0, bytes_, stream)
        assert rc == 0 and (lib.sglamd_last_strip_shape() != 0) == strip
        _check(out, ref, f"workspace of {bytes_}")
