"""Fused-MoE GEMMs over weights whose row pitch is a multiple of 4096 bytes: every expert starts its K walk at another
block and wraps round, in the tile kernel and in the persistent walk.  Scales that differ from block to block, so that a
scale taken from the wrong block shows."""
import numpy as np
import pytest
import torch

from oracle import moe as om
from tests.test_moe_gpu import _moe_case
from tests.test_widened_gpu import _dev_w, _moe_weights
from tests.util import assert_gemm_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("M,H,I,E,topk,block_m", [
    (100, 4096, 256, 12, 2, 64),    # tile kernel; experts 7 and up start past the end and wrap (32 K blocks, 5 apart)
    (90, 512, 4096, 3, 2, 128),     # the second GEMM's K
    (40, 8192, 128, 14, 1, 64),     # 64 K blocks
    (3000, 4096, 512, 8, 3, 128),   # persistent walk (first GEMM: four column tiles of some 75 blocks)
    (4000, 4096, 512, 8, 3, 192),
])
def test_block_scaled(dev, int8, M, H, I, E, topk, block_m):
    from tests.util import moe_layer as fused_moe

    print(f"pitch M={M} H={H} I={I} E={E} block_m={block_m} int8={int8}", flush=True)
    x, w13q, w13s, w2q, w2s, tw, ti = _moe_case(M, H, I, E, topk, M + H, dst="int8" if int8 else "fp8")
    rng = np.random.default_rng(M)
    w13s = (w13s * rng.uniform(0.25, 2, w13s.shape)).astype(np.float32)
    w2s = (w2s * rng.uniform(0.25, 2, w2s.shape)).astype(np.float32)
    ref = om.fused_moe_block_fp8(x, w13q, w2q, w13s, w2s, tw, ti, quant_form="reciprocal", int8=int8)
    conv = lambda a: torch.from_numpy(a).to(dev) if int8 else torch.from_numpy(a).to(dev).view(torch.float8_e4m3fn)  # noqa: E731
    kw = {"use_int8_w8a8": True} if int8 else {"use_fp8_w8a8": True}
    out = fused_moe(x.to(dev), conv(w13q), conv(w2q), (tw.to(dev), ti.to(dev), None), w1_scale=torch.from_numpy(w13s).to(dev),
                    w2_scale=torch.from_numpy(w2s).to(dev), block_shape=[128, 128], config={"BLOCK_SIZE_M": block_m}, **kw)
    assert_gemm_close(out, ref.float(), f"pitch M={M} H={H} I={I} block_m={block_m}")


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("M,H,I,E,topk", [(100, 4096, 256, 12, 2), (90, 512, 4096, 3, 2)])
def test_row_scaled(dev, int8, M, H, I, E, topk):
    from tests.util import moe_layer as fused_moe

    g = torch.Generator().manual_seed(M + H)
    x = torch.randn(M, H, generator=g).to(torch.bfloat16)
    q13, s13, q2, s2 = _moe_weights(E, I, H, g, "int8" if int8 else "fp8")
    tw, ti = om.topk_softmax(torch.randn(M, E, generator=g), topk, True)
    tw, ti = torch.as_tensor(tw), torch.as_tensor(ti)
    ref = om.fused_moe_row_scaled(x, q13, q2, s13, s2, tw, ti, int8=int8)
    kw = dict(use_int8_w8a8=True) if int8 else dict(use_fp8_w8a8=True)
    out = fused_moe(x.to(dev), _dev_w(q13, dev, int8), _dev_w(q2, dev, int8), (tw.to(dev), ti.to(dev), None),
                    w1_scale=torch.from_numpy(s13).to(dev), w2_scale=torch.from_numpy(s2).to(dev), per_channel_quant=True,
                    **kw)
    assert_gemm_close(out, ref.float(), f"pitch, row scales M={M} H={H} I={I} int8={int8}")
