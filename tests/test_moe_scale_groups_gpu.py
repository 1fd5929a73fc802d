"""The persistent MoE walk fetches activation scales in groups of four K blocks: numbers of K blocks around the group, whole
and padded rows, walks that start inside a group and wrap.  Scales that differ from block to block and from row to row, so
that one taken from the wrong place shows."""
import numpy as np
import pytest
import torch

from oracle import moe as om
from tests.test_moe_gpu import _moe_case
from tests.util import assert_gemm_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block_m", [128, 192])
@pytest.mark.parametrize("M,H,I,E,topk", [
    (2200, 256, 640, 24, 4),    # 2 and 5 K blocks: one group of two; a whole group and a padded one
    (1500, 384, 768, 32, 4),    # 3 and 6
    (1500, 512, 1152, 16, 5),   # 4 and 9: rows of one whole group; two and one block of a third
    (1100, 1152, 512, 24, 6),   # 9 and 4
    (3000, 4096, 384, 10, 3),   # 32, the walk turned by 5 blocks per expert; 3
])
def test_scale_groups(dev, M, H, I, E, topk, block_m):
    from tests.util import moe_layer as fused_moe

    print(f"scale groups M={M} H={H} I={I} E={E} block_m={block_m}", flush=True)
    x, w13q, w13s, w2q, w2s, tw, ti = _moe_case(M, H, I, E, topk, M + H)
    rng = np.random.default_rng(M)
    x = (x.float() * torch.from_numpy(rng.uniform(0.25, 4, (M, H // 128)).astype(np.float32)).repeat_interleave(128, 1)).to(x.dtype)
    w13s = (w13s * rng.uniform(0.25, 2, w13s.shape)).astype(np.float32)
    w2s = (w2s * rng.uniform(0.25, 2, w2s.shape)).astype(np.float32)
    ref = om.fused_moe_block_fp8(x, w13q, w2q, w13s, w2s, tw, ti, quant_form="reciprocal")
    conv = lambda a: torch.from_numpy(a).to(dev).view(torch.float8_e4m3fn)  # noqa: E731
    out = fused_moe(x.to(dev), conv(w13q), conv(w2q), (tw.to(dev), ti.to(dev), None), w1_scale=torch.from_numpy(w13s).to(dev),
                    w2_scale=torch.from_numpy(w2s).to(dev), block_shape=[128, 128], config={"BLOCK_SIZE_M": block_m},
                    use_fp8_w8a8=True)
    assert_gemm_close(out, ref.float(), f"scale groups M={M} H={H} I={I} block_m={block_m}")
