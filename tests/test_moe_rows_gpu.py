"""Row-scaled fused-MoE layers (per-channel FP8 / INT8 experts) on the streaming and tile kernels: every sorted-block
height the layer picks by itself, column counts that leave a tile partly filled, ids of -1, int64 ids; and the per-token
quantisers at the edges of the shapes they cut a row into."""
import numpy as np
import pytest
import torch

from oracle import moe as om
from oracle import quant as oq
from tests.test_widened_gpu import _dev_w, _moe_weights
from tests.util import assert_gemm_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("M,H,I,E,topk,bias", [
    (3, 384, 128, 4, 2, True),     # streaming kernel, 16-slot blocks
    (61, 640, 384, 4, 2, False),   # 64-slot blocks, a last column tile of 128
    (90, 256, 256, 3, 3, True),    # 128-slot blocks, more than one per expert for some
    (150, 384, 128, 2, 2, False),  # 192-slot blocks
])
def test_row_scaled_layer_at_every_block_height(dev, int8, M, H, I, E, topk, bias):
    from tests.util import moe_layer as fused_moe

    g = torch.Generator().manual_seed(7 * M + H)
    x = torch.randn(M, H, generator=g).to(torch.bfloat16)
    q13, s13, q2, s2 = _moe_weights(E, I, H, g, "int8" if int8 else "fp8")
    b1 = (torch.randn(E, 2 * I, generator=g) * 0.1).to(torch.bfloat16) if bias else None
    b2 = (torch.randn(E, H, generator=g) * 0.1).to(torch.bfloat16) if bias else None
    tw, ti = om.topk_softmax(torch.randn(M, E, generator=g), topk, True)
    tw, ti = torch.as_tensor(tw), torch.as_tensor(ti)
    ti[M // 2, 0] = -1  # an expert that lives elsewhere: contributes nothing
    ref = om.fused_moe_row_scaled(x, q13, q2, s13, s2, tw, ti, int8=int8, b1=b1, b2=b2)
    kw = dict(use_int8_w8a8=True) if int8 else dict(use_fp8_w8a8=True)
    d = lambda t: None if t is None else t.to(dev)  # noqa: E731
    for ids in (ti.to(torch.int32), ti.to(torch.int64)):
        out = fused_moe(d(x), _dev_w(q13, dev, int8), _dev_w(q2, dev, int8), (d(tw), d(ids), None), b1=d(b1), b2=d(b2),
                        w1_scale=torch.from_numpy(s13).to(dev), w2_scale=torch.from_numpy(s2).to(dev),
                        per_channel_quant=True, **kw)
        assert_gemm_close(out, ref.float(), f"row-scaled M={M} E={E} int8={int8} {ids.dtype}")


@pytest.mark.parametrize("rows,hidden", [(1, 8), (3, 2048), (2, 2056), (5, 8192), (2, 8200), (1, 16392), (3, 32768),
                                         (1, 32776), (520, 4096), (520, 8192), (515, 8200)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_per_token_quant_at_the_edges_of_its_row_shapes(dev, rows, hidden, dtype):
    from sglang_amd.quantization.fp8_kernel import sglang_per_token_quant_fp8
    from sglang_amd.quantization.int8_kernel import per_token_quant_int8

    g = torch.Generator().manual_seed(rows + hidden)
    x = torch.randn(rows, hidden, generator=g).to(dtype)
    x[0, -1] = 9.0  # the maximum of the first row in its last piece
    if rows > 1:
        x[1] = 0
    q, s = sglang_per_token_quant_fp8(x.to(dev))
    rq, rs = oq.per_token_quant_fp8(x)
    assert np.array_equal(q.cpu().view(torch.uint8).numpy(), rq) and np.array_equal(s.cpu().numpy(), rs.reshape(rows, 1))
    q, s = per_token_quant_int8(x.to(dev))
    rq, rs = oq.per_token_quant_int8(x)
    assert np.array_equal(q.cpu().numpy(), rq) and np.array_equal(s.cpu().numpy(), rs.reshape(rows, 1))
