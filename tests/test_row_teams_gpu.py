"""Many short rows quantised several to a workgroup: at the edges of the row lengths each team takes, with a last workgroup
that is partly empty; and the row-scaled MoE layer at the sizes where its prologue and its activations do the same."""
import numpy as np
import pytest
import torch

from oracle import moe as om
from oracle import quant as oq
from tests.test_widened_gpu import _dev_w, _moe_weights
from tests.util import assert_gemm_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,hidden", [(1023, 256), (1024, 8), (1029, 256), (1030, 264), (1027, 512), (1025, 520), (1026, 1024),
                                         (1024, 1032), (4095, 2048), (4097, 1032), (4098, 2048), (4099, 2056)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_short_rows(dev, rows, hidden, dtype):
    from sglang_amd.quantization.fp8_kernel import sglang_per_token_quant_fp8
    from sglang_amd.quantization.int8_kernel import per_token_quant_int8

    g = torch.Generator().manual_seed(rows + hidden)
    x = torch.randn(rows, hidden, generator=g).to(dtype)
    x[:, -1] += torch.arange(rows) % 7  # maxima in the last piece too
    x[rows - 1], x[3] = 0, 0
    q, s = sglang_per_token_quant_fp8(x.to(dev))
    rq, rs = oq.per_token_quant_fp8(x)
    assert np.array_equal(q.cpu().view(torch.uint8).numpy(), rq) and np.array_equal(s.cpu().numpy(), rs.reshape(rows, 1))
    q, s = per_token_quant_int8(x.to(dev))
    rq, rs = oq.per_token_quant_int8(x)
    assert np.array_equal(q.cpu().numpy(), rq) and np.array_equal(s.cpu().numpy(), rs.reshape(rows, 1))


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("M,H,I,E,topk", [(1025, 256, 128, 4, 1), (1026, 2176, 256, 4, 1), (600, 256, 640, 4, 2)])
def test_row_scaled_layer(dev, int8, M, H, I, E, topk):
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
    assert_gemm_close(out, ref.float(), f"row teams M={M} H={H} I={I} int8={int8}")
