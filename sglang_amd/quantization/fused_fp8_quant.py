"""Fused RMSNorm + per-token-group FP8 quantisation with the call signature of
aiter.ops.triton.fused_fp8_quant.fused_rms_fp8_group_quant, as the reference uses it on gfx95
(python/sglang/srt/layers/communicator.py:552-624,
python/sglang/srt/models/deepseek_common/attention_forward_methods/forward_mla.py:175-203): the (fp8, scale)
pair it returns is what the block-FP8 linears accept as a pre-quantised input
(python/sglang/srt/layers/quantization/fp8.py:794-802)."""
from typing import Optional, Tuple

import torch

from ..ops import _C


def fused_rms_fp8_group_quant(
    inp1: torch.Tensor,
    inp1_weight: torch.Tensor,
    inp1_epsilon: float,
    inp2: Optional[torch.Tensor] = None,
    inp2_weight: Optional[torch.Tensor] = None,
    inp2_epsilon: Optional[float] = None,
    group_size: int = 128,
    dtype_quant: torch.dtype = torch.float8_e4m3fn,
    res1: Optional[torch.Tensor] = None,
    output_unquantized_inp1: bool = False,
) -> Tuple[Tuple[torch.Tensor, torch.Tensor], Optional[torch.Tensor], Optional[torch.Tensor], Optional[torch.Tensor]]:
    """((y1_q [M, N1] fp8, y1_s [M, ceil(N1/128)] fp32), y1 or None, y2 or None, inp1 + res1 or None).
    inp1 [M, N1] and inp2 [M, N2] half/bfloat16, rows contiguous (a row stride is fine); res1 like inp1;
    weights fp32 or the activation dtype.  Everything is computed in fp32 from one read of each row; y1 is
    quantised before it is rounded to the activation dtype."""
    if dtype_quant != torch.float8_e4m3fn:
        raise NotImplementedError("only torch.float8_e4m3fn is implemented as dtype_quant")
    if group_size != 128:
        raise NotImplementedError("only group_size 128 is implemented")
    y1_q, y1_s, y1, y2, res_out = _C.fused_rms_group_quant(inp1, inp1_weight, inp1_epsilon, inp2, inp2_weight,
                                                           inp2_epsilon, res1, output_unquantized_inp1)
    return (y1_q, y1_s), y1, y2, res_out
