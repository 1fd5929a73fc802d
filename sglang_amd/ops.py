"""The quantized-linear operators: ``torch.ops.sgl_kernel`` with the reference's schema strings
(sgl-kernel/csrc/common_extension.cc:76-77,116-142,164-168,180-181) and the launchers that the Python wrappers of this
package use.

Both live in the native module ``_C`` (csrc/host.cpp): it unpacks the tensors into raw pointers / sizes / element
strides, takes the current HIP stream and calls the C-ABI library.  Its checks raise RuntimeError with the reference's
message text before anything is launched, mirroring its TORCH_CHECKs.  Nothing there allocates except the
value-returning GEMMs, which allocate their output like the reference does, and split-K or layer scratch.

This module must be the only provider of the ``sgl_kernel`` namespace in the process: a second library defining the
same schemas is a hard error in the dispatcher.
"""
import torch  # noqa: F401  (_C is linked against it)

from . import _lib  # the library _C calls: loaded first, from wherever SGLAMD_LIBRARY says
from . import _C

_C.set_error_type(_lib.SglAmdError)

from ._C import (  # noqa: E402,F401
    block_scaled_mm_any_,
    fused_moe_block_fp8_,
    fused_moe_block_fp8_gemm_,
    fused_moe_block_fp8_workspace_bytes,
    fused_moe_gemm_any_,
    per_token_quant_int8_,
    static_quant_fp8_,
    tensor_absmax_scale_,
    ue8m0_unpack_,
    w8a8_block_fp8_matmul_,
    w8a8_block_int8_matmul_,
)

_K = torch.ops.sgl_kernel
sgl_per_token_group_quant_8bit = _K.sgl_per_token_group_quant_8bit.default
sgl_per_token_group_quant_8bit_v2 = _K.sgl_per_token_group_quant_8bit_v2.default
sgl_per_token_quant_fp8 = _K.sgl_per_token_quant_fp8.default
fp8_blockwise_scaled_mm = _K.fp8_blockwise_scaled_mm.default
fp8_scaled_mm = _K.fp8_scaled_mm.default
int8_scaled_mm = _K.int8_scaled_mm.default
topk_softmax = _K.topk_softmax.default
topk_sigmoid = _K.topk_sigmoid.default
moe_align_block_size = _K.moe_align_block_size.default
silu_and_mul = _K.silu_and_mul.default
gelu_tanh_and_mul = _K.gelu_tanh_and_mul.default
gelu_and_mul = _K.gelu_and_mul.default
moe_sum_reduce = _K.moe_sum_reduce.default
prepare_moe_input = _K.prepare_moe_input.default
shuffle_rows = _K.shuffle_rows.default
apply_shuffle_mul_sum = _K.apply_shuffle_mul_sum.default
fp8_blockwise_scaled_grouped_mm = _K.fp8_blockwise_scaled_grouped_mm.default
es_fp8_blockwise_scaled_grouped_mm = _K.es_fp8_blockwise_scaled_grouped_mm.default

_is_dynamo_compiling, _Tensor = torch.compiler.is_dynamo_compiling, torch.Tensor


def eager(x: torch.Tensor) -> bool:
    """Whether the whole-call functions of _C may be tried on `x` at all: a compiler that traces the caller cannot follow
    them, and a tensor subclass would not get its own type back.  They look at the rest themselves (dispatch modes, which
    the other tracers are, transforms, autograd) and answer None; the caller then goes through the operators."""
    return not _is_dynamo_compiling() and type(x) is _Tensor
