"""Sizes of zero that the native host code divides by: an error, not the end of the process.  Nothing is launched, so the
tensors lie on the CPU; the operators, which take device tensors only, get fake ones through their device entry."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

FP8 = torch.float8_e4m3fn


def _quantise(op, hidden, group, *extra):
    with FakeTensorMode():
        x = torch.empty(4, hidden, dtype=torch.bfloat16, device="cuda")
        q = torch.empty(4, hidden, dtype=FP8, device="cuda")
        s = torch.empty(4, 1, device="cuda")
    device_entry = torch._C.DispatchKeySet(torch._C.DispatchKey.CUDA)
    op.redispatch(device_entry, x, q, s, group, 1e-10, -448.0, 448.0, False, *extra)


@pytest.mark.parametrize("hidden,group", [(0, 128), (128, 0), (128, -128)])
def test_group_quant_of_no_columns_or_no_group(hidden, group):
    import sglang_amd  # noqa: F401

    with pytest.raises(RuntimeError, match="must be positive"):
        _quantise(torch.ops.sgl_kernel.sgl_per_token_group_quant_8bit.default, hidden, group)


@pytest.mark.parametrize("group", [0, -128])
def test_group_quant_v2_of_no_group(group):
    import sglang_amd  # noqa: F401

    with pytest.raises(RuntimeError, match="must be positive"):
        _quantise(torch.ops.sgl_kernel.sgl_per_token_group_quant_8bit_v2.default, 128, group, False, None)


def _moe_operands(n, block):
    ids = torch.zeros(16, dtype=torch.int32)
    groups = -(-128 // max(block, 1))
    return (torch.zeros(4, 128).to(FP8), torch.ones(4, groups), torch.zeros(2, n, 128).to(FP8),
            torch.ones(2, max(-(-n // max(block, 1)), 1), groups), torch.zeros(4, n, dtype=torch.bfloat16), None, ids,
            ids[:1], ids[:1], False, 1)


@pytest.mark.parametrize("n,block_m", [(0, 16), (128, 0), (128, -16)])
def test_moe_gemm_of_no_columns_or_no_rows_per_block(n, block_m):
    from sglang_amd import ops

    with pytest.raises(RuntimeError, match="must be positive"):
        ops.fused_moe_block_fp8_gemm_(*_moe_operands(n, 128), block_m)


@pytest.mark.parametrize("n,block_m,block_shape", [(0, 16, [64, 64]), (128, 0, [64, 64]), (128, 16, [0, 64]),
                                                   (128, 16, [64, 0]), (128, 0, None), (0, 16, None)])
def test_generic_moe_gemm_of_no_columns_rows_or_scale_block(n, block_m, block_shape):
    from sglang_amd import ops

    with pytest.raises(RuntimeError, match="must be positive"):
        ops.fused_moe_gemm_any_(*_moe_operands(n, 64), block_m, block_shape=block_shape)


def test_moe_kernel_configuration_without_a_block_height(monkeypatch):
    """The public caller: BLOCK_SIZE_M = 0 in the launch configuration."""
    import importlib

    module = importlib.import_module("sglang_amd.moe_runner.fused_moe")
    a, a_scale, b, b_scale, c, _, ids, expert, post, *_ = _moe_operands(128, 128)
    monkeypatch.setattr(module, "_quantise_activations", lambda *args: (a, a_scale))  # the quantiser needs a device
    with pytest.raises(RuntimeError, match="block_m must be positive"):
        module.invoke_fused_moe_kernel(torch.zeros(4, 128, dtype=torch.bfloat16), b, c, b_scale, None, ids, expert, post,
                                       False, 1, {"BLOCK_SIZE_M": 0}, [128, 128])


@pytest.mark.parametrize("shape", [(0, 2), (0,), (0, 0), (0, 5)])
def test_prequantised_linear_refuses_scales_of_no_rows(shape):
    from sglang_amd.quantization.fp8_utils import aiter_w8a8_block_fp8_linear

    q, w = (torch.zeros(rows, 256).to(torch.float8_e4m3fn) for rows in (0, 256))
    with pytest.raises(RuntimeError, match="reshape tensor of 0 elements"):
        aiter_w8a8_block_fp8_linear(q, w, [128, 128], torch.ones(2, 2), input_scale=torch.empty(shape))
