"""The quantisers under a tracer: their operators return nothing, so a compiler or a fake-tensor mode follows the wrappers
down to one operator node each without a fake implementation.  Nothing is launched."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from sglang_amd.quantization import fp8_kernel as fk
from sglang_amd.quantization import int8_kernel as ik

FP8 = torch.float8_e4m3fn
CASES = {
    "fp8": (lambda x: fk.sglang_per_token_group_quant_fp8(x, 128), "v2", FP8, (6, 256), (6, 2), (2, 1)),
    "fp8_columns": (lambda x: fk.sglang_per_token_group_quant_fp8(x, 128, column_major_scales=True), "v2", FP8, (6, 256),
                    (6, 2), (1, 6)),
    "fp8_aligned": (lambda x: fk.sglang_per_token_group_quant_fp8(x, 64, column_major_scales=True, scale_tma_aligned=True),
                    "v2", FP8, (6, 256), (6, 4), (1, 8)),
    "fp8_ue8m0": (lambda x: fk.sglang_per_token_group_quant_fp8(x, 128, column_major_scales=True, scale_tma_aligned=True,
                                                                scale_ue8m0=True), "v2", FP8, (6, 256), (6, 1), (1, 8)),
    "fp8_silu": (lambda x: fk.sglang_per_token_group_quant_fp8(x, 128, fuse_silu_and_mul=True), "v2", FP8, (6, 128),
                 (6, 1), (1, 1)),
    "fp8_v1": (lambda x: fk.sglang_per_token_group_quant_fp8(x, 128, enable_v2=False), "8bit", FP8, (6, 256), (6, 2),
               (2, 1)),
    "fp8_rows": (lambda x: fk.sglang_per_token_quant_fp8(x), "per_token_quant_fp8", FP8, (6, 256), (6, 1), (1, 1)),
    "int8": (lambda x: fk.sglang_per_token_group_quant_int8(x, 128), "v2", torch.int8, (6, 256), (6, 2), (2, 1)),
    "int8_wrapper": (lambda x: ik.per_token_group_quant_int8(x, 128), "v2", torch.int8, (6, 256), (6, 2), (2, 1)),
}


@pytest.mark.parametrize("name", CASES)
def test_one_operator_node_under_the_compiler(name):
    fn, op, *_ = CASES[name]
    nodes = []

    def backend(graph, inputs):
        nodes.extend(str(n.target) for n in graph.graph.nodes if "sgl_kernel" in str(n.target))
        return lambda *args: tuple(o.meta["example_value"].shape for o in graph.graph.output_node().args[0])

    torch._dynamo.reset()
    torch.compile(fn, backend=backend, fullgraph=True)(torch.zeros(6, 256, dtype=torch.bfloat16))
    assert len(nodes) == 1 and op in nodes[0], nodes


@pytest.mark.parametrize("name", CASES)
def test_shapes_in_a_fake_tensor_mode(name):
    fn, _, dtype, q_shape, s_shape, s_stride = CASES[name]
    with FakeTensorMode():
        q, s = fn(torch.empty(6, 256, dtype=torch.bfloat16, device="cuda"))
    assert q.device.type == "cuda" and q.dtype == dtype and q.shape == q_shape
    assert s.shape == s_shape and s.stride() == s_stride


def test_whole_layers_leave_fake_tensors_to_their_operators():
    from sglang_amd import _C

    with FakeTensorMode():
        x = torch.empty(6, 256, dtype=torch.bfloat16, device="cuda")
        x_q, x_s = torch.empty(6, 256, dtype=FP8, device="cuda"), torch.empty(6, 2, device="cuda")
        w, ws = torch.empty(384, 256, dtype=FP8, device="cuda"), torch.empty(3, 2, device="cuda")
        rows = torch.empty(384, 1, device="cuda")
        w1, w2 = torch.empty(4, 256, 256, dtype=FP8, device="cuda"), torch.empty(4, 256, 128, dtype=FP8, device="cuda")
        s1, s2 = torch.empty(4, 2, 2, device="cuda"), torch.empty(4, 2, 1, device="cuda")
        tw, ids = torch.empty(6, 2, device="cuda"), torch.empty(6, 2, dtype=torch.int32, device="cuda")
        table = torch.empty(16, dtype=torch.int32, device="cuda")
    assert _C.block_linear(x, w, ws, None) is None
    assert _C.block_matmul(x_q, w, x_s, ws, torch.bfloat16, None) is None
    assert _C.row_linear(x, w.t(), rows, None) is None
    assert _C.moe_layer(x, w1, w2, s1, s2, None, None, tw, ids, True, False, False, 1.0, 0) is None
    assert _C.moe_grouped_layer(x, w1.mT, w2.mT, s1.mT, s2.mT, tw, ids, table, table, table, None) is None
