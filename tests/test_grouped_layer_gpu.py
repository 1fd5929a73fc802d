"""The expert-major MoE layer in one call against its separate operators (same bits, same tables), at every sorted-block
height, and the grouped GEMM's schedule when several workgroups fill it."""
import types

import numpy as np
import pytest
import torch

from oracle import moe as om

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,H,I,E,topk", [(1, 384, 256, 8, 2), (4, 256, 128, 4, 4), (40, 256, 384, 8, 2), (50, 512, 256, 8, 2),
                                         (300, 256, 256, 8, 2), (700, 256, 128, 6, 3), (4100, 256, 128, 300, 5)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_one_call_equals_the_separate_operators(dev, monkeypatch, M, H, I, E, topk, dtype):
    from sglang_amd.moe_runner import cutlass_moe

    g = torch.Generator(device=dev).manual_seed(M + H + E)
    codes = lambda *s: (torch.randn(*s, generator=g, device=dev) * 100).clamp(-448, 448).to(torch.float8_e4m3fn)  # noqa: E731
    scale = lambda *s: torch.rand(*s, generator=g, device=dev) * 2e-4 + 1e-5  # noqa: E731
    x = torch.randn(M, H, generator=g, device=dev).to(dtype)
    w13, w2 = codes(E, 2 * I, H), codes(E, H, I)
    s13, s2 = scale(E, 2 * I // 128, H // 128), scale(E, H // 128, I // 128)
    tw, ti = torch.topk(torch.softmax(torch.randn(M, E, generator=g, device=dev), dim=-1), topk, dim=-1)
    ti = ti.to(torch.int32).contiguous()

    def call():
        i32 = lambda *s: torch.full(s, -1, device=dev, dtype=torch.int32)  # noqa: E731
        i64 = lambda v: torch.full((E,), v, device=dev, dtype=torch.int64)  # noqa: E731
        tables = i32(E + 1), i32(E, 3), i32(E, 3)
        out = cutlass_moe.cutlass_fused_experts_fp8(
            x, w13.transpose(1, 2), w2.transpose(1, 2), s13.transpose(1, 2), s2.transpose(1, 2), tw, ti, i64(H), i64(2 * I),
            i64(I), i64(H), torch.empty(1 << 22, device=dev, dtype=torch.uint8), *(i64(0) for _ in range(5)), *tables)
        return out, [t.cpu().numpy() for t in tables]

    one, tables = call()
    monkeypatch.setattr(cutlass_moe, "_C", types.SimpleNamespace(moe_grouped_layer=lambda *a: None))
    steps, step_tables = call()
    assert torch.isfinite(one.float()).all() and torch.equal(one, steps)
    want = om.prepare_moe_input(ti.cpu().numpy(), E, I, H)
    for got, again, ref in zip(tables, step_tables, (want[0], want[2], want[3])):
        assert np.array_equal(got, again) and np.array_equal(got, ref)
