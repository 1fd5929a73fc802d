"""Row-scaled GEMMs that split K: scales and bias of four columns are read as one piece where they are aligned, one by one
where they are not -- the same bits either way, and the right ones."""
import pytest
import torch

from oracle import gemm as og
from tests.util import assert_gemm_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("M,N,K", [(65, 264, 4096), (130, 512, 16384), (300, 1000, 4096)])
@pytest.mark.parametrize("bias", [False, True])
def test_alignment_of_scales_and_bias(dev, int8, M, N, K, bias):
    import sglang_amd as sa
    from sglang_amd._lib import lib

    assert lib.sglamd_gemm_workspace_bytes(M, N, K) > 0, "this shape is meant to split K"
    g = torch.Generator().manual_seed(M + N)
    if int8:
        a, b = (torch.randint(-127, 128, s, generator=g, dtype=torch.int8) for s in ((M, K), (N, K)))
    else:
        a, b = ((torch.randn(s, generator=g) * 50).clamp(-448, 448).to(torch.float8_e4m3fn) for s in ((M, K), (N, K)))
    s_a, s_b = torch.rand(M, 1, generator=g) * 1e-2, torch.rand(N, 1, generator=g) * 1e-2
    bi = torch.randn(N, generator=g).to(torch.bfloat16) if bias else None
    mm, ref_mm = (sa.int8_scaled_mm, og.int8_scaled_mm) if int8 else (sa.fp8_scaled_mm, og.fp8_scaled_mm)
    outs = []
    for off in (0, 1):  # the second time a view one element into its storage
        sb_d = torch.cat([torch.zeros(off, 1), s_b]).to(dev)[off:]
        bi_d = None if bi is None else torch.cat([torch.zeros(off, dtype=bi.dtype), bi]).to(dev)[off:]
        outs.append(mm(a.to(dev), b.to(dev).t(), s_a.to(dev), sb_d, torch.bfloat16, bi_d))
    assert torch.equal(*outs)
    raw = lambda t: t.numpy() if int8 else t.view(torch.uint8).numpy()  # noqa: E731
    ref = ref_mm(raw(a), raw(b), s_a.numpy().reshape(-1), s_b.numpy().reshape(-1), out_dtype=torch.bfloat16, bias=bi)
    assert_gemm_close(outs[0], ref.float(), f"split-K rows M={M} N={N} K={K}")
