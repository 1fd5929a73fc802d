"""silu_rounded over every 16-bit gate value, and the fused SiLU*mul group quantisation where its scale words are whole,
ragged and shared between workgroups."""
import numpy as np
import pytest
import torch

from oracle import quant as oq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_silu_of_every_16_bit_value(dev, dtype):
    from sglang_amd import silu_and_mul

    gate = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(dtype).view(64, 1024)
    out = silu_and_mul(torch.cat([gate, torch.ones_like(gate)], dim=1).to(dev)).cpu()
    x = gate.double()
    exact = torch.where(x == -np.inf, torch.full_like(x, np.nan), x * torch.sigmoid(x))
    nan = torch.isnan(exact)
    assert torch.equal(torch.isnan(out.double()), nan)
    # the fp32 value under the 16-bit rounding is within 8 parts in 2^23 of the true one (exp overflows past -88: zero)
    slack = torch.where(torch.isinf(exact), torch.zeros_like(exact), 1e-6 * exact.abs() + 1e-37)
    low, high = (exact - slack).to(dtype).double(), (exact + slack).to(dtype).double()
    got = out.double()
    ok = nan | ((got >= low) & (got <= high)) | ((x < -87) & (got == 0))
    assert bool(ok.all()), [(float(a), float(b)) for a, b in zip(x[~ok][:4], got[~ok][:4])]


def _defined_silu(gate):
    """x / (1 + expf(-x)) through the device's expf and the IEEE division, rounded to the gate's type."""
    x = gate.float()
    return (x / (1.0 + torch.exp(-x))).to(gate.dtype)


def _every_gate(dtype, dev):
    return torch.arange(65536, dtype=torch.int32).to(torch.int16).view(dtype).to(dev)


@pytest.mark.parametrize("up", [1.0, -0.73, 0.0])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_silu_has_the_bits_of_the_defined_form(dev, dtype, up):
    """The fast form and its fallback next to rounding boundaries, against the form that defines the value."""
    from sglang_amd import silu_and_mul

    gate = _every_gate(dtype, dev).view(64, 1024)
    ups = torch.full_like(gate, up)
    got = silu_and_mul(torch.cat([gate, ups], dim=1))
    want = (_defined_silu(gate).float() * ups.float()).to(dtype)
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(got), nan)
    bad = (got.view(torch.int16) != want.view(torch.int16)) & ~nan
    assert not bool(bad.any()), [(float(a), float(b), float(c)) for a, b, c in
                                 zip(gate[bad][:4], got[bad][:4], want[bad][:4])]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_fused_quantisation_has_the_bits_of_the_defined_form(dev, dtype):
    """Each gate alone in a group of 16 (the other products are zeros): the group's scale and byte show all of its bits."""
    from sglang_amd.quantization.fp8_kernel import sglang_per_token_group_quant_fp8

    gate = _every_gate(dtype, dev)
    gate = torch.where(torch.isfinite(gate), gate, torch.ones_like(gate))
    x = torch.zeros(64, 2, 1024, 16, dtype=dtype, device=dev)
    place = torch.arange(65536, device=dev).view(64, 1024, 1) % 16
    x[:, 0].scatter_(2, place, gate.view(64, 1024, 1))
    x[:, 1].scatter_(2, place, torch.ones_like(gate).view(64, 1024, 1))
    x = x.view(64, 2 * 16384)
    q, s = sglang_per_token_group_quant_fp8(x, 16, fuse_silu_and_mul=True)
    act = _defined_silu(x[:, :16384]) * x[:, 16384:]
    rq, rs, _ = oq.group_quant(act.cpu(), 16, form="reciprocal")
    assert np.array_equal(s.cpu().numpy(), rs)
    assert np.array_equal(q.cpu().view(torch.uint8).numpy(), rq)


@pytest.mark.parametrize("layout", ["row", "col", "ue8m0"])
@pytest.mark.parametrize("rows,hidden", [(1, 128), (7, 512), (5, 640), (33, 1024), (3, 4608)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_silu_group_quant_layouts(dev, layout, rows, hidden, dtype):
    """Against the plain quantisation of what silu_and_mul stores: same bytes, same scales, whatever the layout."""
    from sglang_amd import silu_and_mul
    from sglang_amd.quantization.fp8_kernel import sglang_per_token_group_quant_fp8

    g = torch.Generator().manual_seed(rows + hidden)
    x = (torch.randn(rows, 2 * hidden, generator=g) * 3).to(dtype)
    kw = dict(column_major_scales=layout != "row", scale_tma_aligned=layout == "ue8m0", scale_ue8m0=layout == "ue8m0")
    q, s = sglang_per_token_group_quant_fp8(x.to(dev), 128, fuse_silu_and_mul=True, **kw)
    act = silu_and_mul(x.to(dev)).cpu()
    rq, rs, ebytes = oq.group_quant(act, 128, form="reciprocal", scale_ue8m0=layout == "ue8m0")
    assert np.array_equal(q.cpu().view(torch.uint8).numpy(), rq)
    want = oq.pack_ue8m0(ebytes) if layout == "ue8m0" else rs
    assert np.array_equal(s.cpu().numpy(), want)
