"""INT8 rows round halves away from zero, and the scaled value is rounded to fp32 before it is rounded to an integer: products
that end on and beside a half, in every kernel that quantises a 16-bit row (one piece to sixteen per lane)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,hidden", [(3, 256), (1500, 512), (1500, 1024), (5000, 2048), (600, 4096), (600, 8192), (5, 16384),
                                         (513, 16392), (1024, 28672), (1025, 32768)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_halves_round_away_from_zero(dev, rows, hidden, dtype):
    from sglang_amd.quantization.int8_kernel import per_token_quant_int8

    g = torch.Generator().manual_seed(rows + hidden)
    x = torch.randint(-254, 255, (rows, hidden), generator=g).float() / 2  # with a maximum of 127 the halves are exact
    x[:, 0] = 127.0
    x[1::3] *= 1.375  # and with others they are not
    x = x.to(dtype)
    print(f"INT8 rows {rows} x {hidden} {dtype}", flush=True)
    q, s = per_token_quant_int8(x.to(dev))
    amax = x.float().abs().amax(1, keepdim=True)
    scaled = x.float() * (torch.tensor(127.0) / amax)
    whole = scaled.abs().floor()
    ref = torch.sign(scaled) * (whole + (scaled.abs() - whole >= 0.5))
    assert torch.equal(q.cpu().float(), ref)
    assert torch.allclose(s.cpu().view(-1), (amax / 127.0).view(-1), rtol=2e-7, atol=0)
