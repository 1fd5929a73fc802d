"""The MoE layer of one token runs as two GEMM launches: the pairs take the experts straight from topk_ids, the rows are
quantised in the workgroups, and the last pair to finish a column tile sums the tile.  Against the same token five times over,
which takes the general sequence: rows that fit few and many passes, and more than a chunk of them; fewer K blocks than the
ring; workgroups that walk several tiles; a row too long for LDS, which goes back to the launch in front."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,I,E,topk", [(256, 256, 4, 1), (384, 512, 8, 3), (7168, 256, 16, 8), (2176, 768, 32, 32),
                                        (1408, 8320, 32, 32), (33024, 256, 4, 4)])
@pytest.mark.parametrize("ids_dtype,dtype,scaling", [(torch.int32, torch.bfloat16, None), (torch.int64, torch.float16, 2.5)])
def test_one_token_is_a_row_of_the_general_layer(dev, H, I, E, topk, ids_dtype, dtype, scaling):
    from tests.util import moe_layer

    g = torch.Generator(device=dev).manual_seed(H + I + topk)
    fp8 = lambda *shape: (torch.randint(0, 256, shape, generator=g, device=dev, dtype=torch.uint8) & 0xB7).view(torch.float8_e4m3fn)
    w13, w2 = fp8(E, 2 * I, H), fp8(E, H, I)
    s13 = torch.rand(E, 2 * I // 128, H // 128, generator=g, device=dev) * (0.4 / H ** 0.5) + 0.01 / H ** 0.5
    s2 = torch.rand(E, H // 128, I // 128, generator=g, device=dev) / I ** 0.5
    x = torch.randn(1, H, generator=g, device=dev).to(dtype)
    ids = torch.randperm(E, generator=g, device=dev)[:topk].view(1, topk)
    ids[0, topk // 2] = -1 if topk > 1 else ids[0, 0]  # an expert that lives elsewhere
    w = torch.rand(1, topk, generator=g, device=dev)
    print(f"one token H={H} I={I} E={E} topk={topk} {dtype}", flush=True)
    kw = dict(use_fp8_w8a8=True, w1_scale=s13, w2_scale=s2, block_shape=[128, 128], routed_scaling_factor=scaling)
    many = moe_layer(x.repeat(5, 1), w13, w2, (w.repeat(5, 1), ids.to(ids_dtype).repeat(5, 1), None), **kw)[:1].float()
    for _ in range(3):  # arrivals are counted from zero every time
        one = moe_layer(x, w13, w2, (w, ids.to(ids_dtype), None), **kw).float()
        # sums in another order: a bit of the 16-bit intermediate, and with it a step (1/16) of single quantised values
        assert torch.isfinite(one).all()
        assert (one - many).abs().max() <= 0.01 * many.abs().max()
