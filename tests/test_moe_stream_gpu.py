"""The weight-streaming MoE tile kernel (gemm_moe_stream.h): experts with numbers of rows around the 32-row tile and the
block, idle experts, experts of several blocks, short and long K, walks that start inside a group of scales and wrap, widths
that do not fill the last column tile, in every scaling mode.  Scales that differ from block to block, so that one taken
from the wrong place shows."""
import numpy as np
import pytest
import torch

from oracle import moe as om
from tests.test_moe_gpu import _moe_case
from tests.test_widened_gpu import _dev_w, _moe_weights
from tests.util import assert_gemm_close

pytestmark = pytest.mark.gpu

COUNTS = [0, 1, 31, 32, 33, 63, 64, 65, 127, 128, 129, 200, 5, 16]


def _ids(E, g):
    """One expert per token, expert e named COUNTS[e % len] times; the tokens in random order."""
    ids = torch.cat([torch.full((COUNTS[e % len(COUNTS)],), e, dtype=torch.int32) for e in range(E)])
    return ids[torch.randperm(ids.numel(), generator=g)].view(-1, 1)


# enough (expert, column tile) pairs that both GEMMs have one tile per CU and more
SHAPES = [
    (70, 1024, 768),   # 8 and 6 K blocks: the fewest the kernel takes; 4 column tiles
    (60, 1152, 1152),  # 9 and 9: padded rows of scales; a half-filled column tile
    (32, 4096, 1024),  # 32 K blocks, the walk turned by 5 per expert
    (24, 2944, 4096),  # 23 and 32
]


@pytest.mark.parametrize("int8,E,H,I", [(False, *s) for s in SHAPES] + [(True, *s) for s in SHAPES[:2]])
def test_block_scaled(dev, int8, E, H, I, block_m=64):
    from tests.util import moe_layer as fused_moe

    g = torch.Generator().manual_seed(E + H)
    ti = _ids(E, g)
    M = ti.numel()
    print(f"moe stream M={M} H={H} I={I} E={E} block_m={block_m} int8={int8}", flush=True)
    x, w13q, w13s, w2q, w2s, tw, _ = _moe_case(M, H, I, E, 1, E + H, dst="int8" if int8 else "fp8")
    rng = np.random.default_rng(M)
    tw = torch.from_numpy(rng.uniform(0.25, 2, (M, 1)).astype(np.float32))
    w13s = (w13s * rng.uniform(0.25, 2, w13s.shape)).astype(np.float32)
    w2s = (w2s * rng.uniform(0.25, 2, w2s.shape)).astype(np.float32)
    x = (x.float() * torch.from_numpy(rng.uniform(0.25, 4, (M, H // 128)).astype(np.float32)).repeat_interleave(128, 1)).to(x.dtype)
    ref = om.fused_moe_block_fp8(x, w13q, w2q, w13s, w2s, tw, ti, quant_form="reciprocal", int8=int8)
    conv = lambda a: torch.from_numpy(a).to(dev) if int8 else torch.from_numpy(a).to(dev).view(torch.float8_e4m3fn)  # noqa: E731
    kw = {"use_int8_w8a8": True} if int8 else {"use_fp8_w8a8": True}
    out = fused_moe(x.to(dev), conv(w13q), conv(w2q), (tw.to(dev), ti.to(dev), None), w1_scale=torch.from_numpy(w13s).to(dev),
                    w2_scale=torch.from_numpy(w2s).to(dev), block_shape=[128, 128], config={"BLOCK_SIZE_M": block_m}, **kw)
    assert_gemm_close(out, ref.float(), f"moe stream H={H} I={I} block_m={block_m}")


@pytest.mark.parametrize("int8,E,H,I,block_m", [(True, *SHAPES[0], 64), (True, *SHAPES[2], 128), (False, *SHAPES[1], 64),
                                                (False, *SHAPES[1], 128), (True, *SHAPES[1], 128)])
def test_row_scaled(dev, int8, E, H, I, block_m):
    from sglang_amd import _C

    g = torch.Generator().manual_seed(E + H)
    ti = _ids(E, g)
    M = ti.numel()
    print(f"moe stream, row scales M={M} H={H} I={I} E={E} block_m={block_m} int8={int8}", flush=True)
    x = torch.randn(M, H, generator=g).to(torch.float16)
    q13, s13, q2, s2 = _moe_weights(E, I, H, g, "int8" if int8 else "fp8")
    tw = torch.rand(M, 1, generator=g) + 0.25
    ref = om.fused_moe_row_scaled(x, q13, q2, s13, s2, tw, ti, int8=int8)
    out = _C.moe_layer(x.to(dev), _dev_w(q13, dev, int8), _dev_w(q2, dev, int8), torch.from_numpy(s13).to(dev),
                       torch.from_numpy(s2).to(dev), None, None, tw.to(dev), ti.to(dev), False, int8, False, 1.0, block_m)
    assert_gemm_close(out, ref.float(), f"moe stream, row scales H={H} I={I} block_m={block_m}")


def test_ids_that_live_elsewhere(dev):
    """Pairs with the id -1 come as blocks of an expert that is not here: zeros, in both heights of row tile."""
    from tests.util import moe_layer as fused_moe

    M, H, I, E = 600, 1024, 1024, 64
    x, w13q, w13s, w2q, w2s, tw, ti = _moe_case(M, H, I, E, 2, 9)
    ti = ti.clone()
    ti[::5, 1] = -1
    ti[7::50] = -1
    ref = om.fused_moe_block_fp8(x, w13q, w2q, w13s, w2s, tw, ti, quant_form="reciprocal")
    conv = lambda a: torch.from_numpy(a).to(dev).view(torch.float8_e4m3fn)  # noqa: E731
    out = fused_moe(x.to(dev), conv(w13q), conv(w2q), (tw.to(dev), ti.to(dev), None), w1_scale=torch.from_numpy(w13s).to(dev),
                    w2_scale=torch.from_numpy(w2s).to(dev), block_shape=[128, 128], config={"BLOCK_SIZE_M": 64}, use_fp8_w8a8=True)
    assert_gemm_close(out, ref.float(), "moe stream, ids of -1")
    assert not out[7::50].any()


@pytest.mark.parametrize("mode,block_m", [("block_fp8", 64), ("row_int8", 64), ("row_int8", 128), ("row_fp8", 128)])
def test_slots_anywhere_in_a_block(dev, mode, block_m):
    """The grouped GEMMs take every slot below num_valid_tokens, wherever a caller's list has it: blocks whose tiles begin with
    padding, or hold nothing else in front of their rows, give the bits of the sorted list."""
    from sglang_amd.moe_runner.moe_align_block_size import moe_align_block_size
    from sglang_amd.ops import fused_moe_block_fp8_gemm_, fused_moe_gemm_any_

    E, N, K = 70, 1024, 1024
    g = torch.Generator().manual_seed(block_m)
    ti = _ids(E, g).to(dev)
    M = ti.numel()
    print(f"moe stream, slots anywhere mode={mode} block_m={block_m} M={M}", flush=True)
    int8 = mode.endswith("int8")
    q13, s13, _, _ = _moe_weights(E, N // 2, K, g, "int8" if int8 else "fp8")
    w = _dev_w(q13, dev, int8)
    a = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8).to(dev) if int8 else (
        torch.randn(M, K, generator=g).mul_(50).clamp_(-448, 448).to(dev).to(torch.float8_e4m3fn))
    tw = torch.rand(M, 1, generator=g).add_(0.25).to(dev)
    if mode == "block_fp8":
        sa, sb = torch.rand(M, K // 128, generator=g).to(dev), torch.rand(E, N // 128, K // 128, generator=g).to(dev)
    else:
        sa, sb = torch.rand(M, 1, generator=g).to(dev), torch.from_numpy(s13).to(dev)

    def gemm(slots, experts, post):
        c = torch.full((M, N), float("nan"), device=dev, dtype=torch.bfloat16)
        if mode == "block_fp8":
            fused_moe_block_fp8_gemm_(a, sa, w, sb, c, tw, slots, experts, post, True, 1, block_m)
        else:
            fused_moe_gemm_any_(a, sa, w, sb, c, tw, slots, experts, post, True, 1, block_m, block_shape=None, bias=None)
        return c

    slots, experts, post = moe_align_block_size(ti, block_m, E)
    want = gemm(slots, experts, post)
    assert torch.isfinite(want.float()).all()
    whole = slots[: slots.numel() // block_m * block_m].view(-1, block_m)
    shuffled = torch.stack([block[torch.randperm(block_m, generator=g).to(dev)] for block in whole])
    for other in (whole.flip(1), whole.roll(7, 1), whole.roll(-1, 1), shuffled):
        assert torch.equal(gemm(torch.cat([other.reshape(-1), slots[whole.numel():]]), experts, post), want)
