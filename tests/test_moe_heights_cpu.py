"""The sorted-block height that a fused-MoE layer picks by itself, on layers whose weights come from HBM: the fastest of the
measured ones, within 3 %.  The layer times (us, by height) are of one MI355X; the height shows in the workspace that the
layer asks for."""
import pytest

from sglang_amd import _lib

BLOCK_FP8, ROW_FP8, ROW_INT8, BLOCK_INT8 = 0, 1, 2, 3  # sglamd_moe_mode


def _picked(mode, m, h, i, e, topk):
    if mode == BLOCK_FP8:
        need = lambda height: _lib.lib.sglamd_fused_moe_block_fp8_workspace(m, h, i, e, topk, height)  # noqa: E731
    else:
        need = lambda height: _lib.lib.sglamd_fused_moe_layer_workspace(mode, m, h, i, e, topk, height)  # noqa: E731
    sizes = {height: need(height) for height in (16, 64, 128, 192)}
    assert len(set(sizes.values())) == 4
    return next(height for height, size in sizes.items() if size == need(0))


CASES = [
    # mode, tokens, hidden, intermediate, experts, topk, times
    (BLOCK_FP8, 600, 4096, 1536, 8, 2, {64: 113, 128: 79.4, 192: 94}),
    (BLOCK_FP8, 600, 7168, 1536, 8, 2, {64: 175, 128: 122.6, 192: 135}),
    (BLOCK_FP8, 1400, 2048, 512, 32, 4, {64: 92.6, 128: 70, 192: 87.5}),
    (BLOCK_FP8, 933, 4096, 1024, 32, 6, {64: 238, 128: 169, 192: 201}),
    (BLOCK_FP8, 1400, 2048, 1024, 16, 2, {64: 79.5, 128: 63.9, 192: 76}),
    (BLOCK_FP8, 1867, 4096, 512, 64, 6, {64: 280, 128: 195, 192: 221}),
    (BLOCK_FP8, 1920, 4096, 1536, 64, 6, {64: 577, 128: 444, 192: 404}),
    (BLOCK_FP8, 2880, 2048, 1024, 128, 8, {64: 436, 128: 348, 192: 313}),
    (BLOCK_FP8, 2219, 4096, 1536, 64, 6, {64: 688, 128: 460, 192: 512}),
    (BLOCK_FP8, 6656, 7168, 2048, 256, 8, {64: 5808, 128: 3901, 192: 4189}),
    (BLOCK_FP8, 512, 7168, 2048, 256, 8, {16: 2911, 64: 1756, 128: 2013, 192: 2042}),
    (BLOCK_FP8, 600, 6144, 2048, 16, 4, {64: 269, 128: 217, 192: 184}),
    (BLOCK_FP8, 416, 4096, 1536, 8, 2, {64: 71.6, 128: 82, 192: 86.1}),
    (BLOCK_FP8, 40, 6144, 384, 32, 4, {16: 67.3, 64: 81.7, 128: 86.3, 192: 94.2}),
    (BLOCK_INT8, 53, 4096, 512, 64, 6, {16: 92.5, 64: 99.8, 128: 104, 192: 112}),
    (BLOCK_INT8, 16, 4096, 1024, 32, 6, {16: 89.8, 64: 85.9, 128: 95.4, 192: 102}),
    (BLOCK_INT8, 600, 4096, 1536, 8, 2, {64: 117, 128: 81.5, 192: 95.3}),
    (ROW_FP8, 32, 4096, 896, 16, 4, {16: 53.5, 64: 58.4, 128: 62.3, 192: 73}),
    (ROW_INT8, 600, 4096, 1536, 8, 2, {64: 103, 128: 79.7, 192: 87.2}),
    (ROW_INT8, 933, 4096, 1024, 32, 6, {64: 213, 128: 168, 192: 209}),
    (ROW_INT8, 256, 4096, 1536, 64, 6, {16: 422, 64: 225, 128: 228, 192: 277}),
    (ROW_INT8, 1200, 7168, 1536, 8, 2, {64: 204, 128: 205, 192: 157}),
]


@pytest.mark.parametrize("mode,m,h,i,e,topk,times", CASES)
def test_picked_height_is_the_fastest_measured(mode, m, h, i, e, topk, times):
    assert times[_picked(mode, m, h, i, e, topk)] <= 1.03 * min(times.values())


def test_heights_of_extreme_layers():
    for mode in (BLOCK_FP8, ROW_FP8, ROW_INT8, BLOCK_INT8):
        # every expert named by every token (no spread), one expert, more rows than blocks of any height hold, one token
        for m, h, i, e, topk in ((64, 7168, 2048, 8, 8), (192, 7168, 2048, 8, 8), (200, 8192, 8192, 1, 1),
                                 (1 << 20, 7168, 2048, 8, 8), (1, 7168, 2048, 256, 8), (4096, 4096, 1536, 2047, 8)):
            assert _picked(mode, m, h, i, e, topk) in (16, 64, 128, 192)


@pytest.mark.parametrize("block_m", [64, 128])
@pytest.mark.parametrize("experts", [1, 4, 8, 64, 256])
def test_separate_grouped_gemms_count_experts_not_blocks(experts, block_m):
    """A list made for `experts` experts (and the ids of -1), or for fewer pairs than that, of any number of pairs."""
    n, k = 1024, 1024
    for pairs in (1, 5, 60, 64, 1000, 8192, 100000):
        for buckets in (experts, experts + 1):
            blocks = -(-(pairs + min(pairs, buckets) * (block_m - 1)) // block_m)
            got = _lib.lib.sglamd_moe_list_streams(pairs, blocks, block_m, n, k)
            assert got == (min(pairs, buckets) * n * k >= 64000000)
