"""What the launch heuristics of the dense GEMMs choose, as far as it decides whether a launch is right: host code, no GPU."""
import ctypes

import pytest

from sglang_amd import _lib

STREAMING, ROW_TILES, STRIPS, TILES = 1, 2, 3, 4  # SGLAMD_PLAN_* of include/sglamd.h
CUS = 256  # what the library takes without a GPU


def _plan(M, N, K, block=True):
    plan = (ctypes.c_int32 * 4)()
    form = _lib.lib.sglamd_dense_plan(int(block), M, N, K, plan)
    assert form in (STREAMING, ROW_TILES, STRIPS, TILES)
    return form, list(plan)


def _wrong_scales(blocks, depth):
    """The strip kernel's order of requests, barriers and reads of one workgroup: how many blocks of its items (of blocks[j] K
    blocks each) read a weight-scale table that another item's request has been written over or may be."""
    stream = [(j, k) for j, n in enumerate(blocks) for k in range(n)]
    table, wrong, at = [None, None], 0, 0

    def request():
        nonlocal at
        if at < len(stream):
            item, k = stream[at]
            if k == 0:
                table[item & 1] = item
            at += 1

    for _ in range(depth):
        request()
    # block 0's scales are read behind the first barrier, before anything else is requested
    wrong += table[0] != 0
    for b in range(len(stream)):
        # behind block b's barrier the loading waves request one block, the others read block b + 1's scales, in either order
        item = stream[b + 1][0] if b + 1 < len(stream) else None
        before = item is not None and table[item & 1] != item
        request()
        wrong += item is not None and (before or table[item & 1] != item)
    return wrong


def test_model_of_the_scale_tables():
    assert _wrong_scales([1] * 12, 5) == 10 and _wrong_scales([2] * 12, 5) > 0 and _wrong_scales([3] * 12, 5) > 0
    for depth in (3, 5, 6, 8):
        assert _wrong_scales([depth - 1] * 12, depth) == 0 and _wrong_scales([depth - 2] * 12, depth) > 0
        assert _wrong_scales([1, 1], depth) == 0


@pytest.mark.parametrize("K", [128, 256, 384, 512, 640, 768, 896, 1024, 2048])
def test_strips_keep_the_scales_of_every_item(K):
    """Few K blocks and many weight rows: no workgroup of a strip launch asks for an item's scales while the item two before
    still needs the place."""
    strips = 0
    for M in (17, 24, 32, 33, 64, 65, 96, 97, 128):
        for N in [1 << p for p in range(12, 22)] + [3 << p for p in range(11, 20)] + [261376, 398592, 790016, 791808, 200008]:
            if N * K >= 2**31:
                continue
            form, (_, cols, slices, depth) = _plan(M, N, K)
            if form != STRIPS:
                continue
            strips += 1
            items, nkb = -(-N // cols) * slices, K // 128
            mine = range(0, items, CUS)  # of the workgroup with the most of them
            blocks = [nkb * (i * slices // items + 1) // slices - nkb * (i * slices // items) // slices for i in mine]
            if len(blocks) > 12:
                blocks = blocks[:12]
            assert _wrong_scales(blocks, depth) == 0, f"M={M} N={N} K={K}: {blocks} K blocks, {depth} stages"
    assert strips or K < 512


@pytest.mark.parametrize("M,N,K", [(17, 791808, 128), (24, 398592, 256), (32, 261376, 384)])
def test_too_few_k_blocks_for_strips(M, N, K):
    assert _plan(M, N, K)[0] == STREAMING
    assert _plan(M, N, K, block=False)[0] == STRIPS  # the row modes have no such tables


def test_scratch_is_asked_for_where_it_is_used():
    """Slabs for the K slices that the launch has, and none for one that does not split K.  (Row modes; a tile launch that is cut in
    two along N splits K on its second part alone.)"""
    seen = set()
    for M in (1, 16, 17, 32, 40, 64, 65, 96, 128, 129, 200, 320, 700, 1024, 1500):
        for N in (256, 512, 1000, 1152, 2048, 2050, 4096, 7168, 9000, 14336, 24576, 36864):
            for K in (512, 1024, 1664, 2048, 4096, 7168, 8192, 16384):
                form, (_, _, slices, _) = _plan(M, N, K, block=False)
                need = _lib.lib.sglamd_gemm_workspace_bytes(M, N, K)
                split = form in (STRIPS, TILES) and slices > 1
                seen.add((form, split))
                if form == TILES and not split and N > 256 * CUS // -(-M // 256):
                    continue  # (may be cut in two)
                assert need == (slices * M * N * 4 if split else 0), f"M={M} N={N} K={K}: form {form}, {slices} slices, {need} bytes"
    assert seen == {(STREAMING, False), (ROW_TILES, False), (STRIPS, False), (STRIPS, True), (TILES, False), (TILES, True)}


@pytest.mark.parametrize("M,N,K,rows", [
    # K too short for 192-row tiles: the fastest height measured (us in 64-, 128-, 256-row tiles)
    (150, 33792, 640, 256),    # 16.0, -, 15.3
    (150, 33792, 1024, 256),   # 19.2, -, 18.4
    (192, 36864, 1024, 256),   # 20.1, -, 19.3
    (131, 49152, 512, 256),    # -, 18.5, 15.1
    (160, 57344, 896, 256),    # -, 24.8, 21.0
    (192, 65536, 1024, 256),   # -, 32.0, 24.7
    (140, 30720, 640, 128),    # -, 13.2, 15.1
    (192, 31744, 1024, 128),   # -, 16.6, 18.9
    (150, 36864, 7168, 192),
    (150, 8192, 28672, 256),
])
@pytest.mark.parametrize("block", [False, True])
def test_tile_heights_at_129_to_192_rows(M, N, K, rows, block):
    form, plan = _plan(M, N, K, block)
    assert form == TILES and plan[0] == rows


@pytest.mark.parametrize("M,N,K,rows", [
    # four rounds of 64-row tiles or three of 128 (us)
    (420, 33280, 896, 64),     # 32.1, 35.2
    (448, 33792, 640, 64),     # 28.2, 30.6
    (1466, 10816, 768, 64),    # 33.8, 36.8
    (545, 28480, 512, 128),    # 32.1, 29.3
    (1038, 14976, 896, 128),   # 43.3, 40.8
    (2090, 7808, 768, 128),    # 43.4, 40.2
    (315, 25024, 768, 256),    # 21.2, - (256-row tiles 19.8)
    (420, 33280, 384, 128),    # 24.6, 24.0
])
def test_tile_heights_of_a_short_k(M, N, K, rows):
    form, plan = _plan(M, N, K, block=False)
    assert form == TILES and plan[0] == rows
