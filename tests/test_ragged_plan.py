"""Which body runs an FP32 product that the exact ring and narrow forms do not
take (host logic, no GPU)."""

import ctypes

import pytest

NONE, WIDE, WIDE8 = 0, 1, 6


@pytest.mark.parametrize("m,n,k,depth,want", [
    (2000, 1001, 1023, 1, (WIDE8, 128, 512)),   # 16 x 8 tiles: one per CU at most
    (3648, 2176, 423, 1, (WIDE, 493, 256)),
    (1000, 1000, 1000, 4, (WIDE8, 256, 512)),
    (128, 4, 64, 1, (WIDE8, 1, 512)),
    (128, 3, 64, 1, (NONE, 0, 0)), (128, 4, 63, 1, (NONE, 0, 0)),  # the two-stage body's
    (64, 2 << 20, 33, 1, (NONE, 0, 0)),
])
def test_the_ragged_ring_runs_one_block_per_tile_and_split(mc, m, n, k, depth, want):
    f = mc.library().mchip_f32_ragged_ring_plan
    grid, block = ctypes.c_uint(), ctypes.c_uint()
    assert (f(m, n, k, depth, 256, ctypes.byref(grid), ctypes.byref(block)), grid.value, block.value) == want


@pytest.mark.parametrize("m,n,k,splits,want", [
    (16, 1001, 777, 8, (5, 1, 784)),   # as 16x1004x784
    (16, 1001, 1300, 8, (1, 8, 176)),
    (256, 513, 2047, 8, (2, 1, 2048)),
    (8, 3, 100, 1, None), (8, 4, 15, 1, None),
])
def test_the_ragged_narrow_plan_is_the_exact_one_rounded_up(mc, m, n, k, splits, want):
    f = mc.library().mchip_f32_ragged_narrow_plan
    out = [ctypes.c_int() for _ in range(3)]
    ok = f(m, n, k, splits, 256, *[ctypes.byref(x) for x in out])
    assert (tuple(x.value for x in out) if ok else None) == want


@pytest.mark.parametrize("m,n,k,splits,want", [
    (1, 2048, 512, 8, (5, 1, 512)), (4, 512, 1024, 16, (5, 1, 1024)),
    (16, 4096, 1024, 4, (5, 1, 1024)), (128, 512, 512, 8, (5, 1, 512)),
    (16, 4096, 1040, 4, (1, 4, 272)), (1, 512, 2048, 32, (1, 32, 64)), (2, 512, 2048, 32, (1, 32, 64)),  # K too long
    (16, 4112, 1024, 4, (1, 2, 512)),     # 257 tiles of 16x16
    (16, 4096, 1024, 1, (1, 1, 1024)),    # no ranges to avoid
])
def test_short_k_products_that_would_split_run_16x16_tiles(mc, m, n, k, splits, want):
    f = mc.library().mchip_f32_narrow_plan
    out = [ctypes.c_int() for _ in range(3)]
    assert f(m, n, k, splits, 256, 0, *[ctypes.byref(x) for x in out]) and tuple(x.value for x in out) == want


@pytest.mark.parametrize("m,n,k,splits,want", [
    (96, 2192, 8100, 14, (4, 3, 2704)), (544, 464, 3896, 12, (4, 3, 1312)),   # 70 and 72 tiles: three ranges, not two
    (96, 2192, 8100, 2, (4, 2, 4064)),                                        # no more than asked for
    (193, 2240, 4444, 7, (0, 1, 4448)), (394, 1204, 3128, 6, (0, 1, 3136)),   # 140 and 133 tiles: 245 and 247 of 32x64
    (333, 2112, 5516, 5, (4, 1, 5520)),                                       # 198 tiles: 363 of 32x64 are too many
    (618, 1792, 904, 3, (0, 1, 912)),                                         # 280 tiles: 1.1 rounds
    (1000, 1001, 1023, 4, (4, 1, 1024)), (2000, 1001, 1023, 2, (4, 1, 1024)),  # one and two whole rounds
    (300, 424, 4968, 21, (0, 2, 2496)),                                       # 32x64 tiles to begin with
])
def test_ragged_64x64_tiles_fill_the_chip(mc, m, n, k, splits, want):
    f = mc.library().mchip_f32_ragged_narrow_plan
    out = [ctypes.c_int() for _ in range(3)]
    assert f(m, n, k, splits, 256, *[ctypes.byref(x) for x in out]) and tuple(x.value for x in out) == want
