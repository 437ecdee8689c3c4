"""Which tiles a bf16/fp16 product on packed operands runs (host logic, no
GPU), and that every such GEMM body compiles with a fused epilogue. Shapes:
-1 = 256x256 tiles, else 3 log2(rows / 16) + log2(columns / 16)."""

import pytest


@pytest.mark.parametrize("m,n,want", [
    (1, 4096, 0), (16, 4096, 0),          # 256 tiles of 16x16
    (16, 16384, 2),                       # 16x64 still gives every CU a tile
    (32, 4096, 3), (64, 4096, 6),
    (128, 4096, 7), (256, 4096, 8), (512, 4096, 8),
    (64, 65536, 8),                       # few rows: never the 256-row tiles
    (1024, 4096, -1), (4096, 14336, -1),  # more than three rounds of 64x64 tiles
    (100, 1000, 6), (1000, 1000, 8), (1, 1, 0),
])
def test_the_plan_picks_the_widest_tile_that_fills_the_chip(mc, want, m, n):
    assert mc.library().mchip_mfma16_packed_plan(m, n, 256) == want


def test_sizes_past_the_kernels_offsets_are_refused(mc):
    fits = mc.library().mchip_pack16_fits
    assert fits(1, 1, 1) and fits(8192, 8192, 8192)
    assert not fits(0, 8, 8) and not fits(8, 8, (1 << 21) + 1) and not fits((1 << 31) - 200, 8, 8)


@pytest.mark.parametrize("body,call", [("bf16_packed", "mc_gemm16_packed<true>"),
                                       ("f16_packed", "mc_gemm16_packed<false>"),
                                       ("bf16_frag", "mc_gemm16_frag<true, McFragCfg<1, 1>>"),
                                       ("f16_frag", "mc_gemm16_frag<false, McFragCfg<1, 1>>")])
def test_the_packed_bodies_compile_for_gfx950(mc, body, call):
    text = "r0 = load in0\nr1 = load in1\nr2 = add r0, r1\nr3 = tanh r2\n"
    src = mc.generate_gemm_epilogue_kernel(text, 0, [(96, 257), (257,)], (96, 257), True, body)
    assert call in src
    ok, log = mc.compile_kernel_source(src, "gfx950")
    assert ok, log
