"""Both operands of a bf16/fp16 product packed from fp32 (any M, N, K) and the
products on them: the layouts against a numpy rearrangement of the rounded
matrices, every small tile shape and the 256x256 tiles against float64, and
compiled graphs on ragged sizes. Error bound: FP32 accumulation of exact
products of the rounded operands (gamma_k sum|ab|), plus the final rounding."""

import ctypes

import numpy as np
import pytest

from helpers import U32, gamma, run_into_prefilled

pytestmark = pytest.mark.gpu

SMALL_SHAPES = range(9)  # MCHIP_FRAG_*: 16, 32, 64 rows x 16, 32, 64 columns
TILES_256 = -1
TWO_SUMS = -2  # 128x256 tiles, the halves of K summed apart
GUARD = 4096


@pytest.fixture(scope="module")
def ops(mc):
    lib = mc.library()
    vp, i = ctypes.c_void_p, ctypes.c_int
    for name, args in {"mchip_pack16_a_f32": [i, vp, vp, i, i, vp], "mchip_pack16_b_f32": [i, vp, vp, i, i, vp],
                       "mchip_launch_mfma16_packed": [i, i, vp, vp, vp, i, i, i, vp]}.items():
        fn = getattr(lib, name)
        fn.argtypes, fn.restype = args, i
    return lib


def up(x, q):
    return (x + q - 1) // q * q


def packed_index(row, kk, kp):
    return (row // 256 * 256 * kp + kk // 32 * 8192 + row % 256 // 16 * 512 + kk % 32 // 8 * 128 + row % 16 * 8
            + kk % 8)


def pack(mc, ops, which, dtype, m32, rows, k):
    """The packed operand's buffer; `m32` is fp32 A [rows, k] or B [k, rows]."""
    src = mc.DeviceBuffer.from_array(m32)
    dst = mc.DeviceBuffer(up(rows, 256) * up(k, 64) * 2)
    dst.fill_bytes(0xFF)
    fn = ops.mchip_pack16_a_f32 if which == "a" else ops.mchip_pack16_b_f32
    args = (rows, k) if which == "a" else (k, rows)
    assert fn(dtype, src.ptr, dst.ptr, *args, None) == 0
    mc.synchronize()
    return dst


@pytest.mark.parametrize("dtype", [1, 2], ids=["bf16", "f16"])
@pytest.mark.parametrize("rows,k", [(1, 1), (16, 64), (17, 33), (300, 127), (257, 128), (513, 200)])
def test_packing_writes_the_layout_and_pads_k_with_zeros(device, mc, oracle, ops, dtype, rows, k):
    rnd = oracle.round_bf16 if dtype == 1 else oracle.round_f16
    bits = (lambda x: (x.view(np.uint32) >> 16).astype(np.uint16)) if dtype == 1 else \
        (lambda x: x.astype(np.float16).view(np.uint16))
    a = oracle.uniform(rows * k, 3, -1.0, 1.0)
    want = np.zeros((rows, up(k, 64)), np.uint16)
    want[:, :k] = bits(rnd(a)).reshape(rows, k)
    rr, kk = np.meshgrid(np.arange(rows), np.arange(up(k, 64)), indexing="ij")
    at = packed_index(rr, kk, up(k, 64))
    for which, m32 in (("a", a), ("b", np.ascontiguousarray(a.reshape(rows, k).T))):
        print(f"case pack {which} {rows}x{k} dtype {dtype}", flush=True)
        got = pack(mc, ops, which, dtype, m32, rows, k).download(np.uint16)
        assert np.array_equal(got[at], want), which


# (m, n, k): one element; below, at and one past tile edges of every shape; K below, at and past a padded step, with
# more and fewer steps than a block has waves; N odd, N % 4 and N % 8; one and several 256-row bands.
PRODUCTS = [(1, 1, 1), (16, 16, 64), (17, 33, 65), (5, 250, 31), (63, 70, 1000), (64, 64, 512), (65, 129, 577),
            (300, 259, 96), (257, 255, 2047), (32, 260, 520)]
# K long enough that every wave of every shape runs its two-batch loop (more than 2 kU steps of 32 k per wave: K past
# 4096 for 16x16 tiles, 2048 for three-fragment ones), then each way of ending it: one batch left or two, whole or not,
# and a last wave with fewer steps than the others.
LONG_PRODUCTS = [(5, 37, 4200), (17, 33, 6400), (33, 70, 8257), (16, 16, 12288), (64, 64, 5000), (7, 100, 6144)]


@pytest.mark.parametrize("dtype", [1, 2], ids=["bf16", "f16"])
@pytest.mark.parametrize("m,n,k", PRODUCTS + LONG_PRODUCTS)
def test_every_tile_shape_is_within_the_accumulation_bound(device, mc, oracle, ops, dtype, m, n, k):
    a, b = oracle.uniform(m * k, 7, -1.0, 1.0), oracle.uniform(k * n, 8, -1.0, 1.0)
    rnd = oracle.round_bf16 if dtype == 1 else oracle.round_f16
    exact, absdot = oracle.gemm_f64(rnd(a), rnd(b), m, k, n)
    bound = gamma(k) * absdot + 2 * U32 * np.abs(exact) + 1e-30
    pa, pb = pack(mc, ops, "a", dtype, a, m, k), pack(mc, ops, "b", dtype, b, n, k)
    for shape in [TWO_SUMS, TILES_256, *SMALL_SHAPES]:
        print(f"case product {m}x{n}x{k} dtype {dtype} shape {shape}", flush=True)
        c = mc.DeviceBuffer.from_array(np.full(m * n + GUARD, np.nan, np.float32))
        assert ops.mchip_launch_mfma16_packed(dtype, shape, pa.ptr, pb.ptr, c.ptr, m, n, k, None) == 0
        mc.synchronize()
        out = c.download()
        assert np.all(np.isnan(out[m * n:])), "a write past the end of C"
        assert np.all(np.abs(out[:m * n].astype(np.float64) - exact) <= bound), f"shape {shape}"


def test_infinities_stay_in_their_row_and_column(device, mc, oracle, ops):
    m, n, k = 70, 70, 100
    a, b = oracle.uniform(m * k, 7, 0.5, 1.0).reshape(m, k), oracle.uniform(k * n, 8, 0.5, 1.0).reshape(k, n)
    a[3, 0] = np.inf
    b[k - 1, 5] = np.nan
    pa, pb = pack(mc, ops, "a", 1, a.ravel(), m, k), pack(mc, ops, "b", 1, b.ravel(), n, k)
    for shape in [TWO_SUMS, TILES_256, *SMALL_SHAPES]:
        c = mc.DeviceBuffer(m * n * 4)
        assert ops.mchip_launch_mfma16_packed(1, shape, pa.ptr, pb.ptr, c.ptr, m, n, k, None) == 0
        mc.synchronize()
        out = c.download().reshape(m, n)
        odd = ~np.isfinite(out)
        want = np.zeros((m, n), bool)
        want[3, :], want[:, 5] = True, True
        assert np.array_equal(odd, want), f"shape {shape}"


@pytest.mark.parametrize("kernel,dtype", [("tensor_core_bf16", 1), ("tensor_core_f16", 2)])
@pytest.mark.parametrize("m,k,n", [(1, 70, 129), (33, 64, 72), (100, 1023, 1001), (700, 333, 515)])
def test_graphs_on_ragged_sizes_fuse_and_match_float64(device, mc, oracle, kernel, dtype, m, k, n):
    text = (f"input x : f32[{m}, {k}]\nconst w : f32[{k}, {n}] = uniform(seed=2, lo=-1, hi=1)\n"
            f"const b : f32[{n}] = uniform(seed=3, lo=-1, hi=1)\nh = matmul x, w\ny = add h, b\nz = relu y\noutput z\n")
    x, w, b = oracle.uniform(m * k, 1, -1.0, 1.0), oracle.uniform(k * n, 2, -1.0, 1.0), oracle.uniform(n, 3, -1.0, 1.0)
    rnd = oracle.round_bf16 if dtype == 1 else oracle.round_f16
    exact, absdot = oracle.gemm_f64(rnd(x), rnd(w), m, k, n)
    want = np.maximum(exact + np.tile(b.astype(np.float64), m), 0.0)
    bound = gamma(k) * absdot + 4 * U32 * (np.abs(exact) + 1.0)
    for epilogue in (1, 0):
        c = mc.Compiled(text, options={"matmul": kernel, "epilogue": epilogue})
        assert len(c.launch_nodes) == (1 if epilogue else 2)
        out = run_into_prefilled(mc, c, [x])[0].astype(np.float64)
        assert np.all(np.abs(out - want) <= bound), f"epilogue {epilogue}"


# A residual read element by element at the matrix edge, its last element at the end of its buffer: N of each remainder
# by 4, on 256x256, two-sum and small tiles; and B fed per run (whole chunks at every edge).
@pytest.mark.parametrize("m,k,n,fed", [(1100, 70, 4000, False), (1031, 65, 4001, False), (2305, 40, 1794, False),
                                       (1792, 130, 1791, False), (33, 64, 71, False), (300, 96, 130, False),
                                       (300, 64, 264, True), (65, 128, 1000, True)])
def test_fused_groups_at_the_edges(device, mc, oracle, m, k, n, fed):
    text = (f"input x : f32[{m}, {k}]\ninput r : f32[{m}, {n}]\n"
            + (f"input w : f32[{k}, {n}]\n" if fed else f"const w : f32[{k}, {n}] = uniform(seed=2, lo=-1, hi=1)\n")
            + f"const b : f32[{n}] = uniform(seed=3, lo=-1, hi=1)\nh = matmul x, w\nhb = add h, b\ny = add hb, r\noutput y\n")
    x, w, b = oracle.uniform(m * k, 1, -1.0, 1.0), oracle.uniform(k * n, 2, -1.0, 1.0), oracle.uniform(n, 3, -1.0, 1.0)
    r = oracle.uniform(m * n, 4, -1.0, 1.0)
    print(f"case fused edge {m}x{k}x{n} fed {fed}", flush=True)
    exact, absdot = oracle.gemm_f64(oracle.round_bf16(x), oracle.round_bf16(w), m, k, n)
    want = exact + np.tile(b.astype(np.float64), m) + r
    c = mc.Compiled(text, options={"matmul": "tensor_core_bf16"})
    assert len(c.launch_nodes) == 1
    out = run_into_prefilled(mc, c, [x, r, w] if fed else [x, r])[0].astype(np.float64)
    assert np.all(np.abs(out - want) <= gamma(k) * absdot + 4 * U32 * (np.abs(exact) + 2.0))
