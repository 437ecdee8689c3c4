"""The FP32 matrix-core GEMMs on what their exact forms do not take: K not a
multiple of 32 (16), N not of 4, operands at any float address; and the 16x16
tiles of short K, exact and ragged. Edges of the
tiles, of the K steps and of the K ranges, the epilogue at the matrix edge,
against float64 within the FP32 dot-product bound."""

import numpy as np
import pytest

from helpers import fp32_gemm_bound, run_into_prefilled

pytestmark = pytest.mark.gpu

GUARD = 4096
# (m, n, k): 128x128 tiles (one to a CU and more), a last tile of 1, 2 and 3 columns past a tile and of one row; K one
# past and one short of a step, N odd, N % 4 = 2; a last K range of one short step; narrow tiles of every shape.
DOUBLE_BUFFERED = [(128, 129, 65), (129, 130, 95), (300, 131, 1023), (2100, 2049, 100), (2311, 2050, 127),
                   (257, 4, 64), (130, 5, 70), (64, 300, 129)]
SPLIT_K = [(1, 5, 17, 1), (16, 1001, 777, 6), (20, 70, 33, 1), (65, 513, 2049, 8), (33, 1030, 1000, 4),
           (1000, 1001, 1023, 4), (257, 515, 4097, 16), (512, 130, 130, 3), (200, 18, 1000, 15), (7, 6, 100, 4),
           (1, 2048, 512, 8), (1, 516, 2048, 8), (17, 1000, 1023, 4), (128, 512, 144, 2), (31, 33, 129, 2),
           # 64x64 tiles in three ranges, the last one short; 32x64 tiles in their place, K long and short
           (96, 2192, 2084, 14), (128, 2181, 2051, 14), (200, 2181, 2050, 7), (618, 1797, 130, 3),
           # 16x32 tiles with four accumulators and, past K = 1536, with eight
           (231, 261, 1536, 10), (231, 261, 1537, 10), (157, 693, 334, 5)]


def check(mc, oracle, kernel, m, n, k, splits, offsets):
    a, b = oracle.uniform(m * k, 7, -1.0, 1.0), oracle.uniform(k * n, 8, -1.0, 1.0)
    exact, absdot = oracle.gemm_f64(a, b, m, k, n)
    src = [mc.DeviceBuffer.from_array(x) for x in (a, b)]
    buf = [mc.DeviceBuffer(4 * x.size + 16) for x in (a, b)]
    for s, d, off, x in zip(src, buf, offsets, (a, b)):
        mc.memcpy_dtod_async(d.ptr + off, s.ptr, 4 * x.size)
    c = mc.DeviceBuffer.from_array(np.full(m * n + GUARD + 1, np.nan, np.float32))
    ws = mc.DeviceBuffer(max(4, mc.matmul_workspace_bytes(kernel, m, n, splits)))
    mc.synchronize()
    mc.launch_matmul(kernel, buf[0].ptr + offsets[0], buf[1].ptr + offsets[1], c.ptr + offsets[2], m, n, k, None, splits,
                     ws.ptr)
    mc.synchronize()
    out = c.download()[offsets[2] // 4:]
    assert np.all(np.isnan(out[m * n:])), "a write past the end of C"
    got = out[:m * n].astype(np.float64)
    assert np.all(np.abs(got - exact) <= fp32_gemm_bound(exact, absdot, k))


@pytest.mark.parametrize("m,n,k", DOUBLE_BUFFERED)
def test_unsplit_products(device, mc, oracle, m, n, k):
    print(f"case ragged double_buffered {m}x{n}x{k}", flush=True)
    check(mc, oracle, "double_buffered", m, n, k, 1, (0, 0, 0))


@pytest.mark.parametrize("m,n,k,splits", SPLIT_K)
def test_split_products(device, mc, oracle, m, n, k, splits):
    print(f"case ragged split_k {m}x{n}x{k} splits {splits}", flush=True)
    check(mc, oracle, "split_k", m, n, k, splits, (0, 0, 0))


@pytest.mark.parametrize("kernel,m,n,k,splits", [("double_buffered", 300, 260, 96, 1), ("split_k", 300, 260, 96, 2),
                                                 ("split_k", 16, 512, 256, 4)])
@pytest.mark.parametrize("offsets", [(4, 0, 0), (0, 8, 0), (0, 0, 4), (12, 4, 8)])
def test_operands_at_any_float_address(device, mc, oracle, kernel, m, n, k, splits, offsets):
    print(f"case unaligned {kernel} {m}x{n}x{k} {offsets}", flush=True)
    check(mc, oracle, kernel, m, n, k, splits, offsets)


@pytest.mark.parametrize("kernel,m,n,k,splits", [("double_buffered", 200, 131, 100, 1), ("split_k", 70, 131, 100, 1),
                                                 ("split_k", 20, 70, 1000, 8)])
def test_infinities_and_nans_stay_in_their_row_and_column(device, mc, oracle, kernel, m, n, k, splits):
    a, b = oracle.uniform(m * k, 7, 0.5, 1.0).reshape(m, k), oracle.uniform(k * n, 8, 0.5, 1.0).reshape(k, n)
    a[4, 0], a[m - 1, k - 1], b[0, 5], b[k - 1, n - 1] = np.inf, np.nan, np.inf, np.inf
    want = np.zeros((m, n), bool)
    want[4, :], want[m - 1, :], want[:, 5], want[:, n - 1] = True, True, True, True
    da, db, c = mc.DeviceBuffer.from_array(a), mc.DeviceBuffer.from_array(b), mc.DeviceBuffer(4 * m * n)
    ws = mc.DeviceBuffer(4 * splits * m * n)
    mc.launch_matmul(kernel, da.ptr, db.ptr, c.ptr, m, n, k, None, splits, ws.ptr)
    mc.synchronize()
    assert np.array_equal(~np.isfinite(c.download().reshape(m, n)), want)


# A bias (periodic operand) and a residual (contiguous, its last element at the end of its buffer).
@pytest.mark.parametrize("m,n,k", [(300, 131, 1023), (2100, 2050, 70), (20, 71, 500), (1, 1001, 1023), (129, 9, 66),
                                   (96, 2192, 2084)])
@pytest.mark.parametrize("matmul", ["auto", "double_buffered", "split_k"])
def test_fused_groups_at_the_matrix_edge(device, mc, oracle, m, n, k, matmul):
    print(f"case ragged fused {matmul} {m}x{n}x{k}", flush=True)
    text = (f"input x : f32[{m}, {k}]\ninput w : f32[{k}, {n}]\ninput b : f32[{n}]\ninput r : f32[{m}, {n}]\n"
            "h = matmul x, w\nhb = add h, b\ny = add hb, r\noutput y\n")
    sizes = (m * k, k * n, n, m * n)
    x, w, b, r = (oracle.uniform(s, 1 + i, -1.0, 1.0) for i, s in enumerate(sizes))
    exact, absdot = oracle.gemm_f64(x, w, m, k, n)
    want = exact + np.tile(b.astype(np.float64), m) + r
    c = mc.Compiled(text, options={"matmul": matmul})
    assert len(c.launch_nodes) == 1 and len(c.launch_nodes[0]) == 2
    got = run_into_prefilled(mc, c, [x, w, b, r])[0].astype(np.float64)
    assert np.all(np.abs(got - want) <= fp32_gemm_bound(exact, absdot, k) + 4 * 2.0 ** -24 * (np.abs(exact) + 2.0))


# 16x16 tiles (exact and ragged), ragged narrow tiles unsplit, the ragged ring; last, products of one range, which need
# no workspace, whatever is asked for.
@pytest.mark.parametrize("m,n,k,splits,offset,refused", [
    (16, 512, 1024, 4, 0, True), (1, 2048, 512, 8, 0, True), (17, 1000, 1023, 4, 0, True), (300, 260, 100, 2, 0, True),
    (256, 517, 2047, 8, 0, True), (256, 512, 2048, 8, 4, True), (1300, 1301, 1500, 2, 0, True),
    (256, 512, 2048, 8, 0, False), (300, 260, 30, 4, 0, False), (300, 260, 100, 1, 0, False)])
def test_ranges_without_a_workspace_are_refused_whatever_number_of_them_runs(device, mc, m, n, k, splits, offset, refused):
    a, b, c = (mc.DeviceBuffer(4 * x + 16) for x in (m * k, k * n, m * n))
    run = lambda: mc.launch_matmul("split_k", a.ptr + offset, b.ptr, c.ptr, m, n, k, None, splits, None)
    if refused:
        with pytest.raises(mc.HipError):
            run()
    else:
        run()
    mc.synchronize()
