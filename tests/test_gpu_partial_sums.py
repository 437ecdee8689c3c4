"""Rounding error where the library hands out K ranges: the kernels may run
fewer ranges than that on smaller tiles, but with no larger an error than the
ranges would have. The comparison sums each range's product (the operator
unsplit on that slice of K) in range order in FP32."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# The 2-norm error of N independent elements scatters by about 1 / sqrt(2 N): 0.4% at the smallest of these sizes, and
# the two errors are of the same inputs. 3% leaves room for it.
SLACK = 1.03


def rel(c, exact):
    return np.linalg.norm(c.astype(np.float64) - exact) / np.linalg.norm(exact)


def unsplit(mc, kernel, a, b):
    m, n = a.shape[0], b.shape[1]
    da, db = mc.DeviceBuffer.from_array(a), mc.DeviceBuffer.from_array(b)
    c = mc.DeviceBuffer(4 * m * n)
    mc.launch_matmul(kernel, da.ptr, db.ptr, c.ptr, m, n, a.shape[1])
    mc.synchronize()
    return c.download().reshape(m, n)


def in_ranges(mc, kernel, a, b, splits, step=64):
    k = a.shape[1]
    length = -(-(-(-k // splits)) // step) * step
    total = None
    for k0 in range(0, k, length):
        part = unsplit(mc, kernel, a[:, k0:k0 + length], b[k0:k0 + length])
        total = part if total is None else total + part
    return total


def rounded(oracle, kernel, x):
    rnd = oracle.round_bf16 if kernel == "tensor_core_bf16" else oracle.round_f16
    return rnd(x.reshape(-1)).reshape(x.shape).astype(np.float64)


# 36 to 51 tiles of 128x128 (5 to 7 ranges asked for, none run), 13 to 25 (10 to 19 asked for, 2 to 4 run), few rows;
# last, both sides of the lengths from which fp32 operands run two groups of waves, in one, two and three ranges.
@pytest.mark.parametrize("kernel", ["tensor_core_bf16", "tensor_core_f16"])
@pytest.mark.parametrize("m,n,k", [(704, 768, 2048), (640, 832, 4096), (1024, 768, 4095), (640, 640, 4096),
                                   (1664, 128, 4096), (32, 2048, 4096),
                                   (96, 5440, 320), (768, 768, 448), (96, 5440, 576), (96, 5440, 577),
                                   (256, 1400, 1536), (256, 1400, 1537), (128, 2176, 4032), (128, 2176, 4033)])
def test_the_operator_keeps_the_error_of_the_ranges_it_was_asked_for(device, mc, oracle, kernel, m, n, k):
    a = oracle.uniform(m * k, 7, -1.0, 1.0).reshape(m, k)
    b = oracle.uniform(k * n, 8, -1.0, 1.0).reshape(k, n)
    splits = mc.matmul_splits(kernel, m, n, k, device["cu_count"])
    da, db, c = mc.DeviceBuffer.from_array(a), mc.DeviceBuffer.from_array(b), mc.DeviceBuffer(4 * m * n)
    ws = mc.DeviceBuffer(mc.matmul_workspace_bytes(kernel, m, n, splits))
    print(f"case {kernel} {m}x{n}x{k} splits {splits}", flush=True)
    mc.launch_matmul(kernel, da.ptr, db.ptr, c.ptr, m, n, k, None, splits, ws.ptr)
    mc.synchronize()
    exact = rounded(oracle, kernel, a) @ rounded(oracle, kernel, b)
    got, want = rel(c.download().reshape(m, n), exact), rel(in_ranges(mc, kernel, a, b, splits), exact)
    assert splits > 1 and got <= SLACK * want, f"{got:.3e} against {want:.3e} in {splits} ranges"


def test_ranges_that_the_library_would_not_ask_for_run_as_given(device, mc, oracle):
    # 225 tiles of 128x128: the split rule asks for one range; a caller's own count is that of its sums.
    m, n, k, splits = 1920, 1900, 520, 4
    a = oracle.uniform(m * k, 7, -1.0, 1.0).reshape(m, k)
    b = oracle.uniform(k * n, 8, -1.0, 1.0).reshape(k, n)
    assert mc.matmul_splits("tensor_core_bf16", m, n, k, device["cu_count"]) == 1
    assert mc.matmul_k_ranges("tensor_core_bf16", m, n, k, splits) == 3
    da, db, c = mc.DeviceBuffer.from_array(a), mc.DeviceBuffer.from_array(b), mc.DeviceBuffer(4 * m * n)
    ws = mc.DeviceBuffer(4 * splits * m * n)
    mc.launch_matmul("tensor_core_bf16", da.ptr, db.ptr, c.ptr, m, n, k, None, splits, ws.ptr)
    mc.synchronize()
    assert np.array_equal(c.download().reshape(m, n), in_ranges(mc, "tensor_core_bf16", a, b, splits))


def graph_against_ranges(mc, oracle, device, kernel, m, n, k):
    """The graph's and the ranges' errors for a constant B whose K the operator would cut (K not a multiple of 64)."""
    a = oracle.uniform(m * k, 7, -1.0, 1.0).reshape(m, k)
    b = oracle.uniform(k * n, 8, -1.0, 1.0).reshape(k, n)
    splits = mc.matmul_splits(kernel, m, n, k, device["cu_count"])
    assert splits > 1 and k % 64 != 0
    print(f"case graph {kernel} {m}x{n}x{k} splits {splits}", flush=True)
    c = mc.Compiled(f"input x : f32[{m}, {k}]\nconst w : f32[{k}, {n}] = uniform(seed=8, lo=-1, hi=1)\n"
                    "h = matmul x, w\noutput h\n", options={"matmul": kernel})
    exact = rounded(oracle, kernel, a) @ rounded(oracle, kernel, b)
    return rel(c.run([a.reshape(-1)])[0].reshape(m, n), exact), rel(in_ranges(mc, kernel, a, b, splits), exact)


# Tiles of one fragment's width (16, 32 and 64 rows), K as long as they are used for.
@pytest.mark.parametrize("kernel", ["tensor_core_bf16", "tensor_core_f16"])
@pytest.mark.parametrize("m,n,k", [(16, 2048, 4095), (8, 1395, 2279), (32, 3001, 4000), (184, 512, 2205), (384, 512, 4095)])
def test_graphs_on_small_tiles_keep_the_error_of_the_operators_ranges(device, mc, oracle, kernel, m, n, k):
    got, want = graph_against_ranges(mc, oracle, device, kernel, m, n, k)
    assert got <= SLACK * want, f"{got:.3e} against {want:.3e} in ranges"


# 193 to 204 tiles of 128x128: past the small tiles' line, and still two ranges. K on and off 128, one row and one column
# of a tile; a fused group must not change the product.
@pytest.mark.parametrize("kernel", ["tensor_core_bf16", "tensor_core_f16"])
@pytest.mark.parametrize("m,n,k", [(1792, 1792, 1000), (1660, 1909, 1025), (65, 25500, 2047), (3584, 896, 200)])
def test_graphs_past_the_small_tiles_have_the_bits_of_the_operators_two_ranges(device, mc, oracle, kernel, m, n, k):
    a = oracle.uniform(m * k, 7, -1.0, 1.0).reshape(m, k)
    b = oracle.uniform(k * n, 8, -1.0, 1.0).reshape(k, n)
    assert mc.matmul_splits(kernel, m, n, k, device["cu_count"]) == 2
    want = in_ranges(mc, kernel, a, b, 2).reshape(-1)
    text = (f"input x : f32[{m}, {k}]\nconst w : f32[{k}, {n}] = uniform(seed=8, lo=-1, hi=1)\nh = matmul x, w\n")
    for tail, ref in (("output h\n", want), ("y = neg h\nz = relu y\noutput z\n", np.maximum(-want, 0))):
        print(f"case two sums {kernel} {m}x{n}x{k} {tail!r}", flush=True)
        c = mc.Compiled(text + tail, options={"matmul": kernel})
        assert len(c.launch_nodes) == 1
        assert np.array_equal(c.run([a.reshape(-1)])[0], ref)


# FP32, N or K off the exact forms' steps, on the narrow tiles of each width that run one range where many are asked for.
@pytest.mark.parametrize("m,n,k", [(256, 261, 2047), (250, 300, 1700), (231, 261, 1537), (231, 262, 1535),
                                   (512, 261, 2047), (1000, 1001, 1023), (64, 2032, 1327)])
def test_ragged_fp32_products_keep_the_error_of_the_ranges_they_were_asked_for(device, mc, oracle, m, n, k):
    a = oracle.uniform(m * k, 7, -1.0, 1.0).reshape(m, k)
    b = oracle.uniform(k * n, 8, -1.0, 1.0).reshape(k, n)
    splits = mc.matmul_splits("split_k", m, n, k, device["cu_count"])
    da, db, c = mc.DeviceBuffer.from_array(a), mc.DeviceBuffer.from_array(b), mc.DeviceBuffer(4 * m * n)
    ws = mc.DeviceBuffer(mc.matmul_workspace_bytes("split_k", m, n, splits))
    print(f"case ragged fp32 {m}x{n}x{k} splits {splits}", flush=True)
    mc.launch_matmul("split_k", da.ptr, db.ptr, c.ptr, m, n, k, None, splits, ws.ptr)
    mc.synchronize()
    exact = a.astype(np.float64) @ b.astype(np.float64)
    got = rel(c.download().reshape(m, n), exact)
    want = rel(in_ranges(mc, "double_buffered", a, b, splits, step=32), exact)
    assert splits > 1 and got <= SLACK * want, f"{got:.3e} against {want:.3e} in {splits} ranges"
