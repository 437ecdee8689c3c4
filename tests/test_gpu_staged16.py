"""The bf16/fp16 kernel on row-major operands (fp32, rounded inside, or 16-bit)
at the sizes where it can go wrong: tile and K-step edges, matrices narrower
than a lane's columns, unaligned pointers, K ranges; and the packed hardware
rounding against the software one. Bound: FP32 accumulation of exact products
of the rounded operands (gamma_k sum|ab|) plus the final rounding."""

import numpy as np
import pytest

from helpers import U32, gamma

pytestmark = pytest.mark.gpu

FORMATS = [("tensor_core_bf16", 1), ("tensor_core_f16", 2)]
GUARD = 4096
# (m, n, k, splits): N below a lane's 4 columns and just past a tile (the last lanes' columns start before the
# tile); K below, at and just past a step, an odd number of steps, K odd; 32-row, 64x64 (one and several tiles per
# CU, with and without a second group of waves) and 128x128 tiles (up to one per CU and more); K in ranges.
CASES = [(1, 1, 1, 1), (3, 2, 70, 1), (40, 3, 64, 1), (130, 129, 63, 1), (20, 130, 65, 1), (64, 65, 192, 1),
         (33, 66, 200, 4), (100, 67, 1000, 16), (16, 515, 777, 8), (1000, 1001, 129, 2), (1030, 1100, 320, 4),
         (1900, 2049, 100, 1), (2100, 2179, 72, 1), (2307, 2050, 191, 1)]


@pytest.mark.parametrize("kernel,dtype", FORMATS)
@pytest.mark.parametrize("m,n,k,splits", CASES)
@pytest.mark.parametrize("operands,offset", [("f32", 0), ("f32", 4), ("16", 0), ("16", 2)])
def test_every_edge_is_within_the_accumulation_bound(device, mc, oracle, kernel, dtype, m, n, k, splits, operands, offset):
    print(f"case staged {kernel} {m}x{n}x{k} splits {splits} operands {operands} +{offset}", flush=True)
    a, b = oracle.uniform(m * k, 7, -1.0, 1.0), oracle.uniform(k * n, 8, -1.0, 1.0)
    rnd = oracle.round_bf16 if dtype == 1 else oracle.round_f16
    exact, absdot = oracle.gemm_f64(rnd(a), rnd(b), m, k, n)
    size = 4 if operands == "f32" else 2
    da, db = mc.DeviceBuffer(m * k * size + 16), mc.DeviceBuffer(k * n * size + 16)
    for buf, x in ((da, a), (db, b)):
        src = mc.DeviceBuffer.from_array(x)
        if operands == "f32":
            mc.memcpy_dtod_async(buf.ptr + offset, src.ptr, 4 * x.size)
        else:
            mc.convert_f32(dtype, src.ptr, buf.ptr + offset, x.size)
        mc.synchronize()
    c = mc.DeviceBuffer.from_array(np.full(m * n + GUARD, np.nan, np.float32))
    ws = mc.DeviceBuffer(max(4, mc.matmul_workspace_bytes(kernel, m, n, splits)))
    pa, pb = da.ptr + offset, db.ptr + offset
    if operands == "f32":
        mc.launch_matmul(kernel, pa, pb, c.ptr, m, n, k, None, splits, ws.ptr)
    else:
        mc.launch_matmul_lowp(kernel, dtype, pa, pb, c.ptr, m, n, k, None, splits, ws.ptr)
    mc.synchronize()
    out = c.download()
    assert np.all(np.isnan(out[m * n:])), "a write past the end of C"
    bound = gamma(k) * absdot + 2 * U32 * np.abs(exact) + 1e-30
    assert np.all(np.abs(out[:m * n].astype(np.float64) - exact) <= bound)


@pytest.mark.parametrize("kernel,dtype", FORMATS)
def test_infinities_and_nans_stay_in_their_row_and_column(device, mc, oracle, kernel, dtype):
    m, n, k = 70, 131, 100  # a partial last step
    a, b = oracle.uniform(m * k, 7, 0.5, 1.0).reshape(m, k), oracle.uniform(k * n, 8, 0.5, 1.0).reshape(k, n)
    a[4, 0], a[m - 1, k - 1], b[0, 5] = np.inf, np.nan, np.inf
    want = np.zeros((m, n), bool)
    want[4, :], want[m - 1, :], want[:, 5] = True, True, True
    da, db, c = mc.DeviceBuffer.from_array(a), mc.DeviceBuffer.from_array(b), mc.DeviceBuffer(4 * m * n)
    mc.launch_matmul(kernel, da.ptr, db.ptr, c.ptr, m, n, k)
    mc.synchronize()
    assert np.array_equal(~np.isfinite(c.download().reshape(m, n)), want)


def test_a_missing_workspace_is_still_refused(device, mc):
    d = mc.DeviceBuffer(4 * 256 * 256)
    for m in (64, 256):
        with pytest.raises(mc.HipError):
            mc.launch_matmul("tensor_core_bf16", d.ptr, d.ptr, d.ptr, m, 64, 256, None, 4, None)
        with pytest.raises(mc.HipError):
            mc.launch_matmul_lowp("tensor_core_bf16", 1, d.ptr, d.ptr, d.ptr, m, 64, 256, None, 4, None)


@pytest.mark.parametrize("dtype", [1, 2], ids=["bf16", "f16"])
def test_the_packed_rounding_has_the_bits_of_the_plain_one(device, mc, dtype):
    # Every exponent with mantissas around each rounding point, both signs:
    # subnormals, infinities and NaNs among them.
    mant = np.array([0, 1, 0xFFF, 0x1000, 0x1001, 0x1FFF, 0x2000, 0x3000, 0x7FFF, 0x8000, 0x8001, 0xFFFF, 0x10000,
                     0x17FFF, 0x18000, 0x18001, 0x400000, 0x7FFFFF], np.uint32)
    bits = (np.arange(512, dtype=np.uint32)[:, None] << 23 | mant[None, :]).reshape(-1)
    k = 64
    x = bits[: bits.size // k * k].view(np.float32)
    m = x.size // k
    src, plain = mc.DeviceBuffer.from_array(x), mc.DeviceBuffer(2 * x.size)
    mc.convert_f32(dtype, src.ptr, plain.ptr, x.size)
    packed, want = mc.DeviceBuffer(mc.packed_a16_bytes(m, k)), mc.DeviceBuffer(mc.packed_a16_bytes(m, k))
    mc.convert_pack_a_f32(dtype, src.ptr, packed.ptr, m, k)
    mc.pack_a16(plain.ptr, want.ptr, m, k)
    mc.synchronize()
    got, ref = packed.download(np.uint16), want.download(np.uint16)
    inf = 0x7F80 if dtype == 1 else 0x7C00
    nan = (ref & 0x7FFF) > inf
    assert np.array_equal((got & 0x7FFF) > inf, nan)
    assert np.array_equal(got[~nan], ref[~nan])
