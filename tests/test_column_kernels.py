"""The column form of the elementwise kernels (broadcast inputs, odd counts),
without a GPU: the generated source compiled as host C++ and run lane by lane
against numpy's broadcasting, over every form of access it accepts."""

import ctypes
import itertools
import os
import subprocess

import numpy as np
import pytest

CLANG = "/opt/rocm/llvm/bin/clang++"

HOST = """
#include <cmath>
struct Dim { unsigned x; };
static thread_local Dim blockIdx, threadIdx, gridDim;
#define __device__
#define __forceinline__ inline
#define __global__ static
#define __launch_bounds__(n)
#define __restrict__
#define __builtin_amdgcn_sched_barrier(x)
#define extern
#define mc_c "C"
"""

# Output shape and the inputs' beside it: rows whose period is and is not a multiple of 4 or of 8, several periods, one
# longer than half the tensor; values per row (run a multiple of 4, odd, below 4) and per outer dimension; a middle
# dimension broadcast with a last one of either kind; scalars; odd counts; one row.
FORMS = [((512, 8), [(512, 8), (8,), ()]), ((333, 129), [(333, 129), (129,), (333, 1)]),
         ((401, 6), [(401, 6), (6,), (1, 6)]), ((64, 3, 40), [(3, 40), (40,), (64, 1, 1)]),
         ((5000, 3), [(5000, 3), (3,), (5000, 1)]), ((2, 2051), [(2051,), (2, 1), (2, 2051)]),
         ((1, 1027), [(1027,), (1, 1), (1, 1027)]), ((9, 20, 12), [(9, 1, 12), (20, 12), (9, 20, 1)]),
         ((9, 20, 13), [(9, 1, 13), (20, 13), (1, 20, 1)]), ((1025,), [(1025,), (1,), ()]),
         ((7, 5, 2, 31), [(7, 1, 1, 31), (5, 1, 1), (7, 5, 1, 1)]), ((1031, 2), [(1031, 1), (2,), (1031, 2)])]


def host_run(tmp_path, tag, src, out_count, inputs):
    src = src.replace('extern "C"', "")
    ptrs = ", ".join(f"in[{k}]" for k in range(len(inputs)))
    text = HOST + src + f"""
#undef extern
extern "C" void run(float* out, const float* const* in, unsigned n, unsigned blocks) {{
    gridDim.x = blocks;
    for (unsigned b = 0; b < blocks; ++b)
        for (unsigned t = 0; t < 256; ++t) {{ blockIdx.x = b; threadIdx.x = t; mc_elementwise(out, {ptrs}, n); }}
}}
"""
    cpp, so = tmp_path / f"{tag}.cpp", tmp_path / f"{tag}.so"
    cpp.write_text(text)
    subprocess.run([CLANG, "-x", "c++", "-std=c++17", "-O1", "-shared", "-fPIC", "-w", "-ffp-contract=off", str(cpp),
                    "-o", str(so)], check=True)
    fn = ctypes.CDLL(str(so)).run
    results = []
    for blocks in (1, 3, 64):  # fewer blocks loop; the same result from every grid
        out = np.full(out_count + 64, np.nan, np.float32)
        raw = np.zeros(out_count + 80, np.float32)
        shift = (-raw.ctypes.data % 16) // 4  # 16-byte aligned, as device buffers are
        buf = raw[shift:shift + out_count + 64]
        buf[:] = np.nan
        keep, args = [], (ctypes.c_void_p * len(inputs))()
        for k, a in enumerate(inputs):
            r = np.zeros(a.size + 4, np.float32)
            s = (-r.ctypes.data % 16) // 4
            r[s:s + a.size] = a.reshape(-1)
            keep.append(r)
            args[k] = r.ctypes.data + 4 * s
        fn(ctypes.c_void_p(buf.ctypes.data), args, out_count, blocks)
        assert np.all(np.isnan(buf[out_count:])), "a write past the end"
        results.append(buf[:out_count].copy())
    assert all(np.array_equal(results[0], r) for r in results[1:])
    return results[0]


@pytest.mark.parametrize("form", range(len(FORMS)))
@pytest.mark.parametrize("items", [1, 4])
def test_every_access_form_reads_what_broadcasting_says(mc, tmp_path, form, items):
    assert os.path.exists(CLANG)
    out, shapes = FORMS[form]
    rng, hoisted = np.random.default_rng(form), False
    for n, order in enumerate(itertools.permutations(range(3))):
        sh = [shapes[o] for o in order]
        decl = "".join(f"input x{k} : f32[{', '.join(map(str, s))}]\n" for k, s in enumerate(sh))
        full = f"input z : f32[{', '.join(map(str, out))}]\n"
        text = decl + full + "a = add z, x0\nb = mul a, x1\nc = sub b, x2\noutput c\n"
        c = mc.Compiled(text, passes="fuse", backend="none", options={"ew_items": items})
        (src,) = c.kernel_sources
        assert f"{items} item(s) per lane" in src and "vectors apart" in src
        hoisted = hoisted or "const mc_f32x4 h" in src
        ins = [rng.integers(-8, 9, size=s).astype(np.float32) for s in sh + [out]]
        want = (ins[3] + ins[0]) * ins[1] - ins[2]
        order_of = [int(i) for i in c.graph()["nodes"][c.graph()["outputs"][0]]["inputs"]]
        args = [ins[c.graph()["inputs"].index(i)] for i in order_of]
        got = host_run(tmp_path, f"k{n}", src, int(np.prod(out)), args)
        assert np.array_equal(got, want.reshape(-1).astype(np.float32)), (out, sh)
    assert hoisted == (items > 1 and form in (0, 1, 2, 3, 4, 7, 8, 11))


def test_small_counts_scalars_and_whole_vectors_keep_the_flat_form(mc):
    for text, column in (("input x : f32[40, 6]\ninput b : f32[6]\ny = add x, b\noutput y\n", False),
                         ("input x : f32[4096]\ninput s : f32[]\ny = add x, s\noutput y\n", False),
                         ("input x : f32[4097]\ny = neg x\noutput y\n", True),
                         ("input x : f32[256, 16]\ninput b : f32[16]\ny = add x, b\noutput y\n", True)):
        (src,) = mc.Compiled(text, passes="none", backend="none").kernel_sources
        assert ("vectors apart" in src) == column
        (flat,) = mc.Compiled(text, passes="none", backend="none", options={"vectorize": 0}).kernel_sources
        assert "vectors apart" not in flat


def test_rows_of_odd_period_take_the_column_form_for_large_counts_only(mc):
    for rows, cols, column in ((2032, 129, False), (2033, 129, True), (16, 250, True), (16, 129, False), (16384, 16, True)):
        text = f"input x : f32[{rows}, {cols}]\ninput b : f32[{cols}]\ny = add x, b\noutput y\n"
        (src,) = mc.Compiled(text, passes="none", backend="none").kernel_sources
        assert ("vectors apart" in src) == column, (rows, cols)
