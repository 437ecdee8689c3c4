"""The column form of the elementwise kernels on the GPU: every form of access
that tests/test_column_kernels.py runs as host code, against numpy's
broadcasting. The inputs are small whole numbers, so every result is exact."""

import numpy as np
import pytest

from helpers import run_into_prefilled
from test_column_kernels import FORMS

pytestmark = pytest.mark.gpu

# Beside the host's forms: sizes at which a lane keeps its columns over several items by default, an odd row read once
# per lane and one read per vector, one value per row whose runs are odd, and counts that leave one to three elements.
LARGE = [((8001, 129), [(8001, 129), (129,), (8001, 1)]), ((7, 87383), [(87383,), (7, 1), ()]),
         ((70001, 15), [(15,), (70001, 1), (70001, 15)]), ((17, 60, 1027), [(17, 1, 1027), (60, 1027), (17, 60, 1)])]


def graph(out, shapes):
    decl = "".join(f"input x{k} : f32[{', '.join(map(str, s))}]\n" for k, s in enumerate(shapes))
    return decl + f"input z : f32[{', '.join(map(str, out))}]\na = add z, x0\nb = mul a, x1\nc = sub b, x2\noutput c\n"


def run(mc, out, shapes, seed, options):
    c = mc.Compiled(graph(out, shapes), options=options)
    (src,) = c.kernel_sources
    assert "vectors apart" in src
    rng = np.random.default_rng(seed)
    ins = [rng.integers(-8, 9, size=s).astype(np.float32) for s in [*shapes, out]]
    print(f"case column {out} {shapes} {options}", flush=True)
    got = run_into_prefilled(mc, c, [x.reshape(-1) for x in ins])[0]
    assert np.array_equal(got, ((ins[3] + ins[0]) * ins[1] - ins[2]).reshape(-1))
    return src


@pytest.mark.parametrize("items", [1, 4])
@pytest.mark.parametrize("form", range(len(FORMS)))
def test_small_forms(device, mc, form, items):
    out, shapes = FORMS[form]
    run(mc, out, shapes, form, {"ew_items": items})


@pytest.mark.parametrize("out,shapes", LARGE)
def test_several_items_per_lane(device, mc, out, shapes):
    run(mc, out, shapes, 7, {})


def test_the_forms_reach_the_wrapped_and_the_straddling_loads(device, mc):
    sources = [run(mc, out, shapes, 3, {}) for out, shapes in LARGE]
    assert any("mc_wrap4<" in s for s in sources) and any("mc_straddle<" in s for s in sources)
    assert any("const mc_f32x4 h" in s for s in sources)
