"""Air stages cut into z-slabs (flux kernels of a slab on a side stream, updates on the context stream as the
next slab's fluxes arrive) against the same stages unsliced: the same kernels compute the same values, so the
state after SSP-RK3 steps replayed from a hipGraph agrees bitwise, for the default setting and for thin slabs (8
planes), with the viscous node fluxes running beside the flux kernels.  The default cuts slabs of 16 planes where one of
them gives a direction's fluxes 2048 work-groups of 256 nodes, and leaves smaller blocks whole."""
import numpy as np
import pytest

import cases
import corefl
from parity import make_solver

pytestmark = pytest.mark.gpu


def _run(case, slab, steps=3):
    c = dict(case)
    c["setup"] = case["setup"] + f"\nint stage_slab_planes = {slab}\n"
    S = make_solver(c)
    S.advance(steps, graph=True)
    S.sync()
    out = S.get(corefl.CV), S.get(corefl.BV)
    S.close()
    return out


def _box(mx, my, mz, visc):
    """A Taylor-Green box on mx x my x mz nodes: that of the longest side, cut."""
    case = cases.tgv(max(mx, my, mz), recon=5, inviscid=3, visc=visc, cfl=0.5)
    return dict(case, grid=tuple(c[:mx, :my, :mz].copy() for c in case["grid"]),
                boundary=cases.boundary_text(cases.box_faces(mx, my, mz, 8)))


@pytest.mark.parametrize("visc", [4, 2])
@pytest.mark.parametrize("dims", [(97, 97, 97), (193, 170, 41)])
def test_slabbed_stages_equal_unsliced(dims, visc):
    # the first is whole by default and has 13 slabs of 8 planes, the second three by default, the last one thinner
    assert ((dims[0] * dims[1] + 255) // 256 * 16 >= 2048 and dims[2] >= 32) == (dims[0] == 193)
    case = _box(*dims, visc)
    print("case: tgv", dims, "viscous order", visc, flush=True)
    ref = _run(case, 0)
    for slab in (-1, 8):
        got = _run(case, slab)
        for a, b in zip(got, ref):
            np.testing.assert_array_equal(a, b, err_msg=f"slab {slab}")


def test_slab_setting_is_checked():
    case = cases.tgv(17)
    c = dict(case)
    c["setup"] = case["setup"] + "\nint stage_slab_planes = 12\n"
    with pytest.raises(corefl.CoreflError, match="stage_slab_planes"):
        make_solver(c)
