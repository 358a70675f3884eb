"""The collision integrals by table and series, from far below to far above the temperatures of a flame: the viscous
residual and the viscous time step of a mixture against the oracle's powers."""
import numpy as np
import pytest

import cases
import chem_cases as CC
import corefl
from parity import make_mix_pair, make_solver, rel_err

pytestmark = pytest.mark.gpu

N = 13


@pytest.mark.parametrize("factor", [0.01, 0.1, 1.0, 30.0])
def test_viscous_residual_over_temperatures(factor):
    """Every T* + 0.55909 from the table's first sixteenths (3 K) to its tenth octave (70 000 K).  The bound is the one the
    viscous residual has elsewhere: rounding of its differences."""
    case = cases.reactive_box(N, recon=2, inviscid=4, temporal=3, reaction=0, visc=2)
    S, B = make_mix_pair(case)
    bv, sv = cases.reactive_state(N, S.get_int("ngg"))
    bv = bv.copy()
    bv[0] /= factor
    bv[5] *= factor
    S.set_state(bv, sv=sv)
    B.set_state(bv.ravel(), sv.ravel())
    S.rhs()
    err = rel_err(S.get(corefl.DQ).reshape(14, -1), B.rhs().reshape(14, -1))
    print("factor", factor, "rhs rel err", err, flush=True)
    assert np.max(err) < 1e-12
    dt = B.cfl_dt()
    assert abs(S.compute_dt() - dt) <= 1e-13 * dt


@pytest.mark.parametrize("depth", ["0.000", "-97.53"])
def test_well_depth_of_zero_or_less_gives_nan(depth, tmp_path):
    """T* is infinite, negative or NaN: no place in the table, and not a number in the fluxes that use it."""
    text = open(CC.TRAN_FILE).read()
    line = next(l for l in text.split("\n") if l.startswith("N2 "))
    path = tmp_path / "tran.dat"
    path.write_text(text.replace(line, line.replace("97.530", depth)))
    case = cases.reactive_box(N, recon=2, inviscid=4, temporal=3, reaction=0, visc=2)
    assert CC.TRAN_FILE in case["setup"]
    S = make_solver(dict(case, setup=case["setup"].replace(CC.TRAN_FILE, str(path))))
    S.rhs()
    S.sync()
    dq = S.get(corefl.DQ).reshape(14, -1)
    assert np.all(np.isfinite(dq[0]))
    assert np.all(np.isnan(dq[4:]))
