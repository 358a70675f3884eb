"""Cells on either side of the thermo fits' middle temperature and outside their range, in wavefronts that lie on one side
or mix both: the fits' uniform and per-lane reads give the same cell the same result."""
import numpy as np
import pytest

import chem_cases as CC
import corefl

pytestmark = pytest.mark.gpu


def mechanism(common, both_sides=False):
    """The H2/air mechanism; common False: one species' middle temperature moved, so that no range is common; both_sides:
    with two reactions more, whose catalyst stands on both sides (once with another coefficient)."""
    therm, mech = open(CC.THERM).read(), open(CC.MECH).read()
    if both_sides:
        first = "H+O2=O+OH "
        assert mech.count(first) == 1
        mech = mech.replace(first, "O2+H2O=O+O+H2O 1.0E+15 -0.50 1.0E+05\nH+H2O=>H+H+OH 1.0E+10 0.30 3.0E+04\n" + first)
    if not common:
        line = next(l for l in therm.split("\n") if l.startswith("H2O2 ") and l.rstrip().endswith("1"))
        therm = therm.replace(line, line.replace("1000.00", " 999.00"))
    return corefl.Chemistry(mech_text=mech, therm_text=therm)


@pytest.mark.parametrize("common", [True, False])
def test_order_of_cells_does_not_change_a_cell(common):
    """The same cells sorted by temperature (waves on one side) and shuffled (mixed waves)."""
    n = 4096 + 37
    rho, T, Y = CC.random_states(n, seed=4, t_lo=250.0, t_hi=2600.0)
    T[:64], T[64:128], T[128:192] = 299.999, 300.0, 1000.0
    T[192:256] = np.linspace(999.0, 1001.0, 64)
    T[256:300] = 5100.0
    rho = CC.density(CC.PATM, T, Y)
    ch = mechanism(common)
    ch.set_launch(1, 64, 300, 0)
    out = []
    for order in (np.argsort(T, kind="stable"), np.random.default_rng(1).permutation(n)):
        ch.set_cells(rho[order], T[order], (rho * Y)[:, order])
        w = ch.source()
        ch.integrate(2e-8)
        g = ch.get_cells()
        inv = np.argsort(order)
        out.append((w[:, inv], g["e"][inv], g["T"][inv], g["rhoY"][:, inv], g["steps"][inv]))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_common_and_separate_ranges_agree():
    """Moving one trace species' middle temperature by 1 K changes no cell away from it beyond rounding: the mixture's own
    fit against the species-by-species iteration.  Temperatures differ by the iteration's tolerance (1e-8, squared by the
    quadratic convergence) and the rounding of sums of enthalpies ten times their result: 1e-12."""
    n = 3000
    rho, T, Y = CC.random_states(n, seed=6, t_lo=310.0, t_hi=2600.0)
    keep = np.abs(T - 1000.0) > 40.0
    rho, T, Y = rho[keep], T[keep], Y[:, keep]
    res = []
    for common in (True, False):
        ch = mechanism(common)
        ch.set_launch(0, 64, 0, 0)
        ch.set_cells(rho, T, rho * Y)
        ch.integrate(1e-9)
        g = ch.get_cells()
        res.append(g)
    assert np.max(np.abs(res[0]["T"] / res[1]["T"] - 1)) < 1e-12
    assert np.max(np.abs(res[0]["e"] - res[1]["e"]) / (np.abs(res[1]["e"]) + 1e5)) < 1e-13
