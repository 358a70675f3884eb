"""A cell gets the same bits from every launch of the chemistry, so that a run repeats although cells are handed from the
one-lane to the cooperative kernel at moments that scheduling sets."""
import numpy as np
import pytest

import chem_cases as CC
from test_thermo_sides_gpu import mechanism

pytestmark = pytest.mark.gpu

KEYS = ("T", "rhoY", "steps", "rejects")


def run(chem, cells, dt, *launch):
    rho, T, Y = cells
    chem.set_cells(rho, T, rho * Y)
    if launch:
        chem.set_launch(*launch)
    chem.integrate(dt)
    return chem.get_cells()


@pytest.mark.parametrize("common,both_sides", [(True, False), (False, False), (True, True)])
@pytest.mark.parametrize("n,dt,t_lo", [(1, 1e-6, 1500.0), (65, 1e-6, 900.0), (2001, 1e-6, 250.0)])
def test_modes_give_equal_bits(n, dt, t_lo, common, both_sides):
    """Up to some 1600 attempts a cell; fits read on one side and mixed; species that stand on both sides."""
    chem = mechanism(common, both_sides)
    cells = CC.random_states(n, seed=15, t_lo=t_lo)
    ref = run(chem, cells, dt, 0, 64, 0, 0)
    for launch in ((1, 128, 20, 0), (2, 64, 1, 0), (2, 256, 40, 0), (3, 64, 4, 1), (3, 64, 1024, 1), (3, 256, 64, 7)):
        got = run(chem, cells, dt, *launch)
        for k in KEYS:
            np.testing.assert_array_equal(got[k], ref[k], err_msg=f"{launch} {k}")


def test_default_launch_repeats():
    """More cells than lanes, so that the hand-over begins while waves are at work: the default launch twice, and the
    one-lane queue, which hands nothing over."""
    chem = mechanism(True)
    cells = CC.random_states(120_003, seed=3, t_lo=900.0)
    chem.set_cells(cells[0], cells[1], cells[0] * cells[2])
    first = run(chem, cells, 2e-7)
    assert chem.get_launch()["queue"] == 3
    assert 0 < chem.handed_over() < 120_003
    second = run(chem, cells, 2e-7)
    queue = run(chem, cells, 2e-7, 1, 64, 1024, 0)
    for k in KEYS:
        np.testing.assert_array_equal(first[k], second[k], err_msg=k)
        np.testing.assert_array_equal(first[k], queue[k], err_msg=k)
