"""Periodic and outflow sides in one launch: the same run with every periodic face cut in two (which the library fills
face by face) gives the same arrays, on blocks from the thinnest the ghost layers allow upwards."""
import numpy as np
import pytest

import cases
import corefl

pytestmark = pytest.mark.gpu


def cut_faces(faces):
    """Each face of type 8 as two faces, split along its longest in-face direction."""
    out = []
    for f in faces:
        d = max((q for q in range(3) if f[2 * q] != f[2 * q + 1]), key=lambda q: f[2 * q + 1])
        if f[6] != 8:
            out.append(f)
            continue
        m = f[2 * d + 1] // 2
        lo, hi = list(f), list(f)
        lo[2 * d + 1], hi[2 * d] = m, m + 1
        out += [lo, hi]
    return out


def ragged(case, dims):
    """The case's periodic box cut down to dims nodes (the scheme and setup stay)."""
    mx, my, mz = dims
    grid = tuple(c[:mx, :my, :mz].copy() for c in case["grid"])
    return dict(case, grid=grid, faces=cases.box_faces(mx, my, mz, 8))


def run(case, faces, mixture, steps):
    S = corefl.Solver(setup_text=case["setup"], blocks=[case["grid"]], boundary_text=cases.boundary_text(faces))
    rng = np.random.default_rng(7)
    bv = S.get(corefl.BV).reshape(6, -1)
    noise = 1 + 0.01 * rng.uniform(-1, 1, bv.shape[1])
    bv[4] *= noise
    bv[0] *= noise  # p and rho: T stays
    bv[1:4] += 5.0 * rng.uniform(-1, 1, (3, bv.shape[1]))
    S.set_state(bv, sv=S.get(corefl.SV) if mixture else None)
    S.advance(steps, graph=True)
    S.sync()
    names = [corefl.BV, corefl.CV] + ([corefl.SV] if mixture else [])
    if S.get_int("viscous_order") > 0:
        names += [corefl.FV, corefl.GV, corefl.HV]
    out = [S.get(n) for n in names]
    S.close()
    return out


def compare(case, mixture):
    """The fills copy and average: bv and sv of a set state agree bitwise.  After steps, cv of a ghost may round its
    energy the other way in the other kernel (one ulp, 2.2e-16), which the WENO weights of six stages amplify by at
    most a few hundred."""
    cut = cut_faces(case["faces"])
    a, b = run(case, case["faces"], mixture, 0), run(case, cut, mixture, 0)
    assert np.array_equal(a[0], b[0])
    if mixture:
        assert np.array_equal(a[2], b[2])
    for x, y in zip(run(case, case["faces"], mixture, 2), run(case, cut, mixture, 2)):
        assert np.max(np.abs(x - y)) <= 1e-13 * np.max(np.abs(y))


@pytest.mark.parametrize("dims", [(6, 6, 6), (9, 7, 12), (10, 17, 9), (33, 12, 20)])
@pytest.mark.parametrize("recon,visc", [(5, 4), (4, 8), (4, 2), (4, 0)])
def test_air_periodic_sides_at_once(dims, recon, visc):
    compare(ragged(cases.tgv(33, recon=recon, inviscid=3, visc=visc, cfl=0.2), dims), False)


@pytest.mark.parametrize("dims", [(6, 6, 7), (8, 9, 6), (17, 9, 11)])
@pytest.mark.parametrize("visc", [0, 2, 8])
def test_mixture_periodic_sides_at_once(dims, visc):
    compare(ragged(cases.reactive_box(17, recon=4, inviscid=2, reaction=0, temporal=3, visc=visc, cfl=0.2), dims), True)
