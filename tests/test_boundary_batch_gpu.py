"""Periodic and outflow sides in one launch: the same run with every periodic face cut in two (which the library fills
face by face) and every outflow face in pieces (more than one launch takes) gives the same arrays, on blocks from the
thinnest the ghost layers allow upwards, with one, two and three periodic directions."""
import numpy as np
import pytest

import cases
import corefl

pytestmark = pytest.mark.gpu


def cut_faces(faces):
    """Each face of type 8 as two faces and each other one as three, split along its longest in-face direction."""
    out = []
    for f in faces:
        d = max((q for q in range(3) if f[2 * q] != f[2 * q + 1]), key=lambda q: f[2 * q + 1])
        n = 2 if f[6] == 8 else 3
        at = [round(q * (f[2 * d + 1] + 1) / n) for q in range(n + 1)]
        for lo, hi in zip(at[:-1], at[1:]):
            out.append(f[:2 * d] + [lo, hi - 1] + f[2 * d + 2:])
    return out


def ragged(case, dims, periodic=(0, 1, 2)):
    """The case's periodic box cut down to dims nodes (the scheme and setup stay), with outflow on the sides along which it
    is not periodic."""
    mx, my, mz = dims
    grid = tuple(c[:mx, :my, :mz].copy() for c in case["grid"])
    faces = [f[:6] + [8 if q // 2 in periodic else 6] for q, f in enumerate(cases.box_faces(mx, my, mz, 8))]
    only = "array string boundary_conditions {\n    periodic\n}"
    assert only in case["setup"]
    setup = case["setup"].replace(only, only.replace("periodic", "outflow periodic") +
                                  "\nstruct outflow {\n    string type = outflow\n    int label = 6\n}")
    return dict(case, setup=setup, grid=grid, faces=faces)


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
    assert 8 not in (f[6] for f in case["faces"]) or len(cut) > len(case["faces"])
    a, b = run(case, case["faces"], mixture, 0), run(case, cut, mixture, 0)
    assert np.array_equal(a[0], b[0])
    if mixture:
        assert np.array_equal(a[2], b[2])
    for x, y in zip(run(case, case["faces"], mixture, 2), run(case, cut, mixture, 2)):
        assert np.max(np.abs(x - y)) <= 1e-13 * np.max(np.abs(y))


@pytest.mark.parametrize("dims", [(6, 6, 6), (9, 7, 12), (10, 17, 9), (33, 12, 20), (20, 14, 1)])
@pytest.mark.parametrize("recon,visc", [(5, 4), (4, 8), (4, 2), (4, 0)])
def test_air_periodic_sides_at_once(dims, recon, visc):
    compare(ragged(cases.tgv(33, recon=recon, inviscid=3, visc=visc, cfl=0.2), dims), False)


@pytest.mark.parametrize("periodic", [(0,), (2,), (0, 1), (0, 2), (1, 2), ()])
@pytest.mark.parametrize("mixture", [False, True])
def test_outflow_sides_at_once(mixture, periodic):
    """Two to six outflow faces in one launch against six to eighteen (up to three launches), beside periodic sides; and
    every outflow ghost against the face node it copies."""
    dims = (12, 9, 17)
    if mixture:
        case = cases.reactive_box(17, recon=4, inviscid=2, reaction=0, temporal=3, visc=2, cfl=0.2)
    else:
        case = cases.tgv(33, recon=4, inviscid=3, visc=4, cfl=0.2)
    case = ragged(case, dims, periodic)
    compare(case, mixture)
    out = run(case, cut_faces(case["faces"]), mixture, 0)
    g = next(g for g in range(1, 8) if out[0].size == 6 * np.prod([m + 2 * g for m in dims]))
    shape = tuple(m + 2 * g for m in dims[::-1])
    # the nodes of periodic sides are averaged after they have been copied
    inner = [slice(g + (2 - q in periodic), g + m - (2 - q in periodic)) for q, m in enumerate(dims[::-1])]
    for q in ([out[0], out[2]] if mixture else [out[0]]):
        q = q.reshape((-1,) + shape)
        for d in set(range(3)) - set(periodic):
            ax = 2 - d
            for side, ghosts in ((g, range(g)), (g + dims[d] - 1, range(g + dims[d], 2 * g + dims[d]))):
                at = list(inner)
                at[ax] = side
                face = q[(slice(None), *at)]
                for k in ghosts:
                    at[ax] = k
                    np.testing.assert_array_equal(q[(slice(None), *at)], face)


@pytest.mark.parametrize("dims", [(6, 6, 7), (8, 9, 6), (17, 9, 11)])
@pytest.mark.parametrize("visc", [0, 2, 8])
def test_mixture_periodic_sides_at_once(dims, visc):
    compare(ragged(cases.reactive_box(17, recon=4, inviscid=2, reaction=0, temporal=3, visc=visc, cfl=0.2), dims), True)
