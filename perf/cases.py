"""What this framework is measured on: SSP-RK3 steps of air and of reacting mixtures, residuals, batched chemistry,
the chemistry surrogate and its training, through the entry points of corefl.py.

A case is a dict of plain values; `kind` names the family:
  tube       air shock tube (2D block), `steps` graph steps
  box        air in a periodic box on a uniform (amp 0) or wavy grid, `steps` graph steps
  channel    residual of an air channel with inflow, outflow, symmetry and periodic faces
  mixture    periodic box of igniting H2/air, Strang-split steps
  layer      reacting mixing layer of `blocks` blocks joined in a row, Strang-split steps
  chem       one exact chemistry sub-step of a batch of cells in the caller's device arrays
  surrogate  one surrogate chemistry sub-step of a batch, with the gate and the exact fallback
  train      Adam steps of the surrogate network
"""
import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "corefl-cpc_amd"))
import corefl  # noqa: E402

GOLDEN = os.path.join(ROOT, "tests", "golden")
MECH, THERM, TRAN = (os.path.join(GOLDEN, f) for f in ("h2_li2004.inp", "therm_h2o2n2.dat", "tran.dat"))
SPECIES = ("H2", "H", "O2", "O", "OH", "HO2", "H2O2", "H2O", "N2")
MW = (2.016, 1.008, 31.998, 15.999, 17.007, 33.006, 34.014, 18.015, 28.014)
RU, GAMMA, PATM = 8314.462618, 1.4, 101325.0
R_AIR = RU / 28.9647


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # The smallest call: the 1D shock tube every user starts with (the reference's example deck is 400 nodes),
        # ten steps between two outputs; launches and latency are all there is.
        dict(name="shock_tube_400", kind="tube", mx=400, my=7, recon=4, inviscid=4, steps=10),
        # A scheme-verification run of the Taylor-Green vortex on a coarse wavy grid: still bound by launches.
        dict(name="tgv_33", kind="box", mx=33, my=33, mz=33, amp=0.05, recon=5, inviscid=3, visc=4, steps=4),
        # The usual development size of a direct numerical simulation, uniform grid.
        dict(name="tgv_129", kind="box", mx=129, my=129, mz=129, amp=0.0, recon=5, inviscid=3, visc=4, steps=1),
        # The benchmark workload: 256^3 unique cells on the wavy curvilinear grid.
        dict(name="tgv_257", kind="box", mx=257, my=257, mz=257, amp=0.05, recon=5, inviscid=3, visc=4, steps=1),
        # The reference's own default shock-capturing scheme (Lax-Friedrichs-split characteristic WENO7) on a ragged
        # box.
        dict(name="llf_151x97x74", kind="box", mx=151, my=97, mz=74, amp=0.0, recon=5, inviscid=72, visc=4, steps=1),
        # The residual for an outer time integrator: channel with every physical boundary type, face-centred
        # second-order viscous fluxes.
        dict(name="channel_rhs_161x95x33", kind="channel", mx=161, my=95, mz=33, recon=4, inviscid=4, visc=2),
        # Reacting box with mixture transport at a mesh-study size.
        dict(name="reacting_65", kind="mixture", n=65, recon=4, inviscid=4, visc=2, steps=1),
        # The reacting benchmark: 128^3 unique cells, WENO5 + Roe, Strang-split stiff chemistry.
        dict(name="reacting_129", kind="mixture", n=129, recon=4, inviscid=2, visc=0, steps=1),
        # Reacting mixing layer on joined blocks: inflow noise, sponge, mixture transport, block exchange.
        dict(name="mixing_layer_3x96x64x32", kind="layer", blocks=3, mx=96, my=64, mz=32, recon=4, inviscid=4, steps=1),
        # Chemistry of another solver's cells in its own device arrays.
        dict(name="chem_200k", kind="chem", n=200003, dt=1e-6),
        # The learned sub-step of a reacting box: most cells in the gate, the hot kernels' cores exact.
        dict(name="surrogate_128", kind="surrogate", n=128 ** 3, dt=5e-8),
        # Training of the network: thousands of these steps per surrogate.
        dict(name="train_8192", kind="train", batch=8192, rows=131072, steps=20),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("tube", "box", "box", "box", "channel", "mixture", "mixture", "layer", "chem", "surrogate", "train"))
    if kind == "tube":
        return dict(kind=kind, mx=_log(rng, 101, 1601), my=rng.choice((5, 7, 9)), recon=rng.choice((4, 5)),
                    inviscid=rng.choice((2, 3, 4)), steps=rng.choice((1, 5, 10)))
    if kind == "box":
        return dict(kind=kind, mx=_log(rng, 17, 160), my=_log(rng, 17, 160), mz=_log(rng, 17, 160),
                    amp=rng.choice((0.0, 0.05)), recon=rng.choice((4, 5, 5)), inviscid=rng.choice((2, 3, 3, 4, 51, 52, 71, 72)),
                    visc=rng.choice((0, 2, 4, 4, 8)), steps=rng.choice((1, 2)))
    if kind == "channel":
        return dict(kind=kind, mx=_log(rng, 33, 240), my=_log(rng, 17, 130), mz=_log(rng, 9, 65), recon=rng.choice((4, 5)),
                    inviscid=rng.choice((2, 3, 4)), visc=rng.choice((2, 4)))
    if kind == "mixture":
        return dict(kind=kind, n=_log(rng, 17, 110), recon=4, inviscid=rng.choice((2, 3, 4)), visc=rng.choice((0, 2)),
                    steps=1)
    if kind == "layer":
        return dict(kind=kind, blocks=rng.choice((1, 2, 4)), mx=_log(rng, 33, 97), my=_log(rng, 25, 81),
                    mz=_log(rng, 9, 41), recon=4, inviscid=rng.choice((2, 4)), steps=1)
    if kind == "chem":
        return dict(kind=kind, n=_log(rng, 1000, 1000000), dt=10 ** rng.uniform(-7, -5.7))
    if kind == "surrogate":
        return dict(kind=kind, n=_log(rng, 5000, 3000000), dt=10 ** rng.uniform(-7.7, -7))
    return dict(kind=kind, batch=_log(rng, 500, 8192), rows=_log(rng, 20000, 200000), steps=rng.choice((10, 20)))


# ------------------------------------------------------------------------------------------------ device arrays
class _Device:
    """Device memory of the library as an array torch can wrap; keeps its owner alive as long as the tensor."""

    def __init__(self, ptr, shape, owner, typestr="<f8"):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr=typestr, data=(int(ptr), False), version=2)


def _wrap(ptr, shape, owner):
    return torch.as_tensor(_Device(ptr, shape, owner), device="cuda")


def _conserved(solver, b=0):
    """Density, momentum, energy, species partial densities and the temperature of the block's nodes."""
    v = solver.view(b)
    g, dims = v.ngg, (v.mz + 2 * v.ngg, v.my + 2 * v.ngg, v.mx + 2 * v.ngg)
    cut = (slice(None), slice(g, g + v.mz), slice(g, g + v.my), slice(g, g + v.mx))
    if v.mz == 1:
        return {"cv": _wrap(v.cv, (v.n_var,) + dims, solver)[cut]}
    cv, bv = _wrap(v.cv, (v.n_var,) + dims, solver)[cut], _wrap(v.bv, (6,) + dims, solver)[cut]
    out = {"density": cv[0], "momentum": cv[1:4], "energy": cv[4], "temperature": bv[5]}
    if v.n_spec:
        out["species"] = cv[5:]
    return out


# ------------------------------------------------------------------------------------------------ input decks
def _bounds(faces):
    return "\n".join(["%7d" % len(faces)] + ["".join("%7d" % v for v in f) for f in faces]) + "\n"


def _box_faces(mx, my, mz, kinds):
    """Faces i-, i+, j-, j+, k-, k+ of a block with the given boundary types (None: no face)."""
    r = [[0, 0, 0, my - 1, 0, mz - 1], [mx - 1, mx - 1, 0, my - 1, 0, mz - 1], [0, mx - 1, 0, 0, 0, mz - 1],
         [0, mx - 1, my - 1, my - 1, 0, mz - 1], [0, mx - 1, 0, my - 1, 0, 0], [0, mx - 1, 0, my - 1, mz - 1, mz - 1]]
    return [f + [k] for f, k in zip(r, kinds) if k is not None]


def _deck(scheme, **keys):
    """Setup text from typed keys, and the boundary structs given as text in `extra`."""
    extra = keys.pop("extra", "")
    rows = ["int gridIsBinary = 1", "bool steady = 0", "bool fixed_time_step = 0", "real cfl = 0.5",
            "int reconstruction = %d" % scheme["recon"], "int inviscid_scheme = %d" % scheme["inviscid"],
            "int viscous_order = %d" % scheme.get("visc", 0), "real prandtl_number = 0.72"]
    for k, v in keys.items():
        rows.append("%s %s = %s" % ("string" if isinstance(v, str) else "int" if isinstance(v, int) else "real", k,
                                    v if isinstance(v, (str, int)) else repr(v)))
    return "\n".join(rows) + "\n" + extra


_MIXTURE = dict(species=1, reaction=1, mechanism_file=MECH, therm_file=THERM, transport_file=TRAN, temporal_scheme=5)
_PERIODIC = "struct periodic {\n string type = periodic\n int label = 8\n}\n"
_OUTFLOW = "struct outflow {\n string type = outflow\n int label = 6\n}\n"


def _index_axes(dims, g, device="cuda"):
    """Padded node indices of a block as broadcastable float64 tensors (i, j, k) on axes (k, j, i)."""
    out = []
    for d, m in enumerate(dims):
        gd = 0 if m == 1 else g
        shape = [1, 1, 1]
        shape[2 - d] = -1
        out.append((torch.arange(m + 2 * gd, dtype=torch.float64, device=device) - gd).view(shape))
    return out


def _host(t):
    return np.ascontiguousarray(t.cpu().numpy())


def _rand(seed):
    return random.Random(int(seed) * 7919 + 17)


def _waves(rng, axes, count, amplitude, kmax=4):
    """Sum of `count` seeded sine waves of the angles `axes` (each 2 pi periodic)."""
    total = 0
    for _ in range(count):
        k = [rng.randint(1, kmax) for _ in axes]
        total = total + torch.sin(sum(q * a for q, a in zip(k, axes)) + rng.uniform(0, 2 * math.pi))
    return total * (amplitude / math.sqrt(count))


# ------------------------------------------------------------------------------------------------ air: box
_MACH, _T0 = 0.1, 300.0
_RHO0 = PATM / (R_AIR * _T0)
_V0 = _MACH * math.sqrt(GAMMA * R_AIR * _T0)


def _mu(T):
    return 1.7894e-5 * (T / 288.16) ** 1.5 * (288.16 + 110) / (T + 110)


_LEN = 1600.0 * _mu(_T0) / (_RHO0 * _V0)  # Re 1600


def _box_state(case, seed, g, device="cuda"):
    """rho, u, v, w, p, T on the padded nodes: the Taylor-Green vortex with seeded waves on it (Mach 0.1)."""
    dims, rng = (case["mx"], case["my"], case["mz"]), _rand(seed)
    tp = 2 * math.pi
    a = [tp * (x % (m - 1)) / (m - 1) for x, m in zip(_index_axes(dims, g, device), dims)]
    amp = case["amp"]
    X, Y, Z = (a[d] + tp * amp * torch.sin(a[(d + 1) % 3]) * torch.sin(a[(d + 2) % 3]) for d in range(3))
    u = _V0 * torch.sin(X) * torch.cos(Y) * torch.cos(Z) + _waves(rng, (X, Y, Z), 4, 0.1 * _V0)
    v = -_V0 * torch.cos(X) * torch.sin(Y) * torch.cos(Z) + _waves(rng, (X, Y, Z), 4, 0.1 * _V0)
    w = _waves(rng, (X, Y, Z), 4, 0.1 * _V0)
    p = PATM + _RHO0 * _V0 ** 2 / 16 * (torch.cos(2 * X) + torch.cos(2 * Y)) * (torch.cos(2 * Z) + 2)
    p = p + _waves(rng, (X, Y, Z), 2, 0.05 * _RHO0 * _V0 ** 2)
    T = _T0 + _waves(rng, (X, Y, Z), 3, 3.0)
    return torch.stack([p / (R_AIR * T), u, v, w, p, T])


def _box(case, seed):
    dims = (case["mx"], case["my"], case["mz"])
    s = [torch.arange(m, dtype=torch.float64, device="cuda") / (m - 1) for m in dims]
    s = [x.view([-1 if q == 2 - d else 1 for q in range(3)]) for d, x in enumerate(s)]
    full = (dims[2], dims[1], dims[0])
    tp = 2 * math.pi
    grid = []
    for d in range(3):
        c = tp * (s[d] + case["amp"] * torch.sin(tp * s[(d + 1) % 3]) * torch.sin(tp * s[(d + 2) % 3]))
        grid.append(_host(c.expand(full)).T)
    text = _deck(case, canonical_problem="taylorGreen", gridScale=_LEN, temporal_scheme=3,
                 extra="array string boundary_conditions {\n periodic\n}\n" + _PERIODIC +
                       "struct taylorGreen {\n real mach = 0.1\n real temperature = 300\n real pressure = 101325\n}\n")
    solver = corefl.Solver(setup_text=text, blocks=[grid], boundary_text=_bounds(_box_faces(*dims, [8] * 6)))
    solver.set_state(_host(_box_state(case, seed, solver.get_int("ngg"))))
    return solver


# ------------------------------------------------------------------------------------------------ air: shock tube
def _tube_sides(seed):
    """Density and pressure left and right of the diaphragm: Sod's states within ten per cent."""
    rng = _rand(seed)
    return [q * rng.uniform(0.9, 1.1) for q in (1.0, 1.0, 0.125, 0.1)]


def _tube(case, seed):
    mx, my = case["mx"], case["my"]
    x = np.linspace(0.0, 1.0, mx)
    X, Y, Z = np.meshgrid(x, (np.arange(my) - (my - 1) / 2) / 64.0, [0.0], indexing="ij")
    side = "struct left {\n string type = inflow\n int label = 5\n real velocity = 0\n real pressure = 1\n real density = 1\n}\n"
    text = _deck(case, canonical_problem="general", gridScale=1.0, temporal_scheme=3, default_init="left",
                 reference_state="left", extra="array string boundary_conditions {\n outflow\n}\n" + _OUTFLOW + side)
    faces = [[0, 0, 0, my - 1, 0, 0, 6], [mx - 1, mx - 1, 0, my - 1, 0, 0, 6], [0, mx - 1, 0, 0, 0, 0, 6],
             [0, mx - 1, my - 1, my - 1, 0, 0, 6]]
    solver = corefl.Solver(setup_text=text, blocks=[(X, Y, Z)], boundary_text=_bounds(faces))
    g = solver.get_int("ngg")
    rl, pl, rr, pr = _tube_sides(seed)
    bv = np.zeros((6, solver.view().sz // ((mx + 2 * g) * (my + 2 * g)), my + 2 * g, mx + 2 * g))
    left = (np.arange(mx + 2 * g) - g) / (mx - 1) < 0.5
    bv[0], bv[4] = np.where(left, rl, rr), np.where(left, pl, pr)
    bv[5] = bv[4] / (bv[0] * R_AIR)
    solver.set_state(bv)
    return solver


# ------------------------------------------------------------------------------------------------ air: channel
def _channel(case, seed):
    mx, my, mz = dims = (case["mx"], case["my"], case["mz"])
    size = (0.02, 0.01, 0.004)
    ax = [np.linspace(0.0, s, m) for s, m in zip(size, dims)]
    grid = np.meshgrid(*ax, indexing="ij")
    inlet = ("struct inlet {\n string type = inflow\n int label = 5\n real mach = 0.5\n real pressure = 101325\n"
             " real temperature = 300\n int inflow_sub = 1\n}\n")
    wall = "struct wall {\n string type = symmetry\n int label = 3\n}\n"
    text = _deck(case, canonical_problem="general", gridScale=1.0, temporal_scheme=3, default_init="inlet",
                 reference_state="inlet", extra="array string boundary_conditions {\n inlet outflow wall periodic\n}\n" +
                 inlet + _OUTFLOW + wall + _PERIODIC)
    solver = corefl.Solver(setup_text=text, blocks=[grid], boundary_text=_bounds(_box_faces(mx, my, mz, [5, 6, 3, 3, 8, 8])))
    rng, g = _rand(seed), solver.get_int("ngg")
    i, j, k = _index_axes(dims, g)
    a = (math.pi * i / (mx - 1), math.pi * j / (my - 1), 2 * math.pi * (k % (mz - 1)) / (mz - 1))
    c0 = math.sqrt(GAMMA * R_AIR * 300)
    u, v, w = (_waves(rng, a, 5, 0.05 * c0) for _ in range(3))
    p, T = PATM * (1 + _waves(rng, a, 4, 0.05)), 300 * (1 + _waves(rng, a, 4, 0.03))
    solver.set_state(_host(torch.stack([p / (R_AIR * T), u + 0.5 * c0, v, w, p, T])))
    return solver


# ------------------------------------------------------------------------------------------------ mixtures
def _y_stoich():
    x = [0.295775, 0, 0.147887, 0, 0, 0, 0, 0, 1 - 0.295775 - 0.147887]
    s = sum(a * b for a, b in zip(x, MW))
    return [a * b / s for a, b in zip(x, MW)]


def _y_burnt():
    x = [0, 0, 0, 0, 0, 0, 0, 2 * 0.295775, 1 - 0.295775 - 0.147887]
    s = sum(a * b for a, b in zip(x, MW))
    return [a * b / s for a, b in zip(x, MW)]


def _specific_gas(Y):
    return RU * sum(y / m for y, m in zip(Y, MW))


def _kernels(rng, idx, periods, count, radius):
    """Gaussian hot kernels in a box of `periods` cells: 0 far away, 1 at a centre (indices idx, axes broadcast)."""
    hot = 0
    for _ in range(count):
        r, top, d2 = rng.uniform(*radius), rng.uniform(0.7, 1.0), 0
        for x, n in zip(idx, periods):
            d = (x % n - rng.uniform(0, n)).abs()
            d2 = d2 + torch.minimum(d, n - d) ** 2
        hot = hot + top * torch.exp(-d2 / r ** 2)
    return hot.clamp(max=1.0)


def _mixture(case, seed):
    n = case["n"]
    s = np.linspace(0.0, 1.0, n)
    grid = np.meshgrid(s, s, s, indexing="ij")
    comp = "".join(" real %s = %r\n" % (k, y) for k, y in zip(SPECIES, _y_stoich()) if y > 0)
    fresh = "struct fresh {\n string type = inflow\n int label = 5\n real temperature = 300\n real pressure = 101325\n real velocity = 20\n%s}\n" % comp
    text = _deck(case, gridScale=1e-2, default_init="fresh", reference_state="fresh", **_MIXTURE,
                 extra="array string boundary_conditions {\n periodic\n}\n" + _PERIODIC + fresh)
    solver = corefl.Solver(setup_text=text, blocks=[grid], boundary_text=_bounds(_box_faces(n, n, n, [8] * 6)))
    # stoichiometric H2/air at 1 atm and 300 K with hot kernels (the benchmark's box: 16 in 128^3, radius 4 to 10
    # cells, 1800 to 2400 K), 20 m/s turbulence
    rng, g = _rand(seed), solver.get_int("ngg")
    idx = _index_axes((n, n, n), g)
    hot = _kernels(rng, idx, (n - 1,) * 3, max(2, round(16 * (n / 129) ** 3)), (min(4.0, n / 8), min(10.0, n / 5)))
    T = 300 + 2100 * hot
    a = [2 * math.pi * (x % (n - 1)) / (n - 1) for x in idx]
    u, v, w = (_waves(rng, a, 6, 16.0, kmax=6) for _ in range(3))
    R = _specific_gas(_y_stoich())
    full = T.shape
    bv = torch.stack([PATM / (R * T), u.expand(full), v.expand(full), w.expand(full), torch.full_like(T, PATM), T])
    sv = np.repeat(np.array(_y_stoich())[:, None], T.numel(), axis=1)
    solver.set_state(_host(bv), sv=sv)
    return solver


def _inner(records):
    """inner file text: per block, pairs of (own range + id, partner range + id)."""
    rows = ["%9d" % sum(len(r) for r in records), "".join("%9d\t" % len(r) for r in records),
            "iMin  iMax  jMin  jMax  kMin  kMax   id"]
    rows += ["".join("%9d" % v for v in t) for r in records for pair in r for t in pair]
    return "\n".join(rows) + "\n"


_UPPER = dict(T=600.0, mach=0.32, U=300.0, Y={"H2": 0.2, "N2": 0.8})
_LOWER = dict(T=1200.0, mach=0.89, U=600.0, Y={"O2": 0.233, "N2": 0.767})


def _layer(case, seed):
    nb, mx, my, mz = case["blocks"], case["mx"], case["my"], case["mz"]
    h = 0.08 / (8 * 383)  # the spacing of the full mixing layer: eight blocks of 384 nodes over 8 cm
    length, height = h * nb * (mx - 1), h * (my - 1)
    stream = ""
    for name, st in (("upper_stream", _UPPER), ("lower_stream", _LOWER)):
        stream += "struct %s {\n real temperature = %r\n real pressure = %r\n real mach = %r\n real mixture_fraction = 0\n%s}\n" % (
            name, st["T"], PATM, st["mach"], "".join(" real %s = %r\n" % kv for kv in st["Y"].items()))
    inlet = "struct inlet {\n string type = inflow\n int label = 5\n int fluctuation_type = 1\n real fluctuation_intensity = 0.02\n}\n"
    sponge = ("bool sponge_layer = 1\nint spongeX = 2\nreal spongeXPlusStart = %r\nreal spongeXPlusEnd = %r\n"
              "real spongeCoefficient = 1.0\nint fluctuation_seed = 5\n" % (0.9 * length, length))
    text = _deck(dict(case, visc=2), canonical_problem="mixingLayer", gridScale=1.0, delta_omega=height / 10, ma_c=0.0,
                 default_init="inlet", reference_state="inlet", **_MIXTURE,
                 extra=stream + "array string boundary_conditions {\n inlet outflow periodic\n}\n" + inlet + _OUTFLOW +
                 _PERIODIC + sponge)
    grids, faces, records = [], "", []
    for b in range(nb):
        ax = (h * (np.arange(mx) + b * (mx - 1)), h * (np.arange(my) - (my - 1) / 2), h * np.arange(mz))
        grids.append(np.meshgrid(*ax, indexing="ij"))
        faces += _bounds(_box_faces(mx, my, mz, [5 if b == 0 else None, 6 if b == nb - 1 else None, 6, 6, 8, 8]))
        rec = []
        if b > 0:
            rec.append(((1, 1, -1, -my, 1, mz, b + 1), (mx, mx, -1, -my, 1, mz, b)))
        if b < nb - 1:
            rec.append(((mx, mx, -1, -my, 1, mz, b + 1), (1, 1, -1, -my, 1, mz, b + 2)))
        records.append(rec)
    solver = corefl.Solver(setup_text=text, blocks=grids, boundary_text=faces, inner_text=_inner(records) if nb > 1 else None)
    rng, g = _rand(seed), solver.get_int("ngg")
    waves = [rng.getrandbits(30) for _ in range(3)]
    for b in range(nb):
        i, j, k = _index_axes((mx, my, mz), g)
        i = i + b * (mx - 1)
        y = j - (my - 1) / 2
        mix = 0.5 * (1 + torch.tanh(2 * y / (0.1 * (my - 1))))  # 1: upper stream
        a = (2 * math.pi * i / 64, math.pi * j / (my - 1), 2 * math.pi * (k % (mz - 1)) / (mz - 1))
        d = [_waves(random.Random(s), a, 4, 15.0) for s in waves]
        Y = [mix * _UPPER["Y"].get(s, 0.0) + (1 - mix) * _LOWER["Y"].get(s, 0.0) for s in SPECIES]
        T = mix * _UPPER["T"] + (1 - mix) * _LOWER["T"]
        full = torch.broadcast_shapes(i.shape, j.shape, k.shape)
        u = mix * _UPPER["U"] + (1 - mix) * _LOWER["U"] + d[0]
        rho = PATM / (_specific_gas(Y) * T)
        p = torch.full(full, PATM, dtype=torch.float64, device="cuda")
        bv = torch.stack([q.expand(full) for q in (rho, u, d[1], d[2], p, T)])
        solver.set_state(_host(bv), b, sv=_host(torch.stack([q.expand(full) for q in Y])))
    return solver


# ------------------------------------------------------------------------------------------------ chemistry batches
def _cells(n, seed):
    """rho, T and rhoY (9, n) of a box of n cells in index order: fresh H2/air with hot kernels at a seeded reaction
    progress with radicals in them."""
    side, rng = math.ceil(n ** (1 / 3)), _rand(seed)
    idx = _index_axes((side,) * 3, 0)
    hot = _kernels(rng, idx, (side,) * 3, max(2, round(16 * (side / 128) ** 3)), (min(4.0, side / 8), min(10.0, side / 5)))
    hot = hot.reshape(-1)[:n].contiguous()
    T = 300 + 2100 * hot
    torch.manual_seed(seed)
    noise = torch.rand(n, dtype=torch.float64, device="cuda")
    prog = hot * (0.2 + 0.6 * noise)
    fresh, burnt = (torch.tensor(y, dtype=torch.float64, device="cuda")[:, None] for y in (_y_stoich(), _y_burnt()))
    radical = torch.tensor([0, 2e-3, 0, 2e-3, 4e-3, 5e-4, 2e-4, 0, 0], dtype=torch.float64, device="cuda")[:, None]
    Y = fresh * (1 - prog) + burnt * prog + radical * prog * (1 - prog)
    Y = Y / Y.sum(0)
    rho = PATM / (RU * T * sum(Y[k] / MW[k] for k in range(9)))
    return rho, T, (rho * Y).contiguous()


_stream = None


def _work_stream():
    """One stream for all chemistry batches: corefl_chem_integrate_noalloc shares its working memory per GPU."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


def _chem(case, seed):
    rho, T, rhoY = _cells(case["n"], seed)
    ch = corefl.Chemistry(MECH, THERM)
    # the context's tables, and each cell's internal energy from its state
    ch.set_cells(_host(rho), _host(T), _host(rhoY))
    e = torch.from_numpy(ch.get_cells()["e"]).cuda()
    torch.cuda.synchronize()
    return dict(ch=ch, rho=rho, e=e, T0=T, rhoY0=rhoY, T=T.clone(), rhoY=rhoY.clone(), stream=_work_stream())


def _network(seed):
    """A network of the surrogate's shape with weights as training leaves them (He-scaled)."""
    rng = np.random.default_rng(seed)
    sizes = corefl.SURROGATE_SIZES
    return [((rng.standard_normal((k, n)) * math.sqrt(2 / k) * (0.3 if n == 10 else 1)).astype(np.float32),
             (0.05 * rng.standard_normal(n)).astype(np.float32)) for k, n in zip(sizes[:-1], sizes[1:])]


def _surrogate(case, seed):
    rho, T, rhoY = _cells(case["n"], seed)
    ch = corefl.Chemistry(MECH, THERM)
    ch.set_cells(_host(rho), _host(T), _host(rhoY))
    sur = corefl.Surrogate(1024)
    sur.set_params(_network(seed))
    sur.set_scaling([1000, 11.5] + [0.4] * 9 + [math.log(3e-8)], [800, 0.5] + [0.3] * 9 + [1.0], [0.0] * 10, [1.0] * 10)
    sur.set_transform(0.1, [1e3] * 9 + [1e6])
    # the network inside its box; the kernels' cores are hotter and go to the exact integrator
    sur.set_gate(250.0, 1500.0, 0.2 * PATM, 5 * PATM, 1e-9, 1e-6, 1e30, 1e30)
    v = ch.view()
    state = dict(ch=ch, sur=sur, T=_wrap(v.T, (v.n,), ch), rhoY=_wrap(v.rhoY, (9, v.n), ch), h=_wrap(v.h, (v.n,), ch),
                 T0=T, rhoY0=rhoY)
    torch.cuda.synchronize()
    return state


def _train_data(case, seed):
    """Scaled features and targets: a smooth map of twelve normal features with a little noise, and the first weights."""
    rng = np.random.default_rng(seed)
    X = rng.standard_normal((case["rows"], 12)).astype(np.float32)
    A, B = rng.standard_normal((12, 24)) / math.sqrt(12), rng.standard_normal((24, 10)) / math.sqrt(24)
    Y = (np.tanh(X @ A) @ B + 0.05 * rng.standard_normal((case["rows"], 10))).astype(np.float32)
    return X, Y, _network(seed)


def _train(case, seed):
    X, Y, net = _train_data(case, seed)
    sur = corefl.Surrogate(8192)
    sur.set_params(net)
    sur.set_data(X, Y)
    return dict(sur=sur)


# ------------------------------------------------------------------------------------------------ the interface
def prepare(case, seed):
    kind = case["kind"]
    make = dict(tube=_tube, box=_box, channel=_channel, mixture=_mixture, layer=_layer, chem=_chem, surrogate=_surrogate,
                train=_train)[kind]
    return dict(case=case, of=make(case, seed))


def run(state):
    case, s = state["case"], state["of"]
    kind = case["kind"]
    if kind in ("tube", "box", "mixture", "layer"):
        s.advance(case["steps"])
        out = [_conserved(s, b) for b in range(case.get("blocks", 1))]
        return out if kind == "layer" else out[0]
    if kind == "channel":
        s.rhs()
        v = s.view()
        dq = _wrap(v.dq, (5, v.mz, v.my, v.mx), s)
        return {"density": dq[0], "momentum": dq[1:4], "energy": dq[4]}
    if kind == "chem":
        with torch.cuda.stream(s["stream"]):  # new cells arrive in the caller's arrays
            s["T"].copy_(s["T0"])
            s["rhoY"].copy_(s["rhoY0"])
        s["ch"].integrate_noalloc(s["T"].numel(), s["rho"].data_ptr(), s["e"].data_ptr(), s["T"].data_ptr(),
                                  s["rhoY"].data_ptr(), case["dt"], stream=s["stream"].cuda_stream)
        return {"T": s["T"], "rhoY": s["rhoY"]}
    if kind == "surrogate":
        s["T"].copy_(s["T0"])
        s["rhoY"].copy_(s["rhoY0"])
        s["h"].zero_()
        torch.cuda.current_stream().synchronize()  # the batch is refilled on another stream than the context's
        n_fallback = s["sur"].chem_step(s["ch"], case["dt"])
        return {"T": s["T"], "rhoY": s["rhoY"], "fallback": n_fallback}
    loss = s["sur"].train(case["batch"], case["steps"], 1e-3, seed=11)
    return {"loss": loss, "params": s["sur"].get_params(flat=True)}


# FP64 operations of one interface flux (a fused multiply-add counts twice): the WENO halves of five fields, the
# projection and the Riemann solver; LLF splitting reconstructs two split fluxes per field.
_FLUX_FLOP = {(5, False): 2480, (4, False): 1500, (5, True): 3000, (4, True): 2000}


def work(case):
    """Compulsory traffic of an SSP-RK3 step: per stage the state in and out (8 B x n_var each) and the metrics and
    Jacobian (80 B), and U^n in twice; chemistry reads and writes 112 B per cell and sub-step."""
    kind = case["kind"]
    if kind in ("tube", "box"):
        dims = 2 if kind == "tube" else 3
        cells = case["mx"] * case["my"] * case.get("mz", 1)
        llf = case["inviscid"] > 50
        order = 5 if (case["inviscid"] // 10 == 7 if llf else case["recon"] == 5) else 4
        per = 3 * (dims * _FLUX_FLOP[order, llf] + (300 if case.get("visc", 0) else 0) + 60)
        return {"bytes": 560.0 * cells * case["steps"], "flops": float(per) * cells * case["steps"]}
    if kind == "channel":
        cells = case["mx"] * case["my"] * case["mz"]
        return {"bytes": 160.0 * cells, "flops": (3 * _FLUX_FLOP[case["recon"], False] + 300.0) * cells}
    if kind in ("mixture", "layer"):
        cells = case["n"] ** 3 if kind == "mixture" else case["blocks"] * case["mx"] * case["my"] * case["mz"]
        transport = 3000 if case.get("visc", 2) else 0
        per = 3 * (3 * 5000 + transport + 1500) + 2 * 40000  # one attempt of the stiff integrator per sub-step
        return {"bytes": (1136.0 + 2 * 224) * cells * case["steps"], "flops": float(per) * cells * case["steps"]}
    if kind == "chem":
        return {"bytes": 184.0 * case["n"], "flops": 2 * 40000.0 * case["n"]}
    if kind == "surrogate":
        return {"bytes": 168.0 * case["n"], "flops": 103936.0 * case["n"]}
    params = 52490
    return {"bytes": case["steps"] * (88.0 * case["batch"] + 28 * params), "flops": 3.0 * 103936 * case["batch"] * case["steps"]}


def tolerance(case):
    """FP64 flow: perturbing the inputs by an ulp moves the results by up to 1e-14 (2-norm) and 6e-13 (single values)
    over these ranges, a residual by 3e-14 and 2e-13; two orders above that for other operation orders over ten steps.
    Chemistry: an accept decision of the adaptive integrator (rtol 1e-6) that rounding turns in a cell.  Surrogate and
    training: BF16 rounding of the activations (the training is 6e-4 from its 64-bit result)."""
    kind = case["kind"]
    if kind in ("tube", "box", "channel"):
        return {"rel": 1e-12, "max": 1e-10}
    if kind in ("mixture", "layer"):
        return {"rel": 1e-11, "max": 1e-8}
    if kind == "chem":
        return {"rel": 1e-9, "max": 1e-5}
    if kind == "surrogate":
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 3e-3, "max": 0.3}


# ------------------------------------------------------------------------------------------------ 64-bit results
# Plain torch for the shock tube, the uniform periodic box with collocated fourth-order or no viscous fluxes, and the
# training.  The wavy grid's ghost metrics, the second-order viscous scheme's edge ghosts and the boundary conditions
# of the channel are this framework's input contract rather than a formula, and stiff mixtures integrated adaptively
# to a tolerance have no closed reference: None.
def _shift(U, o, axis, periodic):
    """U at node t + o along `axis`; beyond the ends periodic or the end value."""
    if periodic:
        return torch.roll(U, -o, axis)
    n = U.shape[axis]
    return U.index_select(axis, (torch.arange(n, device=U.device) + o).clamp(0, n - 1))


def _weno5(v, eps):
    q = ((2 * v[0] - 7 * v[1] + 11 * v[2]) / 6, (-v[1] + 5 * v[2] + 2 * v[3]) / 6, (2 * v[2] + 5 * v[3] - v[4]) / 6)
    b = [13 / 12 * (v[k] - 2 * v[k + 1] + v[k + 2]) ** 2 + 0.25 * f ** 2 for k, f in
         enumerate((v[0] - 4 * v[1] + 3 * v[2], v[1] - v[3], 3 * v[2] - 4 * v[3] + v[4]))]
    a = [d / (eps + x) ** 2 for d, x in zip((0.1, 0.6, 0.3), b)]
    return (a[0] * q[0] + a[1] * q[1] + a[2] * q[2]) / (a[0] + a[1] + a[2])


def _weno7(v, eps):
    s1 = ((-2 * v[0] + 9 * v[1] - 18 * v[2] + 11 * v[3]) / 6, (v[1] - 6 * v[2] + 3 * v[3] + 2 * v[4]) / 6,
          (-2 * v[2] - 3 * v[3] + 6 * v[4] - v[5]) / 6, (-11 * v[3] + 18 * v[4] - 9 * v[5] + 2 * v[6]) / 6)
    s2 = (-v[0] + 4 * v[1] - 5 * v[2] + 2 * v[3], v[2] - 2 * v[3] + v[4], v[2] - 2 * v[3] + v[4],
          2 * v[3] - 5 * v[4] + 4 * v[5] - v[6])
    s3 = [-v[k] + 3 * v[k + 1] - 3 * v[k + 2] + v[k + 3] for k in range(4)]
    b = [x * x + 13 / 12 * y * y + 1043 / 960 * z * z + x * z / 12 for x, y, z in zip(s1, s2, s3)]
    tau = (b[0] + 3 * b[1] - 3 * b[2] - b[3]) ** 2
    a = [c / 35 * (1 + tau / (eps + x) ** 2) for c, x in zip((1, 12, 18, 4), b)]
    q = (-3 * v[0] + 13 * v[1] - 23 * v[2] + 25 * v[3], v[1] - 5 * v[2] + 13 * v[3] + 3 * v[4],
         -v[2] + 7 * v[3] + 7 * v[4] - v[5], 3 * v[3] + 13 * v[4] - 5 * v[5] + v[6])
    return sum(x * y for x, y in zip(a, q)) / (12 * sum(a))


def _pressure(U):
    return (GAMMA - 1) * (U[4] - 0.5 * (U[1] ** 2 + U[2] ** 2 + U[3] ** 2) / U[0])


def _ausm(L, R, d):
    (pl, pr), cm = (_pressure(L), _pressure(R)), 1 + d
    c = 0.5 * (torch.sqrt(GAMMA * pl / L[0]) + torch.sqrt(GAMMA * pr / R[0]))
    ml, mr = L[cm] / L[0] / c, R[cm] / R[0] / c
    split = []
    for m, s in ((ml, 1.0), (mr, -1.0)):
        a, b = 0.25 * (m + s) ** 2, (m * m - 1) ** 2
        out = m.abs() > 1
        half = 0.5 * (m + s * m.abs())
        split.append((torch.where(out, half, s * (a + 0.125 * b)),
                      torch.where(out, half / m, a * (2 - s * m) + s * 3 / 16 * m * b)))
    mh = split[0][0] + split[1][0]
    mass = c * (L[0] * 0.5 * (mh + mh.abs()) + R[0] * 0.5 * (mh - mh.abs()))
    S, p = torch.where(mass >= 0, L, R), torch.where(mass >= 0, pl, pr)
    F = mass * torch.stack([torch.ones_like(p), S[1] / S[0], S[2] / S[0], S[3] / S[0], (S[4] + p) / S[0]])
    F[cm] += split[0][1] * pl + split[1][1] * pr
    return F


def _hllc(L, R, d):
    cm = 1 + d
    pl, pr, ul, ur = _pressure(L), _pressure(R), L[cm] / L[0], R[cm] / R[0]
    wl, wr = (torch.sqrt(q[0]) / (torch.sqrt(L[0]) + torch.sqrt(R[0])) for q in (L, R))
    v = [wl * L[q] / L[0] + wr * R[q] / R[0] for q in (1, 2, 3)]
    H = wl * (L[4] + pl) / L[0] + wr * (R[4] + pr) / R[0]
    c = torch.sqrt((GAMMA - 1) * (H - 0.5 * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2)))
    sl = torch.minimum(ul - torch.sqrt(GAMMA * pl / L[0]), v[d] - c)
    sr = torch.maximum(ur + torch.sqrt(GAMMA * pr / R[0]), v[d] + c)
    dl, dr = L[0] * (sl - ul), R[0] * (sr - ur)
    sm = (R[0] * ur * (sr - ur) - L[0] * ul * (sl - ul) + pl - pr) / (dr - dl)
    pm = dl * (sm - ul) + pl

    def side(U, p, u, s):
        F = U * u
        F[cm] += p
        F[4] += p * u
        star = U * ((s - u) / (s - sm))
        star[cm] += (pm - p) / (s - sm)
        star[4] += (pm * sm - p * u) / (s - sm)
        return F, F + s * (star - U)

    (fl, gl), (fr, gr) = side(L, pl, ul, sl), side(R, pr, ur, sr)
    return torch.where(sl >= 0, fl, torch.where(sr < 0, fr, torch.where(sm >= 0, gl, gr)))


def _roe_frame(a, b):
    ca, cb = 1 / (a[0] + torch.sqrt(a[0] * b[0])), 1 / (b[0] + torch.sqrt(a[0] * b[0]))
    pa, pb = _pressure(a), _pressure(b)
    u = [ca * a[q] + cb * b[q] for q in (1, 2, 3)]
    return u, ca * (a[4] + pa) + cb * (b[4] + pb), ca * pa + cb * pb


def _interface(U, d, r, eps, solver, periodic):
    """Flux between nodes t and t + 1 along d per unit area: characteristic WENO of the conserved variables and a
    Riemann solver, or of the Lax-Friedrichs-split fluxes (solver None)."""
    axis, cm = 3 - d, 1 + d
    t1, t2 = [1 + q for q in range(3) if q != d]
    nodes = [_shift(U, m - r + 1, axis, periodic) for m in range(2 * r)]
    u, H, pr = _roe_frame(nodes[r - 1], nodes[r])
    ek = 0.5 * (u[0] ** 2 + u[1] ** 2 + u[2] ** 2)
    c2 = (GAMMA - 1) * (H - ek) if solver else GAMMA * pr
    c, g1 = torch.sqrt(c2), GAMMA - 1

    def project(q):
        X = ek * q[0] + q[4] - u[0] * q[1] - u[1] * q[2] - u[2] * q[3]
        Y = u[d] * q[0] - q[cm]
        return [(g1 * X + c * Y) / (2 * c2), q[t1] - u[t1 - 1] * q[0], q[t2] - u[t2 - 1] * q[0], q[0] - g1 * X / c2,
                (g1 * X - c * Y) / (2 * c2)]

    def back(W):
        s, df = W[0] + W[3] + W[4], c * (W[0] - W[4])
        Q = [s, None, None, None, H * s - u[d] * df + u[t1 - 1] * W[1] + u[t2 - 1] * W[2] - c2 / g1 * W[3]]
        Q[cm], Q[t1], Q[t2] = u[d] * s - df, u[t1 - 1] * s + W[1], u[t2 - 1] * s + W[2]
        return torch.stack(Q)

    weno = _weno7 if r == 4 else _weno5
    if solver:
        w = [project(q) for q in nodes]
        L = back([weno([x[l] for x in w[:-1]], eps) for l in range(5)])
        R = back([weno([x[l] for x in w[:0:-1]], eps) for l in range(5)])
        return solver(L, R, d)
    lam = torch.stack([(q[cm] / q[0]).abs() + torch.sqrt(GAMMA * _pressure(q) / q[0]) for q in nodes]).amax(0)

    def split(q, s):
        F = q * (q[cm] / q[0])
        F[cm] += _pressure(q)
        F[4] += _pressure(q) * q[cm] / q[0]
        return project(0.5 * (F + s * lam * q))

    plus, minus = [split(q, 1.0) for q in nodes[:-1]], [split(q, -1.0) for q in nodes[:0:-1]]
    return back([weno([x[l] for x in plus], eps) + weno([x[l] for x in minus], eps) for l in range(5)])


def _viscous(U, h):
    """Divergence of the collocated viscous fluxes, fourth-order central differences on the periodic box."""
    def dd(f, d):
        s = [torch.roll(f, -o, 2 - d) for o in (-2, -1, 1, 2)]
        return ((s[0] - s[3]) / 12 + 2 / 3 * (s[2] - s[1])) / h[d]

    vel = [U[q] / U[0] for q in (1, 2, 3)]
    T = _pressure(U) / (U[0] * R_AIR)
    g = [[dd(f, d) for d in range(3)] for f in vel]
    mu, cp = _mu(T), GAMMA * R_AIR / (GAMMA - 1)
    div = g[0][0] + g[1][1] + g[2][2]
    out = torch.zeros_like(U)
    for d in range(3):
        tau = [mu * (g[q][d] + g[d][q] - (2 / 3 * div if q == d else 0)) for q in range(3)]
        heat = sum(v * t for v, t in zip(vel, tau)) + mu * cp / 0.72 * dd(T, d)
        for q, f in enumerate(tau + [heat]):
            out[1 + q] += dd(f, d)
    return out


def _march(U, h, steps, r, eps, solver, visc, periodic):
    """SSP-RK3 steps at CFL 0.5 of U[5][z][y][x]; h: the spacing of every direction that is solved."""
    for _ in range(steps):
        T = _pressure(U) / (U[0] * R_AIR)
        c = torch.sqrt(GAMMA * R_AIR * T)
        s = torch.stack([((U[1 + d] / U[0]).abs() + c) / h[d] for d in range(len(h))]).amax(0)
        if visc:
            s = torch.maximum(s, max(GAMMA, 4 / 3) / U[0] * (_mu(T) / 0.72) / min(h) ** 2)
        dt = 0.5 / s.max()
        U0 = U
        for a, b, w in ((1.0, 0.0, 1.0), (0.75, 0.25, 0.25), (1 / 3, 2 / 3, 2 / 3)):
            rhs = _viscous(U, h) if visc else 0
            for d in range(len(h)):
                if not periodic and d > 0:
                    continue  # the shock tube is uniform along y
                F = _interface(U, d, r, eps, solver, periodic)
                low = _interface_low(U, F, d, r, eps, solver, periodic)
                rhs = rhs - (F - low) / h[d]
            U = a * U0 + b * U + w * dt * rhs
    return U


def _interface_low(U, F, d, r, eps, solver, periodic):
    """The flux at t - 1/2: the neighbour's, and at the first node that of the stencil shifted into the ghosts."""
    low = torch.roll(F, 1, 3 - d)
    if not periodic:
        n = U.shape[3 - d]
        first = torch.cat([U[..., :1]] * (r + 1) + [U[..., : min(n, r + 1)]], 3 - d)
        low[..., 0] = _interface(first, d, r, eps, solver, False)[..., r]
    return low


def _exact_flow(case, seed):
    solver = {2: False, 3: _ausm, 4: _hllc, 72: None, 52: None}.get(case["inviscid"], False)
    if solver is False:
        return None
    r = 4 if (case["recon"] == 5 if solver else case["inviscid"] == 72) else 3
    if case["kind"] == "tube":
        if r != 3 and solver is None:
            return None
        mx, my = case["mx"], case["my"]
        rl, pl, rr, pr = _tube_sides(seed)
        left = np.arange(mx) / (mx - 1) < 0.5
        U = torch.zeros((5, 1, my, mx), dtype=torch.float64, device="cuda")
        U[0], U[4] = (torch.from_numpy(a).cuda() for a in (np.where(left, rl, rr), np.where(left, pl, pr) / (GAMMA - 1)))
        U = _march(U, (1 / (mx - 1), 1 / 64), case["steps"], r, 1e-40 * GAMMA, solver, 0, False)
        return {"cv": U}
    dims = (case["mx"], case["my"], case["mz"])
    if case["amp"] != 0 or case["visc"] not in (0, 4) or dims[0] * dims[1] * dims[2] > 5e6:
        return None
    b = _box_state(case, seed, 0)[:, :-1, :-1, :-1]  # the periodic box's unique nodes
    U = torch.stack([b[0], b[0] * b[1], b[0] * b[2], b[0] * b[3],
                     0.5 * b[0] * (b[1] ** 2 + b[2] ** 2 + b[3] ** 2) + b[4] / (GAMMA - 1)])
    h = [2 * math.pi * _LEN / (m - 1) for m in dims]
    U = _march(U, h, case["steps"], r, 1e-40 * (_RHO0 * _V0) ** 2, solver, case["visc"], True)
    for q in (1, 2, 3):  # the coincident end nodes
        U = torch.cat([U, U.narrow(q, 0, 1)], q)
    return {"density": U[0], "momentum": U[1:4], "energy": U[4], "temperature": _pressure(U) / (U[0] * R_AIR)}


def _mix64(x):
    x = x + np.uint64(0x9E3779B97F4A7C15)
    x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return x ^ (x >> np.uint64(31))


def _exact_train(case, seed):
    X, Y, net = _train_data(case, seed)
    X, Y = (torch.from_numpy(a).double().cuda() for a in (X, Y))
    P = [torch.from_numpy(a).double().cuda().requires_grad_() for layer in net for a in layer]
    m, v, losses = [torch.zeros_like(p) for p in P], [torch.zeros_like(p) for p in P], []
    rows = np.arange(case["batch"], dtype=np.uint64)
    for t in range(case["steps"]):
        with np.errstate(over="ignore"):
            pick = _mix64(np.uint64(11) ^ _mix64(np.uint64(t) * np.uint64(0x100000001B3) + rows)) % np.uint64(case["rows"])
        at = torch.from_numpy(pick.astype(np.int64)).cuda()
        h = X[at]
        for q in range(5):
            h = h @ P[2 * q] + P[2 * q + 1]
            if q < 4:
                h = torch.nn.functional.gelu(h, approximate="tanh")
        loss = ((h - Y[at]) ** 2).mean()
        grads = torch.autograd.grad(loss, P)
        losses.append(float(loss.detach()))
        with torch.no_grad():
            for q, g in enumerate(grads):
                m[q] = 0.9 * m[q] + 0.1 * g
                v[q] = 0.999 * v[q] + 0.001 * g * g
                P[q] -= 1e-3 * (m[q] / (1 - 0.9 ** (t + 1))) / (torch.sqrt(v[q] / (1 - 0.999 ** (t + 1))) + 1e-8)
    return {"loss": np.array(losses), "params": torch.cat([p.detach().reshape(-1) for p in P])}


def exact(case, seed):
    if case["kind"] in ("tube", "box"):
        return _exact_flow(case, seed)
    if case["kind"] == "train":
        return _exact_train(case, seed)
    return None
