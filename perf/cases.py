"""Workloads by which the step engine's speed is measured.

Most cases are whole simulations: a state is set up, started and advanced a
few steps (`prepare`), and a pass (`run`) advances it by `steps` more steps
and takes the fields of a frame (positions, velocities, densities, pressures,
accelerations where they are asked for) to the host, as a program does that
writes frames.  The further passes are one call each of the surrogate's
training and the engine's per-pass entry points on a given state.

Sizes are those of bench.py's workloads and of the tests, smaller and odd ones
between; `draw` takes others from the same ranges.
"""
import math

import numpy as np
import torch

from fjsph_amd import abi, cases, surrogate
from fjsph_amd.engine import Engine

WARM = 5  # steps before a state is measured: the first ones iterate several times as often


def listed():
    return [
        # 2D dam break between Adami walls at the bench's spacing, FP64: the
        # smallest run anyone starts, launches and latency count
        dict(name="dam2d_6k_fp64", kind="dam2d", dx=0.02, precision="fp64", steps=10),
        # the same column at a fine spacing with FP32 pair terms
        dict(name="dam2d_92k_mixed", kind="dam2d", dx=0.005, precision="mixed", steps=10),
        # a 1 mm droplet in FP64, the size the smoke check runs
        dict(name="droplet_4k_fp64", kind="droplet", diameter=1.0e-3, precision="fp64", steps=10),
        # the 4 mm droplet in a crossflow, the single-droplet configuration
        dict(name="droplet_268k_mixed", kind="droplet", diameter=4.0e-3, precision="mixed", steps=10),
        # a short jet with ALE shifting in FP64 (the like-for-like precision of the bench)
        dict(name="jet_200k_fp64", kind="jet", n=200_000, precision="fp64", gas="const", integrator="nb", steps=4),
        # a jet under Runge-Kutta 4
        dict(name="jet_100k_rk4", kind="jet", n=100_000, precision="mixed", gas="const", integrator="rk4", steps=6),
        # a medium jet with the gas velocity looked up in a tetrahedral mesh
        dict(name="jet_700k_mesh", kind="jet", n=700_000, precision="mixed", gas="mesh", integrator="nb", steps=8),
        # the headline workload: 4M particles, gas velocity from the MLP surrogate
        dict(name="jet_4m_surrogate", kind="jet", n=4_000_000, precision="mixed", gas="surrogate", integrator="nb",
             steps=10),
        # 256 independent droplets, one launch per pass over all of them
        dict(name="batch_256_drops", kind="batch", n_drops=256, precision="mixed", steps=8),
        # jet in crossflow: ghost-walled pipe, inlet columns, a growing particle set
        dict(name="jicf_1m", kind="jicf", n=1_000_000, precision="mixed", steps=6),
        # one state through the per-pass entry points: neighbour lists,
        # dSPH_PreStep, the force pass (a driver with its own time loop)
        dict(name="passes_113k", kind="passes", diameter=3.0e-3, precision="mixed"),
        # training of the gas surrogate on labelled samples
        dict(name="train_300", kind="train", samples=200_000, batch=16384, steps=300),
    ]


def draw(rng):
    """A case of the listed ones' ranges."""
    def logu(a, b):
        return math.exp(rng.uniform(math.log(a), math.log(b)))

    kind = rng.choice(["dam2d", "droplet", "droplet", "jet", "jet", "jet", "batch", "jicf", "passes", "train"])
    prec = rng.choice(["fp64", "mixed", "mixed"])
    if kind == "dam2d":
        return dict(kind=kind, dx=round(logu(0.005, 0.04), 5), precision=prec, steps=rng.randint(5, 12))
    if kind == "droplet":
        top = 4.0e-3 if prec == "mixed" else 2.0e-3
        return dict(kind=kind, diameter=round(logu(0.8e-3, top), 6), precision=prec, steps=rng.randint(4, 12))
    if kind == "jet":
        top = 4_000_000 if prec == "mixed" else 400_000
        gas = rng.choice(["const", "mesh", "surrogate"])
        integrator = rng.choice(["nb", "nb", "nb", "rk4"]) if gas == "const" else "nb"
        return dict(kind=kind, n=int(logu(50_000, top)), precision=prec, gas=gas, integrator=integrator,
                    steps=rng.randint(3, 8))
    if kind == "batch":
        return dict(kind=kind, n_drops=int(logu(5, 256)), precision="mixed", steps=rng.randint(4, 8))
    if kind == "jicf":
        return dict(kind=kind, n=int(logu(60_000, 1_000_000)), precision="mixed", steps=rng.randint(3, 6))
    if kind == "passes":
        return dict(kind=kind, diameter=round(logu(1.0e-3, 3.0e-3), 6), precision=prec)
    return dict(kind=kind, samples=int(logu(20_000, 400_000)), batch=64 * rng.randint(16, 400),
                steps=rng.randint(50, 300))


def _prec(case):
    return abi.PREC_MIXED if case["precision"] == "mixed" else abi.PREC_FP64


def _gas_mesh(c):
    """Potential flow past a cylinder on a tetrahedral mesh around the jet."""
    cases.with_mesh(c, kind="kuhn", n_cells=200_000)
    return c.mesh


def _surrogate(c, seed):
    """The MLP trained on the mesh field, as a program does once per mesh."""
    mesh = _gas_mesh(c)
    with Engine(c.settings) as lab:
        lab.set_mesh(mesh)
        sg = surrogate.train(mesh, lab, n_samples=100_000, steps=300, seed=seed)
    c.mesh = None
    c.settings.aero_source = abi.SURROGATE
    return sg


def _swirl(c, seed):
    """A droplet's velocities and densities part way through a run: a smooth
    swirl of a few m/s and density variations of about 1e-3."""
    rng = np.random.default_rng(seed)
    k = 2.0 * math.pi / 4.0e-3 * rng.uniform(0.7, 1.3, size=(3, 3))
    ph = rng.uniform(0.0, 2.0 * math.pi, size=4)
    c.v = np.ascontiguousarray(3.0 * np.sin(c.x @ k.T + ph[:3]))
    s = c.settings
    c.rho = s.rho_rest * (1.0 + 1e-3 * np.sin(c.x @ k[0] + ph[3]))
    b = s.rho_rest * s.speed_sound ** 2 / s.gam
    c.p = b * ((c.rho / s.rho_rest) ** s.gam - 1.0)


def _jitter(c, seed, which=slice(None)):
    """The lattice shaken by the seed (the builders' own jitter, which decides
    the lattice points inside a sphere, stays as it is)."""
    r = 0.005 * c.settings.particle_step
    c.x[which] += np.random.default_rng(seed).uniform(-r, r, c.x[which].shape)
    return c


def _passes_case(case, seed):
    c = _jitter(cases.droplet_3d(diameter=case["diameter"], precision=_prec(case)), seed)
    c.settings.aero_case = abi.NO_AERO
    _swirl(c, seed)
    return c


def prepare(case, seed):
    kind = case["kind"]
    if kind == "train":
        c = cases.jet_column_3d(n_target=20_000, seed=seed)
        mesh = _gas_mesh(c)
        eng = Engine(c.settings)
        eng.set_mesh(mesh)
        x, y = surrogate.sample_mesh(mesh, case["samples"], seed=seed, engine=eng)
        lo, hi = mesh.verts.min(axis=0), mesh.verts.max(axis=0)
        scale = y.std(axis=0)
        w, b = surrogate.init_params(3, 4, seed=seed)
        return dict(case=case, engine=eng, args=(x, y, 4, w, b, 0.5 * (lo + hi), 0.5 * (hi - lo), y.mean(axis=0),
                                                 np.where(scale > 0, scale, 1.0)), seed=seed)
    if kind == "passes":
        return dict(case=case, engine=Engine(_passes_case(case, seed)))
    sg = None
    if kind == "dam2d":
        c = cases.dam_break_2d(dx=case["dx"], precision=_prec(case))
        _jitter(c, seed, slice(c.n_bound, None))
    elif kind == "droplet":
        c = _jitter(cases.droplet_3d(diameter=case["diameter"], precision=_prec(case)), seed)
    elif kind == "jet":
        c = cases.jet_column_3d(n_target=case["n"], seed=seed, precision=_prec(case))
        if case["integrator"] == "rk4":
            c.settings.integrator = abi.RUNGE_KUTTA
        if case["gas"] == "mesh":
            _gas_mesh(c)
        elif case["gas"] == "surrogate":
            sg = _surrogate(c, seed)
    elif kind == "batch":
        c = _jitter(cases.batched_droplets(n_drops=case["n_drops"], precision=_prec(case)), seed)
    elif kind == "jicf":
        c = cases.jet_in_crossflow_3d(n_target=case["n"], precision=_prec(case))
        _jitter(c, seed, np.flatnonzero(c.b == abi.FREE))
    else:
        raise ValueError(f"unknown kind {kind}")
    eng = Engine(c)
    if kind == "batch":
        eng.set_groups(c.owner)
    if sg is not None:
        eng.set_surrogate(sg)
    eng.integrate_no_update()
    for _ in range(WARM):
        eng.integrate_step()
    return dict(case=case, engine=eng)


def run(state):
    case, eng = state["case"], state["engine"]
    if case["kind"] == "train":
        w, b, loss = eng.surrogate_train(*state["args"], steps=case["steps"], batch=case["batch"], lr=3e-3,
                                         seed=state["seed"])
        return {"weights": w, "biases": b, "loss": loss}
    if case["kind"] == "passes":
        eng.build_neighbours()
        npd = eng.dsph_prestep()
        eng.acc_rrho(npd)
        return {"counts": eng.neighbour_counts(), "npd": npd, "lam": eng.field("LAM"),
                "gradrho": eng.field("GRADRHO"), "norm": eng.field("NORM"), "colour": eng.field("COLOUR"),
                "acc": eng.field("ACC"), "rrho": eng.field("RRHO")}
    for _ in range(case["steps"]):
        eng.integrate_step()
    return {"x": eng.field("X"), "v": eng.field("V"), "rho": eng.field("RHO"), "p": eng.field("P")}


# particles of a case, and list entries (pairs) per particle of its interior
def _size(case):
    kind = case["kind"]
    if kind == "dam2d":
        dx = case["dx"]
        return round(1.0 / dx) * round(2.0 / dx) + 3 * (round(4.0 / dx) + 6) + 6 * round(3.0 / dx), 21, 2
    if kind in ("droplet", "passes"):
        return int(math.pi / 6.0 * (case["diameter"] / 5e-5) ** 3), 230, 3
    if kind == "batch":
        # drops of log-uniform diameter in [0.5, 2] mm
        mean = (2e-3 ** 3 - 0.5e-3 ** 3) / (3.0 * math.log(4.0))
        return int(case["n_drops"] * math.pi / 6.0 * mean / 5e-5 ** 3), 180, 3
    return case["n"], 230, 3


# force passes (Newmark-Beta sub-iterations) per step the states above need
# at the least: the update needs two to see that it has converged
_SUBITS = 2


def work(case):
    """What a pass cannot do without.  A step: two list builds and two sets
    of pre-passes, each reading the state of a particle (position, velocity,
    density, mass: 64 B in 3D) and writing its results (correction matrix,
    gradients, normals, flags, shifting velocity: about 240 B), and the
    sub-iterations' force passes and updates (176 B + 184 B a particle);
    about 50 operations a pair in each of the three pre-passes, 10 in the
    list build's distance test, and 82 in the force pass.  The frame's fields
    go to the host as 64 B a particle."""
    if case["kind"] == "train":
        # forward and backward products of the 3 - 64 x 4 - 5 network, and each batch's samples
        macs = 64 * 3 + 3 * 64 * 64 + 64 * 5
        return {"bytes": case["steps"] * case["batch"] * 48.0 + case["samples"] * 64.0,
                "flops": 6.0 * macs * case["steps"] * case["batch"]}
    n, pairs, dim = _size(case)
    if case["kind"] == "passes":
        return {"bytes": n * (64.0 + 240.0 + 176.0 + 96.0), "flops": n * pairs * (10.0 + 50.0 + 82.0)}
    rk = case.get("integrator") == "rk4"
    nforce = 4 if rk else _SUBITS
    per_step = n * (2 * (64.0 + 240.0) + nforce * 360.0) * (dim / 3.0)
    flops = n * pairs * (2 * (10.0 + 3 * 50.0) + nforce * 82.0) * (dim / 3.0)
    return {"bytes": case["steps"] * per_step + n * 64.0 * (dim / 3.0), "flops": case["steps"] * flops}


def tolerance(case):
    """About four times what the outputs move by when the pair sums run in
    another order (tile blocks of other lengths): pressures, the most
    sensitive of a run's fields, by 5.6e-7 (6e-5 at the worst particle) with
    FP32 pair terms and 2.6e-11 (2.6e-10) in FP64; of the passes the
    acceleration, 4.5e-7 (3.5e-6).  The training works in BF16."""
    mixed = case.get("precision") == "mixed"
    if case["kind"] == "train":
        return {"rel": 1e-2}
    if case["kind"] == "passes":
        return {"rel": 2e-6, "max": 1.5e-5, "differ": 0.0} if mixed else {"rel": 1e-13, "max": 1e-11, "differ": 0.0}
    return {"rel": 2e-6, "max": 2.5e-4} if mixed else {"rel": 2e-10, "max": 2e-9}


def exact(case, seed):
    """The per-pass case in 64 bits from the equations.  The whole runs have
    none: their adaptive steps are the reference's full algorithm, the
    training a chaotic sequence of updates."""
    if case["kind"] != "passes":
        return None
    c = _passes_case(case, seed)
    s = c.settings
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=dev)
    x, v, rho, p, m = t(c.x), t(c.v), t(c.rho), t(c.p), t(c.m)
    n = c.n
    H = s.H_fac * s.particle_step
    sr = 4.0 * H * H
    Wc = 21.0 / (16.0 * math.pi * H ** 3)
    vol, pr = m / rho, p / (rho * rho)
    # cells of edge 2H, the particles of each in a padded table
    cell = torch.floor((x - x.min(dim=0).values) / (2.0 * H * (1.0 + 1e-9))).long() + 1
    dims = cell.max(dim=0).values + 2
    lin = (cell[:, 2] * dims[1] + cell[:, 1]) * dims[0] + cell[:, 0]
    order = torch.argsort(lin)
    count = torch.bincount(lin, minlength=int(dims.prod()))
    start = torch.cumsum(count, 0) - count
    width = int(count.max())
    table = torch.full((count.numel(), width), -1, dtype=torch.long, device=dev)
    table[lin[order], torch.arange(n, device=dev) - start[lin[order]]] = order
    shift = torch.tensor([(dz * int(dims[1]) + dy) * int(dims[0]) + dx for dz in (-1, 0, 1) for dy in (-1, 0, 1)
                          for dx in (-1, 0, 1)], device=dev)
    counts = torch.zeros(n, dtype=torch.long, device=dev)
    L = torch.zeros((n, 3, 3), dtype=torch.float64, device=dev)
    gr, nr, acc = (torch.zeros((n, 3), dtype=torch.float64, device=dev) for _ in range(3))
    col, rr = (torch.zeros(n, dtype=torch.float64, device=dev) for _ in range(2))
    wsum = torch.zeros((), dtype=torch.float64, device=dev)

    def pairs(i0, i1):
        j = table[lin[i0:i1, None] + shift[None, :]].reshape(i1 - i0, -1)
        i = torch.arange(i0, i1, device=dev)[:, None].expand_as(j)
        keep = (j >= 0) & (j != i)
        i, j = i[keep], j[keep]
        d = x[j] - x[i]
        d2 = d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2]
        near = d2 < sr
        return i[near], j[near], d[near], d2[near]

    chunk = 8192
    for i0 in range(0, n, chunk):
        i, j, d, d2 = pairs(i0, min(n, i0 + chunk))
        q = torch.sqrt(d2) / H
        u = 1.0 - 0.5 * q
        W = Wc * u ** 4 * (2.0 * q + 1.0)
        g = (5.0 * Wc / H ** 2) * (u ** 3)[:, None] * d
        counts.index_add_(0, i, torch.ones_like(i))
        L.index_add_(0, i, vol[j][:, None, None] * d[:, :, None] * g[:, None, :])
        gr.index_add_(0, i, -(vol[j] * (rho[j] - rho[i]))[:, None] * g)
        nr.index_add_(0, i, -vol[j][:, None] * g)
        col.index_add_(0, i, vol[j] * W)
        wsum += W.sum()
    npd = float(wsum) / n
    h2 = 2.0 * H
    lam_st = 6.0 / 81.0 * h2 ** 3 / math.pi ** 4 * (9.0 / 4.0 * math.pi ** 3 - 6.0 * math.pi - 4.0)
    ste = -(0.5 * s.sig / lam_st) / npd ** 2
    nu = s.mu / s.rho_rest
    for i0 in range(0, n, chunk):
        i, j, d, d2 = pairs(i0, min(n, i0 + chunk))
        r = torch.sqrt(d2)
        g = (5.0 * Wc / H ** 2) * ((1.0 - 0.5 * r / H) ** 3)[:, None] * d
        dv = v[j] - v[i]
        visc = m[j] * nu * (1.0 / rho[i] + 1.0 / rho[j]) * (d * g).sum(1) / (d2 + 0.001 * H * H)
        st = ste * torch.cos(3.0 * math.pi / (4.0 * H) * r) / r / m[i]
        acc.index_add_(0, i, visc[:, None] * dv + st[:, None] * d - (m[j] * (pr[i] + pr[j]))[:, None] * g)
        rr.index_add_(0, i, -rho[i] * vol[j] * (dv * g).sum(1))
    acc += t(np.array(list(s.grav)))
    Linv = torch.linalg.inv(L)
    host = lambda a: a.cpu().numpy()
    return {"counts": (host(counts) + 1).astype(np.int32), "npd": npd,  # a particle is its own neighbour
            "lam": host(torch.linalg.eigvalsh(L)[:, 0].contiguous()),
            "gradrho": host((Linv @ gr[:, :, None])[:, :, 0]), "norm": host((Linv @ nr[:, :, None])[:, :, 0]),
            "colour": host(col), "acc": host(acc), "rrho": host(rr)}
