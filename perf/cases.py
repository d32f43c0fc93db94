"""Performance cases: the work a user of the engine has it do, over its range.

Five kinds, each through the public entry points of the Python package:

* "run":       Context.step over an output interval, then the state is read;
* "batch":     the same for many independent simulations in one context;
* "adjoint":   Context.adjoint, the gradient of a loss on the final state;
* "calibrate": a torch calibration step over Trajectory / BatchTrajectory
               (forward, loss, backward);
* "readers":   Context.find_overlaps and Context.porosity of an opened image.

The beds are the repository's own workloads at sizes of its benchmark, its
tests and its configurations: direct-shear cells settled, consolidated and
sheared by sphere_amd.scenes and tiled to size (their number of particles is
cell * tiles, odd cells included), released columns, and jittered lattices for
the readers.  They are made from the seed alone.
"""

import math

import numpy
import torch

from sphere_amd import autograd, engine, scenes
from sphere_amd.sim import sim

RHO = 2600.0
K_N = 1.16e7


def listed():
    return [
        # The smallest call: one base cell (about the size of the smoke run),
        # stepped for an output interval.  Launches and latency are all there is.
        {"name": "run_shear_601", "kind": "run", "scene": "shear", "cell": 601, "tiles": 1,
         "model": 2, "bond_frac": 0.0, "graph": 0, "steps": 400},
        # The 4,096-sphere class: a column released in a closed box, where
        # particles change cell all the time (re-sorts, list rebuilds).
        {"name": "run_column_4096", "kind": "run", "scene": "column", "cell": 4096, "tiles": 1,
         "model": 2, "bond_frac": 0.0, "graph": 0, "steps": 400},
        # Hertzian contacts (model 3) on a mid-size bed.
        {"name": "run_hertz_16533", "kind": "run", "scene": "shear", "cell": 501, "tiles": 33,
         "model": 3, "bond_frac": 0.0, "graph": 0, "steps": 200},
        # Contacts without history (model 1) on a mid-size bed.
        {"name": "run_viscous_16096", "kind": "run", "scene": "shear", "cell": 503, "tiles": 32,
         "model": 1, "bond_frac": 0.0, "graph": 0, "steps": 200},
        # The headline configuration: 1e5 particles, direct shear, replayed
        # from a graph as the benchmark does.
        {"name": "run_shear_100000", "kind": "run", "scene": "shear", "cell": 500, "tiles": 200,
         "model": 2, "bond_frac": 0.0, "graph": 100, "steps": 400},
        # The largest: 1e6 particles, sheared, 2% of the touching pairs bonded.
        {"name": "run_bonded_1000000", "kind": "run", "scene": "shear", "cell": 500,
         "tiles": 2000, "model": 2, "bond_frac": 0.02, "graph": 0, "steps": 100},
        # A sweep of consolidation beds of log-uniform size in one context.
        {"name": "batch_64", "kind": "batch", "nsims": 64, "steps": 200},
        # The gradient of a loss on the final velocities of the 1e5 bed.
        {"name": "adjoint_100000", "kind": "adjoint", "cell": 500, "tiles": 200, "steps": 20},
        # The column-collapse calibration step: trajectory, loss, backward.
        {"name": "calibrate_2000", "kind": "calibrate", "nsims": 1, "np": 2000, "steps": 500,
         "every": 50},
        # Many calibrations at once, one batched trajectory and adjoint.
        {"name": "calibrate_16x1003", "kind": "calibrate", "nsims": 16, "np": 1003,
         "steps": 200, "every": 50},
        # The output-side readers on a small and on a headline-size image
        # (`sphere --contacts`, sim.findOverlaps, sim.porosity).
        {"name": "readers_5000", "kind": "readers", "np": 5000, "slices": 10},
        {"name": "readers_100003", "kind": "readers", "np": 100003, "slices": 12},
    ]


def _loguniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run", "run", "run", "batch", "adjoint", "calibrate", "readers"])
    if kind == "run":
        scene = rng.choice(["shear", "shear", "shear", "column"])
        n = _loguniform(rng, 500, 200000 if scene == "shear" else 8000)
        cell = rng.randint(450, 700) if scene == "shear" else n
        tiles = max(1, int(round(n / cell))) if scene == "shear" else 1
        model = rng.choice([2, 2, 2, 3, 1])
        bonds = rng.choice([0.0, 0.0, 0.02, 0.1]) if scene == "shear" else 0.0
        return {"kind": kind, "scene": scene, "cell": cell, "tiles": tiles, "model": model,
                "bond_frac": bonds, "graph": rng.choice([0, 0, 100]),
                "steps": rng.randint(100, 400)}
    if kind == "batch":
        return {"kind": kind, "nsims": _loguniform(rng, 4, 64), "steps": rng.randint(100, 200)}
    if kind == "adjoint":
        cell = rng.randint(450, 700)
        return {"kind": kind, "cell": cell,
                "tiles": max(1, int(round(_loguniform(rng, 1000, 100000) / cell))),
                "steps": rng.randint(10, 30)}
    if kind == "calibrate":
        nsims = rng.choice([1, 1, 4, 16])
        every = rng.choice([10, 25, 50])
        return {"kind": kind, "nsims": nsims, "np": _loguniform(rng, 400, 4000 / nsims ** 0.5),
                "steps": every * rng.randint(4, 10), "every": every}
    return {"kind": kind, "np": _loguniform(rng, 500, 200000), "slices": rng.randint(3, 14)}


# -- inputs -------------------------------------------------------------------

def _open(image):
    return engine.Context(image)


def _cell(n, seed, r_uniform=None, shear=True):
    """A direct-shear cell settled, consolidated and (optionally) sheared, with
    the stages of the benchmark's base cells: 2 to 3 occupied slots a
    particle."""
    return scenes.settled_shear_cell(n, seed, open_stepper=_open, settle_steps=20000,
                                     consolidate_steps=5000, r_uniform=r_uniform, shear=shear)


def _touching(s):
    """Touching pairs of a small bed (no periodic images), ascending."""
    x, r = s.x, numpy.asarray(s.radius)
    i, j = numpy.triu_indices(len(r), 1)
    d = numpy.sqrt(((x[i] - x[j]) ** 2).sum(axis=1))
    t = d < r[i] + r[j]
    return numpy.stack([i[t], j[t]], axis=1)


def _shear_bed(cell, tiles, seed, model=2, bond_frac=0.0):
    base = _cell(cell, seed)
    mx, my = scenes.near_square(tiles)
    s = scenes.tile_xy(base, mx, my)
    s.contactmodel[0] = model
    if bond_frac > 0.0:
        pairs = _touching(base)
        every = numpy.concatenate([pairs + cell * k for k in range(tiles)])
        rng = numpy.random.default_rng(seed)
        nb = max(1, int(bond_frac * len(every)))
        pick = numpy.sort(rng.choice(len(every), size=nb, replace=False))
        s.bonds = every[pick].astype(numpy.uint32)
        s.nb0[0] = nb
        s.lambda_bar[0] = 1.0
        s.bonds_delta_n = numpy.zeros(nb)
        s.bonds_delta_t = numpy.zeros((nb, 3))
        s.bonds_omega_n = numpy.zeros(nb)
        s.bonds_omega_t = numpy.zeros((nb, 3))
        # A bond breaks at the stress of an extension of 5e-4 m.
        s.sigma_b[0] = s.tau_b[0] = K_N * 5.0e-4
    return s


def _column(n, seed, model=2):
    """A released column, settled at k_n = 1e6 N/m."""
    s = scenes.collapse_column(n, seed=seed, footprint=0.3 * (n / 2000.0) ** (1.0 / 3.0),
                               k_n=1.0e6, damping_frac=0.2, settle_steps=40000,
                               open_stepper=_open)
    s.contactmodel[0] = model
    return s


def _lattice(n, seed):
    """Positions and radii of a jittered cubic lattice with lognormal radii
    (median 0.01 m, at most 0.55 of the spacing): about half of the lattice
    neighbours overlap, as in a settled bed.  Plain numpy."""
    rng = numpy.random.default_rng(seed)
    d = 0.02
    r = numpy.minimum(0.01 * numpy.exp(0.2 * rng.standard_normal(n)), 0.55 * d)
    # About 20 layers deep, fewer in a small bed.
    m = max(3, int(math.ceil((n / 20.0) ** 0.5 if n > 2000 else (n / 2.0) ** (1.0 / 3.0))))
    i = numpy.arange(n)
    x = numpy.stack([i % m, (i // m) % m, i // (m * m)], axis=1) * d + 0.5 * d
    x = x + 0.02 * d * rng.uniform(-1.0, 1.0, (n, 3))
    # Particles come in the order of a packing, not of the lattice.
    order = rng.permutation(n)
    fixed = numpy.where(x[:, 2] < d, 1.0, 0.0)  # a fixed bottom layer, as in shear
    nz = int(math.ceil(n / float(m * m)))
    L = [m * d, m * d, max((nz + 1) * d, 0.4)]
    return x[order], r[order], fixed[order], L


def _readers_image(n, seed):
    x, r, fixed, L = _lattice(n, seed)
    s = sim(np=n, sid="readers-%d" % n)
    s.radius = r.copy()
    s.x = x.copy()
    s.fixvel[:] = fixed
    s.defaultParams(mu_s=0.5, mu_d=0.5, rho=RHO, k_n=K_N, k_t=K_N)
    s.normalBoundariesXY()
    s.defineWorldBoundaries(L=L)
    dt = scenes.dt_rule(float(r.min()), RHO, K_N)
    s.time_dt[0] = dt
    s.time_current[0] = 0.0
    s.time_total[0] = 1.0e3 * dt
    s.time_file_dt[0] = 1.0e3 * dt
    return s.tobytes()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "run":
        if case["scene"] == "column":
            s = _column(case["cell"], seed, case["model"])
        else:
            s = _shear_bed(case["cell"], case["tiles"], seed, case["model"], case["bond_frac"])
        ctx = engine.Context(s.tobytes())
        if case["graph"]:
            ctx.set_scalar("graph_steps", case["graph"])
        ctx.step(20)  # a run under way: contacts and candidate lists exist
        return {"case": case, "ctx": ctx}
    if kind == "batch":
        # The sizes belong to the case, the packings and parameters to the seed.
        sizes = scenes.batch_sizes(case["nsims"])
        bases = [_cell(500, seed, r_uniform=(0.005, 0.01), shear=False)]
        sims = scenes.batch_shear_cells(sizes, bases, seed=seed, kn_range=(1.0e6, 1.0e8))
        ctx = engine.Context(images=[s.tobytes() for s in sims])
        ctx.step(20)
        return {"case": case, "ctx": ctx}
    if kind == "adjoint":
        s = _shear_bed(case["cell"], case["tiles"], seed)
        ctx = engine.Context(s.tobytes())
        ctx.step(20)
        rng = numpy.random.default_rng(seed)
        return {"case": case, "ctx": ctx,
                "dL_dv": rng.standard_normal((case["cell"] * case["tiles"], 3))}
    if kind == "calibrate":
        n, k = case["np"], case["nsims"]
        every, nsamples = case["every"], case["steps"] // case["every"]
        rng = numpy.random.default_rng(seed)
        # One settled column, released with each simulation's own velocities.
        base = _column(n, seed).tobytes()
        sims, stars, starts = [], [], []
        for j in range(k):
            s = sim().frombytes(base)
            s.vel[:, :3] = rng.normal(0.0, 0.01, (n, 3))
            r_min = float(s.radius.min())
            kn = math.exp(rng.uniform(math.log(1.0e6), math.log(4.0e6)))
            stars.append([kn, rng.uniform(0.2, 0.4) * scenes.critical_damping(r_min, RHO, kn),
                          rng.uniform(0.3, 0.7)])
            starts.append([float(s.k_n[0]), float(s.gamma_n[0]), float(s.mu_s[0])])
            sims.append(s)
        params = ("k_n", "gamma_n", "mu")
        if k == 1:
            traj = autograd.Trajectory(sims[0], every, nsamples, params=params)
            stars, starts = stars[0], starts[0]
        else:
            traj = autograd.BatchTrajectory(sims, every, nsamples, params=params)
        with torch.no_grad():
            target = traj(torch.tensor(stars, dtype=torch.float64))
        v0 = torch.as_tensor(numpy.concatenate([s.vel[:, :3] for s in sims]))
        return {"case": case, "traj": traj, "target": target, "theta": starts, "v0": v0}
    if kind == "readers":
        n = case["np"]
        # The program keeps its lists in arrays of a fixed size (at most 1.1
        # overlaps a particle here).
        return {"case": case, "ctx": engine.Context(_readers_image(n, seed)),
                "pairs": numpy.zeros((2 * n, 2), dtype=numpy.uint32),
                "delta": numpy.zeros(2 * n)}
    raise ValueError("unknown kind %r" % kind)


# -- one pass -----------------------------------------------------------------

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "run":
        ctx = state["ctx"]
        ctx.step(case["steps"])
        return {"x": ctx.get("x"), "vel": ctx.get("vel"), "angvel": ctx.get("angvel"),
                "walls_nx": ctx.get("walls_nx"), "walls_mvfd": ctx.get("walls_mvfd")}
    if kind == "batch":
        ctx = state["ctx"]
        ctx.step(case["steps"])
        return {f: numpy.concatenate([ctx.get(f, sim=k) for k in range(ctx.nsims)])
                for f in ("x", "vel", "walls_nx", "walls_mvfd")}
    if kind == "adjoint":
        return state["ctx"].adjoint(case["steps"], None, state["dL_dv"], None)
    if kind == "calibrate":
        theta = torch.tensor(state["theta"], dtype=torch.float64, requires_grad=True)
        v0 = state["v0"].clone().requires_grad_(True)
        samples = state["traj"](theta, v0=v0)
        loss = ((samples - state["target"]) ** 2).mean()
        loss.backward()
        return {"samples": samples.detach(), "loss": float(loss.detach()),
                "theta_grad": theta.grad, "v0_grad": v0.grad}
    ctx = state["ctx"]
    pairs, delta = ctx.find_overlaps()
    k = len(delta)
    state["pairs"][:k] = pairs
    state["delta"][:k] = delta
    z, por = ctx.porosity(case["slices"])
    return {"count": k, "pairs": state["pairs"], "delta": state["delta"], "z": z,
            "porosity": por}


# -- what a pass cannot do without --------------------------------------------

# Occupied contact slots per particle of these beds, rounded.
Z = 2.5
# Bytes per particle and step: the state read and written once, and each
# occupied slot's index and displacement read and written.
STEP_BYTES = 528.0 + 72.0 * Z
# Operations per particle and step: the contact law per slot, the integration.
STEP_FLOPS = 260.0 * Z + 160.0


def work(case):
    kind = case["kind"]
    if kind == "run":
        n = case["cell"] * case["tiles"] * case["steps"]
        return {"bytes": STEP_BYTES * n, "flops": STEP_FLOPS * n}
    if kind == "batch":
        # The mean of a log-uniform size in [500, 20000].
        n = case["nsims"] * (20000 - 500) / math.log(20000 / 500.0) * case["steps"]
        return {"bytes": STEP_BYTES * n, "flops": STEP_FLOPS * n}
    if kind == "adjoint":
        # Forward; the record written and read (100 B of state, 36 B a slot);
        # cotangents of 5 vectors and of the displacements read and written.
        n = case["cell"] * case["tiles"] * case["steps"]
        return {"bytes": (STEP_BYTES + 2.0 * (100.0 + 36.0 * Z) + 2.0 * (120.0 + 24.0 * Z)) * n,
                "flops": 3.0 * STEP_FLOPS * n}
    if kind == "calibrate":
        n = case["nsims"] * case["np"] * case["steps"]
        return {"bytes": (STEP_BYTES + 2.0 * (100.0 + 36.0 * Z) + 2.0 * (120.0 + 24.0 * Z)) * n,
                "flops": 3.0 * STEP_FLOPS * n}
    # Readers: positions, radii and fixed flags read, about 1.2 pairs a
    # particle written; the 27-cell neighbourhood tested, half of it.
    n = case["np"]
    return {"bytes": n * (40.0 + 1.2 * 16.0), "flops": n * (13.0 * 12.0 + 20.0)}


# -- the same in 64 bits ------------------------------------------------------

def _cap(h, r):
    return math.pi * h * h / 3.0 * (3.0 * r - h)


def exact(case, seed):
    """The readers in plain torch and numpy.  The other kinds have no value in
    64 bits: the step rounds every length to FP32 by definition, and a
    trajectory follows those roundings."""
    if case["kind"] != "readers":
        return None
    x, r, fixed, L = _lattice(case["np"], seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    xt, rt = torch.as_tensor(x, device=dev), torch.as_tensor(r, device=dev)
    free = torch.as_tensor(fixed == 0.0, device=dev)
    n = len(r)
    idx = torch.arange(n, device=dev)
    deltas = []
    rows = max(1, 40_000_000 // n)
    for a in range(0, n, rows):
        b = min(n, a + rows)
        d2 = torch.zeros((b - a, n), dtype=torch.float64, device=dev)
        for k in range(3):
            d2 += (xt[None, :, k] - xt[a:b, None, k]) ** 2
        dn = d2.sqrt_() - (rt[a:b, None] + rt[None, :])
        hit = (dn < 0.0) & (idx[None, :] > idx[a:b, None]) & free[a:b, None] & free[None, :]
        i, j = hit.nonzero(as_tuple=True)
        deltas.append(dn[i, j].cpu())
    m = case["slices"]
    h = L[2] / m
    V = h * L[0] * L[1]
    zc, zl, zh = x[:, 2], x[:, 2] - r, x[:, 2] + r
    vs = 4.0 / 3.0 * math.pi * r ** 3
    z, por = numpy.zeros(m), numpy.zeros(m)
    for s in range(m):
        lo, hi = s * h, s * h + h
        inside = (lo <= zl) & (zh <= hi)
        v = vs[inside].sum()
        out = ~inside
        c = out & (lo >= zc) & (lo <= zh)
        v += _cap(zh[c] - lo, r[c]).sum()
        c = out & (lo < zc) & (lo > zl)
        v += (vs[c] + _cap(lo - zl[c], r[c])).sum()
        c = out & (hi <= zc) & (hi >= zl)
        v += _cap(hi - zl[c], r[c]).sum()
        c = out & (hi > zc) & (hi < zh)
        v += (vs[c] + _cap(zh[c] - hi, r[c])).sum()
        z[s] = lo + 0.5 * h
        por[s] = (V - v) / V
    delta = torch.cat(deltas)
    delta = torch.cat([delta, torch.zeros(2 * n - len(delta), dtype=torch.float64)])
    return {"count": None, "pairs": None, "delta": delta, "z": z, "porosity": por}
