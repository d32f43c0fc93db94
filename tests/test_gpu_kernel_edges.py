"""The readers' and contact kernels at the sizes where their tiling can go
wrong (tile edges, remainders, dispatch lines), bit for bit against the
oracle."""

import numpy
import pytest

import oracle
from sphere_amd import engine, scenes
from sphere_amd.sim import sim

from . import cases

pytestmark = pytest.mark.gpu


def _cloud(n, seed, r=(0.008, 0.012), last=None, L=(0.5, 0.5, 0.5)):
    """n spheres at random places of a box (they may overlap)."""
    rng = numpy.random.default_rng(seed)
    s = sim(np=n, sid="cloud-%d" % n)
    s.radius = rng.uniform(r[0], r[1], n)
    if last is not None:
        s.radius[-1] = last
    s.x = rng.uniform(0.02, 0.48, (n, 3))
    s.defaultParams(rho=2600.0, k_n=1.0e6, k_t=1.0e6)
    s.normalBoundariesXY()
    s.defineWorldBoundaries(L=list(L))
    dt = scenes.dt_rule(float(s.radius.min()), 2600.0, 1.0e6)
    s.time_dt[0] = dt
    s.time_current[0] = 0.0
    s.time_total[0] = dt * 1000
    s.time_file_dt[0] = dt * 1000
    return s


# A round of the slice kernel takes 960 particles; a thin slice takes two
# terms from most of them; beyond 8,192 slices (1,024 in a small simulation)
# each work-item takes a slice.
@pytest.mark.parametrize("n,slices,last", [
    (1, 1, None), (64, 3, None), (959, 7, None), (960, 7, None), (961, 20, None),
    (2881, 1, None), (1920, 60, 1.0e-4), (700, 8192, 1.0e-5), (700, 8193, 1.0e-5),
    (20, 1024, 1.0e-5), (20, 1025, 1.0e-5)])
def test_porosity_tile_edges(n, slices, last):
    image = _cloud(n, 7 + n, last=last).tobytes()
    with engine.Context(image) as ctx:
        za, pa = ctx.porosity(slices)
    zb, pb = oracle.Oracle(image).porosity(slices)
    assert numpy.array_equal(za, zb) and numpy.array_equal(pa, pb)


# The reverse pass's sums run over 64-particle workgroups in 256 shares:
# 256 workgroups exactly, one more (np rounds up to 256), and a bonded bed.
@pytest.mark.parametrize("n,bond_frac", [(16384, 0.0), (16385, 0.0), (17000, 0.05)])
def test_adjoint_sums_over_many_workgroups(n, bond_frac):
    s = cases.lattice_bed(n, 5, 0.01, 0.1, bond_frac=bond_frac)
    image, steps = s.tobytes(), 3
    rng = numpy.random.default_rng(n)
    c = rng.standard_normal((n, 3))
    with engine.Context(image) as ctx:
        g = ctx.adjoint(steps, None, c, None)
    for name in ("k_n", "gamma_n", "gamma_wn"):
        t = oracle.TangentOracle(image)
        t.seed_param(name, 1.0)
        t.step(steps)
        want = float(numpy.sum(c * t.tangent("vel")))
        # Forward and reverse mode agree to rounding of sums over n terms of
        # either sign: 1e-6 of the result, as the other tangent checks.
        assert abs(g[name] - want) <= 1e-6 * abs(want), (name, g[name], want)


def _model1(case):
    if case == "crowded":  # 44 overlaps: more than a list or the hit buffer holds
        s = cases.crowded_case()
    elif case == "fcc":
        s = cases.fcc_case()
    elif case == "one":
        s = _cloud(1, 3)
        s.vel[:, 2] = -1.0
    else:
        s = scenes.lattice_box(int(case), seed=4)
    s.contactmodel[0] = 1
    return s


# Lists, list overflow, a list rebuilt every step (no lists), particles that
# change cell, one particle, a last wavefront with few groups.
@pytest.mark.parametrize("case,steps,skin", [
    ("crowded", 20, None), ("crowded", 5, 0.0), ("fcc", 100, None), ("one", 10, None),
    ("66", 400, None), ("1025", 300, None), ("1025", 50, 0.0)])
def test_model1_matches_oracle(case, steps, skin):
    image = _model1(case).tobytes()
    ref = oracle.Oracle(image)
    ref.step(steps)
    with engine.Context(image) as ctx:
        if skin is not None:
            ctx.set_scalar("vl_skin", skin)
        ctx.step(steps)
        for f in ("perm", "x", "vel", "angvel", "force", "torque", "p", "es", "ev"):
            assert numpy.array_equal(ctx.get(f), ref.get(f)), f


# The end-of-step re-sort: one mover, a few, more than get a wavefront for
# their search (64), more than have their runs listed (256), more than it
# merges (2,048), whole and partial last chunks; the finished step's order and
# cells are told from the movers' records.
@pytest.mark.parametrize("n,movers", [
    (1, 1), (256, 1), (257, 3), (3000, 2), (3000, 64), (3000, 65), (3000, 256), (3000, 257),
    (3000, 1900), (3000, 2600)])
def test_resort_of_many_movers(n, movers):
    rng = numpy.random.default_rng(n + movers)
    s = _cloud(n, 11, r=(0.002, 0.003))
    s.x = rng.uniform(0.1, 0.4, (n, 3))
    cell = float(s.L[0]) / int(s.num[0])
    pick = rng.choice(n, size=movers, replace=False)
    step = rng.uniform(-1.3, 1.3, (movers, 3)) * cell
    s.vel[pick, :3] = step / float(s.time_dt[0])
    image = s.tobytes()
    ref = oracle.Oracle(image)
    with engine.Context(image) as ctx:
        ctx.set_scalar("sort_mode", 1)
        for k in range(5):
            ctx.step(1)
            ref.step(1)
            cs, ce = ctx.get("cellstart"), ctx.get("cellend")
            rs, re_ = ref.get("cellstart"), ref.get("cellend")
            occ = rs != 0xffffffff
            assert numpy.array_equal(cs, rs) and numpy.array_equal(ce[occ], re_[occ]), k
            for f in ("perm", "cellid", "contacts", "x", "vel", "force", "delta_t"):
                assert numpy.array_equal(ctx.get(f), ref.get(f)), (k, f)
        assert ctx.scalar("sorts") >= 1


# The reverse pass's wavefronts of 16 particles: several rounds of evaluations
# (about 190 contacts a wavefront), a last wavefront with few particles,
# walls on every side, recorded whole and in segments.
@pytest.mark.parametrize("kind,checkpoint", [("fcc", 0), ("fcc", 2), (17, 0), (65, 0)])
def test_adjoint_wavefront_edges(kind, checkpoint):
    s = cases.fcc_case() if kind == "fcc" else cases.lattice_bed(kind, 3, 0.01, 0.1)
    n, image, steps = int(s.np[0]), s.tobytes(), 5
    rng = numpy.random.default_rng(n)
    cx, cv, dv = (rng.standard_normal((n, 3)) for _ in range(3))
    with engine.Context(image) as ctx:
        ctx.set_scalar("adj_checkpoint", checkpoint)
        g = ctx.adjoint(steps, cx, cv, None)
    got = {"k_n": g["k_n"], "gamma_t": g["gamma_t"], "v0": float(numpy.sum(g["v"] * dv))}
    for name, ad in got.items():
        t = oracle.TangentOracle(image)
        if name == "v0":
            t.seed_field("vel", dv)
        else:
            t.seed_param(name, 1.0)
        t.step(steps)
        want = float(numpy.sum(cx * t.tangent("x")) + numpy.sum(cv * t.tangent("vel")))
        # Forward against reverse mode: 1e-6, as the other tangent checks.
        assert abs(ad - want) <= 1e-6 * abs(want), (name, ad, want)


# Overlap lists: no pair possible, search workgroups of 64 exactly and not,
# particles with more overlaps than are kept (8), lists longer than two a
# particle (written a second time), fixed particles, a buffer too short.
@pytest.mark.parametrize("n,radius", [
    (1, 0.01), (2, 0.07), (63, 0.03), (64, 0.05), (65, 0.07), (700, 0.03), (2049, 0.02),
    (5000, 0.004)])
def test_overlap_list_edges(n, radius):
    import ctypes
    s = _cloud(n, 5, r=(0.5 * radius, radius))
    s.fixvel[::7] = 1.0
    image = s.tobytes()
    pb, db = oracle.Oracle(image).find_overlaps()
    with engine.Context(image) as ctx:
        for _ in range(2):
            pa, da = ctx.find_overlaps()
            assert numpy.array_equal(pa, pb) and numpy.array_equal(da, db)
        L, m = engine.load(), ctypes.c_uint64()
        k = len(pb) // 2
        pairs, delta = numpy.zeros((k, 2), dtype=numpy.uint32), numpy.zeros(k)
        assert L.sph_find_overlaps(ctx._h, 0, pairs.ctypes.data, delta.ctypes.data, k,
                                   ctypes.byref(m)) == 0
        assert m.value == len(pb)
        assert numpy.array_equal(pairs, pb[:k]) and numpy.array_equal(delta, db[:k])


# The two-kernel step of small totals (up to 18,432 particles with their
# padding) and the three-kernel step just above, re-sorting at nearly every
# step: a round of the wall-force sum takes 8,192 particles, and settings are
# changed in between, so that steps of either form, with other list layouts
# and with stale sorted copies, follow each other.
@pytest.mark.parametrize("n", [300, 4097, 8192, 8193, 18432, 18433])
def test_small_total_step_form(n):
    rng = numpy.random.default_rng(n)
    s = _cloud(n, 13, r=(0.002, 0.003))
    s.x = rng.uniform(0.05, 0.45, (n, 3))
    cell = float(s.L[0]) / int(s.num[0])
    pick = rng.choice(n, size=max(3, n // 100), replace=False)
    s.vel[pick, :3] = rng.uniform(-0.3, 0.3, (len(pick), 3)) * cell / float(s.time_dt[0])
    s.x[rng.choice(n, size=n // 3, replace=False), 2] = 0.45
    s.consolidate(1.0e3)
    s.w_x[0] = 0.4515  # pressed into the third of them at the top
    image = s.tobytes()
    ref, pressed = oracle.Oracle(image), 0
    with engine.Context(image) as ctx:
        ctx.set_scalar("sort_mode", 1)
        for name, value in ((None, 0), ("contact_lanes", 16), ("contact_lanes", 4), ("fused", 1),
                            ("fused", 0), ("sort_mode", 0), ("sort_mode", 1),
                            ("graph_steps", 2)):
            if name:
                ctx.set_scalar(name, value)
            ctx.step(4)
            ref.step(4)
            for f in ("perm", "contacts", "x", "vel", "angvel", "force", "delta_t", "walls_mvfd"):
                assert numpy.array_equal(ctx.get(f), ref.get(f)), (name, value, f)
            pressed += ref.get("walls_mvfd")[0, 2] != 0.0
        if n > 300:  # (three movers seldom leave their cells)
            assert ctx.scalar("sorts") >= 8 and pressed


# A closed context's tape serves the next context that fits into it: smaller
# (but not by much), larger, much smaller, after everything was given back,
# recorded whole and in segments, with two contexts open at once.
@pytest.mark.parametrize("checkpoint", [0, 3])
def test_adjoint_tapes_of_successive_contexts(checkpoint):
    beds = {n: cases.lattice_bed(n, 4, 0.01, 0.1).tobytes() for n in (60, 700, 900)}
    seeds = {n: numpy.random.default_rng(n).standard_normal((n, 3)) for n in beds}

    def gradient(ctx, n):
        ctx.set_scalar("adj_checkpoint", checkpoint)
        g = ctx.adjoint(7, seeds[n], None, None)
        return numpy.concatenate([g["x"].ravel(), g["v"].ravel(), [g["k_n"], g["mu_s"]]])

    want = {}
    for n, image in beds.items():
        engine.trim()
        with engine.Context(image) as ctx:
            want[n] = gradient(ctx, n)
    for n in (700, 900, 700, 60, 900):
        with engine.Context(beds[n]) as ctx, engine.Context(beds[700]) as other:
            # The same operations in the same order, whatever the memory held.
            assert numpy.array_equal(gradient(ctx, n), want[n]), n
            assert numpy.array_equal(gradient(other, 700), want[700]), n
    engine.trim()


# Particle nb0's scan of the bond list once bonds have broken: 256 bonds
# exactly, one more, more than one round of 2,048, bonds it holds itself.
@pytest.mark.parametrize("n,bonds", [(900, 256), (900, 257), (6000, 2049), (60, 7)])
def test_many_broken_bonds(n, bonds):
    s = cases.lattice_bed(n, 6, 0.01, 0.1, bond_frac=1.0)
    assert len(s.bonds) >= bonds and bonds < n
    rng = numpy.random.default_rng(n + bonds)
    s.bonds = s.bonds[numpy.sort(rng.choice(len(s.bonds), size=bonds, replace=False))]
    s.bonds[0] = [bonds, bonds + 1]  # a bond of particle nb0's own
    s.nb0[0] = bonds
    for f in ("bonds_delta_n", "bonds_omega_n"):
        setattr(s, f, numpy.zeros(bonds))
    for f in ("bonds_delta_t", "bonds_omega_t"):
        setattr(s, f, numpy.zeros((bonds, 3)))
    s.vel[:, :3] = rng.normal(0.0, 1.0, (n, 3))
    s.sigma_b[0] = s.tau_b[0] = 1.0e7
    image = s.tobytes()
    ref = oracle.Oracle(image)
    with engine.Context(image) as ctx:
        for k in range(4):
            ctx.step(3)
            ref.step(3)
            for f in ("bonds", "bonds_delta", "force", "torque", "x", "vel", "angvel"):
                assert numpy.array_equal(ctx.get(f), ref.get(f)), (k, f)
    assert numpy.count_nonzero(ref.get("bonds")[:, 0] == bonds) > bonds // 8


# A segmented reverse pass goes back to a checkpoint whose hit masks another
# number of lanes wrote.  Particle 0 holds particle 2 (the second entry of its
# list: bit 4 of a mask of eight lanes) and loses it in the very step in which
# particle 3 (the third entry: bit 4 with sixteen lanes) reaches it, the first
# of the reverse pass.
@pytest.mark.parametrize("lanes", [1, 4, 8, 16])
def test_adjoint_segments_after_a_change_of_lanes(lanes):
    r, dt, v = 0.01, 1.0e-5, 0.01
    s = sim(np=5, sid="lanes")
    s.radius[:] = [r, r, r, r, 0.03]
    d = 4.5 * v * dt  # an overlap and a gap that both end after 4.5 steps
    s.x = numpy.array([0.06, 0.03, 0.03]) + numpy.array([
        [0.0, 0.0, 0.0], [2.02 * r, 0.0, 0.0], [0.0, 2.0 * r - d, 0.0], [0.0, 0.0, 2.0 * r + d],
        [0.1, 0.1, 0.1]])
    s.vel[2, 1], s.vel[3, 2] = v, -v
    s.defaultParams(mu_s=0.5, mu_d=0.5, rho=2600.0, k_n=1.0e3, k_t=1.0e3)
    s.g[:] = 0.0
    s.normalBoundariesXY()
    s.defineWorldBoundaries(L=[0.24, 0.24, 0.24])
    s.time_dt[0], s.time_current[0], s.time_total[0], s.time_file_dt[0] = dt, 0.0, 1.0, 1.0
    image = s.tobytes()
    seed = numpy.random.default_rng(3).standard_normal((5, 3))
    ref = oracle.Oracle(image)
    held = []
    for n in (5, 1):
        ref.step(n)
        held.append(set(ref.get("contacts")[0]) - {5})
    assert held == [{2}, {3}]
    got = []
    for checkpoint in (0, 5):
        with engine.Context(image) as ctx:
            ctx.step(5)
            ctx.set_scalar("contact_lanes", lanes)
            ctx.set_scalar("adj_checkpoint", checkpoint)
            g = ctx.adjoint(10, seed, seed, None)
            got.append([g["x"], g["v"], ctx.get("contacts"), ctx.get("x")])
    # The same steps reversed in the same order.
    for a, b in zip(*got):
        assert numpy.array_equal(a, b)


def _contact_case(case):
    s = {"settling": lambda: cases.settling_case(1200, 12), "crowded": cases.crowded_case,
         "fcc": cases.fcc_case, "shear1k": lambda: cases.fixture("shear1k.bin"),
         "bed": lambda: cases.lattice_bed(18500, 8, 0.01, 0.1)}[case.split("-")[0]]()
    if case.endswith("hertz"):
        s.contactmodel[0] = 3
    return s


# The contact pass of large contexts (four lanes, workgroups of 256, apart from
# the integration) on small beds, where the default settings take the pass of
# eight lanes that also integrates (another setting of the integration leaves
# it), that default pass, and a Hertzian bed just above its limit: re-sorts,
# a row that overflows, several rounds of contacts a wavefront, either order of
# the workgroups.
@pytest.mark.parametrize("form", ["four lanes", "default"])
@pytest.mark.parametrize("case", ["settling", "settling-hertz", "crowded", "crowded-hertz", "fcc",
                                  "fcc-hertz", "shear1k-hertz", "shear1k-xcd", "bed-hertz"])
def test_contact_pass_of_either_form(case, form):
    s = _contact_case(case)
    image, steps = s.tobytes(), 10 if case == "bed-hertz" else 50
    ref = oracle.Oracle(image)
    with engine.Context(image) as ctx:
        if case.endswith("xcd"):
            ctx.set_scalar("xcd_order", 1)
        if form == "four lanes":
            ctx.set_scalar("integrate_lanes", 4)
        ctx.profile(True)
        for _ in range(4):
            ctx.step(steps)
            ref.step(steps)
            for f in ("perm", "contacts", "x", "vel", "angvel", "force", "torque", "p", "es", "ev",
                      "delta_t"):
                assert numpy.array_equal(ctx.get(f), ref.get(f)), f
        stages = {k: n for k, (_, n) in ctx.profile_report().items()}
    apart = form == "four lanes" or case == "bed-hertz"
    assert ("integrate" in stages) == apart and ("contact_integrate" in stages) != apart, stages


# A kept tape many times larger than the next context's is given back, and that
# context's own is kept instead.
def test_adjoint_tape_kept_follows_use():
    import torch
    small, large = (cases.lattice_bed(n, 4, 0.01, 0.1).tobytes() for n in (60, 900))

    def adjoint(image, n, steps):
        with engine.Context(image) as ctx:
            return ctx.adjoint(steps, numpy.ones((n, 3)), None, None)["x"]

    def free():
        torch.cuda.synchronize()
        return torch.cuda.mem_get_info()[0]

    want = adjoint(small, 60, 7)
    engine.trim()
    before = free()
    adjoint(large, 900, 300)  # 1,260 bytes a particle and step: 0.39 GB
    assert before - free() > 0.3e9
    for _ in range(2):
        assert numpy.array_equal(adjoint(small, 60, 7), want)
        assert before - free() < 0.1e9
    engine.trim()


# An iteration counter of the other parity right after a step that ended by
# re-sorting for the next one: the request to rebuild the lists in the new
# order was noted for a step of the parity that does not come.
@pytest.mark.parametrize("model", [1, 2, 3])
@pytest.mark.parametrize("n", [3000, 20000])
def test_counter_parity_after_a_resort(n, model):
    rng = numpy.random.default_rng(n)
    s = _cloud(n, 13, r=(0.004, 0.006) if n == 20000 else (0.008, 0.012))
    cell = float(s.L[0]) / int(s.num[0])
    s.vel[:, :3] = rng.uniform(-0.002, 0.002, (n, 3)) * cell / float(s.time_dt[0])
    s.contactmodel[0] = model
    image = s.tobytes()
    ref = oracle.Oracle(image)
    with engine.Context(image) as ctx:
        ctx.set_scalar("sort_mode", 1)
        for k in range(6):
            sorts = ctx.scalar("sorts")
            ctx.step(1 + k % 2)
            ref.step(1 + k % 2)
            assert ctx.scalar("sorts") > sorts
            ctx.set_scalar("iter", ctx.scalar("iter") + 1)
            ctx.step(1)
            ref.step(1)
            for f in ("perm", "contacts", "x", "vel", "force", "p"):
                assert numpy.array_equal(ctx.get(f), ref.get(f)), (k, f)


# Particles of more overlaps than the search keeps (8): the first of a cluster
# of n in which all overlap has n - 1, ordered in LDS (up to 512) or in place,
# beside particles of few; clusters on both sides of a block of 64, and a
# particle that touches 300 others of one small size.
@pytest.mark.parametrize("n", [9, 10, 74, 513, 514, 700, 1500, "one"])
def test_overlap_lists_of_many(n):
    rng = numpy.random.default_rng(7)
    if n == "one":
        s = _cloud(301, 3)
        u = rng.standard_normal((300, 3))
        s.radius[0], s.radius[1:] = 0.2, 0.004
        s.x[0] = 0.25
        s.x[1:] = 0.25 + 0.201 * u / numpy.linalg.norm(u, axis=1)[:, None]
        order = rng.permutation(301)
        s.radius, s.x = s.radius[order], s.x[order]
    else:
        s = _cloud(n + 200, 3, r=(0.004, 0.006))
        s.x[60:60 + n] = 0.25 + rng.uniform(-0.002, 0.002, (n, 3))
    image = s.tobytes()
    pb, db = oracle.Oracle(image).find_overlaps()
    assert numpy.bincount(pb[:, 0]).max() >= (8 if n == "one" else n - 1)
    with engine.Context(image) as ctx:
        pa, da = ctx.find_overlaps()
        assert numpy.array_equal(pa, pb) and numpy.array_equal(da, db)


# The automatic re-sort placement: a falling lattice, whose movers are few but
# shift whole layers of the order at every step, is sorted by the launches; a
# bed whose movers shift little is re-sorted by the walls kernel.  The launches
# measure what the other placement would rewrite, and change nothing.
@pytest.mark.parametrize("n,speed,launched", [(60000, 0.0, True), (40000, 0.05, False)])
def test_resort_placement_follows_what_is_rewritten(n, speed, launched):
    rng = numpy.random.default_rng(n)
    s = cases.lattice_bed(n, 4, 0.01, 0.1)
    if not launched:
        s.radius *= 0.4
        s.g[:] = 0.0
        s.vel[:, :3] = rng.normal(0.0, speed, (n, 3))
        s.fixvel[:] = 0.0
    image = s.tobytes()
    fields = ("perm", "cellid", "contacts", "x", "vel", "force")
    with engine.Context(image) as ctx, engine.Context(image) as other:
        other.set_scalar("sort_mode", 0 if not launched else 1)
        for _ in range(8):
            ctx.step(100)
            other.step(100)
        ctx.profile(True)
        ctx.step(20)
        other.step(20)
        assert ("sort" in ctx.profile_report()) == launched
        assert ctx.scalar("sorts") > 100
        for f in fields:
            assert numpy.array_equal(ctx.get(f), other.get(f)), f
