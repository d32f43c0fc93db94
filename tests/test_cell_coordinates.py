"""The cells searched around a particle exist, however far outside the grid it
is."""

import os
import subprocess

import numpy
import pytest

from sphere_amd import build, engine
from sphere_amd.sim import sim

CSRC = os.path.join(os.path.dirname(os.path.abspath(build.__file__)), "csrc")

# The 27 cells around (x, y, z), unrolled as the kernels unroll them: code and
# target of each.
SOURCE = """
#include "dem_cells.hpp"
struct Params { uint32_t num[3]; int32_t periodic; };
extern "C" void cells(const uint32_t* num, int periodic, double x, double y, double z, int* out) {
    Params p = {{num[0], num[1], num[2]}, periodic};
    const int gx = sphx::cell_coord(x, (int)p.num[0]);
    const int gy = sphx::cell_coord(y, (int)p.num[1]);
    const int gz = sphx::cell_coord(z, (int)p.num[2]);
#pragma unroll
    for (int k = 0; k < 27; ++k) {
        int tx = gx + k % 3 - 1, ty = gy + (k / 3) % 3 - 1;
        const int tz = gz + k / 9 - 1;
        const int code = sphx::find_dist_mod(p, tx, ty, tz);
        out[4 * k] = code;
        out[4 * k + 1] = tx;
        out[4 * k + 2] = ty;
        out[4 * k + 3] = tz;
    }
}
"""


def _want(num, periodic, g):
    """The cells around g by whole numbers of any size."""
    rows = []
    for k in range(27):
        t = [g[0] + k % 3 - 1, g[1] + (k // 3) % 3 - 1, g[2] + k // 9 - 1]
        code = 0
        for d in range(2):
            if periodic == 1 or (periodic == 2 and d == 0):
                if t[d] < 0:
                    t[d] += num[d]
                    code |= 1 << (2 * d)
                if t[d] >= num[d]:
                    t[d] -= num[d]
                    code |= 2 << (2 * d)
        inside = all(0 <= t[d] < num[d] for d in range(3))
        rows.append([code] + t if inside else None)
    return rows


def test_cells_around_any_coordinate(tmp_path):
    import ctypes
    src, lib = str(tmp_path / "cells.hip"), str(tmp_path / "cells.so")
    with open(src, "w") as fh:
        fh.write(SOURCE)
    subprocess.run([build.hipcc(), "--cuda-host-only", "-O3", "-ffp-contract=off", "-fPIC",
                    "-shared", "-I", CSRC, src, "-o", lib], check=True, capture_output=True)
    L = ctypes.CDLL(lib)
    L.cells.argtypes = [ctypes.c_void_p, ctypes.c_int] + [ctypes.c_double] * 3 + [ctypes.c_void_p]
    num = numpy.array([5, 7, 3], dtype=numpy.uint32)
    out = numpy.zeros((27, 4), dtype=numpy.int32)
    big = [2.0 ** 31, 2.0 ** 31 - 1, 2.0 ** 31 - 2, 2.0 ** 32, 5.7e8, 1e19, 1e300, numpy.inf]
    values = [float(v) + 0.25 for v in range(-20, 21)] + big + [-v for v in big]
    for periodic in (0, 1, 2):
        for d in range(3):
            for v in values:
                c = [2.5, 3.5, 1.5]
                c[d] = v
                L.cells(num.ctypes.data, periodic, *c, out.ctypes.data)
                g = [int(numpy.floor(min(max(w, -1e25), 1e25))) for w in c]
                want = _want([int(n) for n in num], periodic, g)
                for k in range(27):
                    got = None if out[k, 0] < 0 else out[k].tolist()
                    assert got == want[k], (periodic, c, k)


@pytest.mark.gpu
@pytest.mark.parametrize("model,lanes,db", [(1, 4, 0.0), (1, 4, 1.0e-4), (2, 1, 0.0), (2, 4, 0.0),
                                            (2, 8, 0.0), (2, 16, 0.0), (3, 4, 0.0)])
@pytest.mark.parametrize("periodic", [0, 1])
def test_particles_far_outside_are_reported(model, lanes, db, periodic):
    """Two particles 5e8 m and 1e200 m outside a grid of 5 x 5 x 5 cells: the
    step runs, the error is reported, and the other particles move as with
    those two a few metres outside."""
    rng = numpy.random.default_rng(2)
    n = 200
    s = sim(np=n, sid="far")
    s.radius[:] = 0.02
    s.x = rng.uniform(0.02, 0.18, (n, 3))
    (s.periodicBoundariesXY if periodic else s.normalBoundariesXY)()
    s.defineWorldBoundaries(L=[0.2, 0.2, 0.2])
    assert list(s.num) == [5, 5, 5]
    s.defaultParams(rho=2600.0, k_n=1.0e5, k_t=1.0e5)
    s.contactmodel[0] = model
    s.kappa[0], s.db[0], s.V_b[0] = 1.0e-3, db, 1.0e-12
    s.initTemporal(total=1.0, file_dt=0.1, dt=1.0e-7)
    image = s.tobytes()
    states = []
    for far in ((5.0e8, 1.0e200), (7.0, 9.0)):
        with engine.Context(image) as ctx:
            ctx.set_scalar("contact_lanes", lanes)
            ctx.step(1)
            x = ctx.get("x").copy()
            x[5, 2], x[9, 2] = far
            ctx.set("x", x)
            ctx.step(2, sync=False)
            keep = numpy.setdiff1d(numpy.arange(n), [5, 9])
            states.append([ctx.get(f)[keep] for f in ("x", "vel", "force", "p")])
            with pytest.raises(engine.EngineError, match="outside the grid"):
                ctx.sync()
    for a, b in zip(*states):
        assert numpy.count_nonzero(a) and numpy.array_equal(a, b)
