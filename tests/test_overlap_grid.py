"""The choice of the overlap search's grid: it always ends, and every
overlapping pair lies in adjacent cells of it."""

import os
import subprocess
import sys

import numpy
import pytest

import oracle
from sphere_amd import build, engine
from sphere_amd.sim import sim

CSRC = os.path.join(os.path.dirname(os.path.abspath(build.__file__)), "csrc")

# (Positions or a radius that are not finite arrive as the flag 0.)
SOURCE = """
#include "overlap_grid.hpp"
extern "C" void choose(const double* v, uint32_t ncap, double* out) {
    double b[8];
    for (int k = 0; k < 8; ++k) b[k] = v[k];
    sphx::OverlapGrid g;
    sphx::choose_overlap_grid(b, ncap, g);
    out[0] = g.use;
    out[1] = g.inv_h;
    for (int d = 0; d < 3; ++d) out[2 + d] = g.n[d];
}
"""

CALL = """
import ctypes, sys
L = ctypes.CDLL(sys.argv[1])
for line in sys.stdin:
    v = [float(x) for x in line.split()]
    out = (ctypes.c_double * 5)()
    L.choose((ctypes.c_double * 8)(*v[:8]), ctypes.c_uint32(int(v[8])), out)
    print(*[repr(x) for x in out])
"""


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    """The device's grid choice compiled for the host, called in a process
    with a time limit."""
    d = tmp_path_factory.mktemp("grid")
    src, lib = str(d / "grid.hip"), str(d / "grid.so")
    with open(src, "w") as fh:
        fh.write(SOURCE)
    subprocess.run([build.hipcc(), "--cuda-host-only", "-O2", "-ffp-contract=off", "-fPIC",
                    "-shared", "-I", CSRC, src, "-o", lib], check=True, capture_output=True)

    def call(rows):
        p = subprocess.run([sys.executable, "-c", CALL, lib], text=True, timeout=60, check=True,
                           input="\n".join(" ".join(repr(float(x)) for x in r) for r in rows),
                           capture_output=True)
        return [[float(x) for x in line.split()] for line in p.stdout.splitlines()]
    return call


def test_extents_that_overflow_have_no_grid(choose):
    big = 1.0e308
    rows = [[-big, 0, 0, big, 1, 1, 0.1, 1, 4096],
            [-big, -big, -big, big, big, big, 0.1, 1, 4096],
            [0, -big, 0, 1, big, 1, big, 1, 200006],
            [0, 0, 0, 1, 1, 1, 0.1, 0, 4096]]
    assert [g[0] for g in choose(rows)] == [0.0] * 4


def test_every_finite_extent_has_a_grid(choose):
    rng = numpy.random.default_rng(5)
    rows = []
    for k in range(2000):
        lo = rng.uniform(-1.0, 1.0, 3) * 10.0 ** rng.uniform(-300, 300)
        ext = rng.uniform(0.0, 1.0, 3) * 10.0 ** rng.uniform(-300, 300, 3)
        ext[rng.uniform(size=3) < 0.2] = 0.0
        r = 0.0 if rng.uniform() < 0.1 else 10.0 ** rng.uniform(-300, 307)
        rows.append([*lo, *(lo + ext), r, 1.0, rng.integers(4096, 1 << 22)])
    # The slowest: a cell from the smallest double up to the largest extent.
    rows.append([0, 0, 0, 5e-324, 0, 0, 0, 1, 4096])
    rows.append([-8e307, 0, 0, 8e307, 0, 0, 0, 1, 4096])
    for r, g in zip(rows, choose(rows)):
        assert g[0] == 1.0, r
        assert numpy.prod(g[2:]) <= r[8], r
        # (Where the cell's side and its inverse are representable.)
        if 1e-300 < 2.0 * r[6] < 1e300 and max(map(abs, r[:6])) < 1e300:
            assert g[1] * 2.0 * r[6] <= 1.0, r


@pytest.mark.gpu
def test_positions_apart_by_more_than_a_double():
    """Finite positions whose distance overflows: the all-pairs search."""
    n = 130
    rng = numpy.random.default_rng(1)
    s = sim(np=n, sid="apart")
    s.radius[:] = 0.01
    s.x = rng.uniform(0.02, 0.18, (n, 3))
    s.defineWorldBoundaries(L=[0.2, 0.2, 0.2])
    s.initTemporal(total=1.0, file_dt=0.1)
    image = s.tobytes()
    with engine.Context(image) as ctx:
        ref = oracle.Oracle(image)
        x = ctx.get("x").copy()
        x[3, 0], x[77, 0] = -1.0e308, 1.0e308
        ctx.set("x", x)
        ref.set("x", x)
        pairs, delta = ctx.find_overlaps()
        want, wdelta = ref.find_overlaps()
        assert len(want) > 10
        assert numpy.array_equal(pairs, want) and numpy.array_equal(delta, wdelta)
