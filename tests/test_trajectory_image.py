"""A trajectory's .bin image is the template's with the given values, however
the template holds its arrays, and the template stays as it is."""

import numpy
import pytest

from sphere_amd.autograd import Trajectory
from sphere_amd.sim import sim

from . import cases


@pytest.mark.parametrize("k_n", [numpy.array([5.0e5]), numpy.array([5])])
@pytest.mark.parametrize("state", [False, True])
def test_image_of_a_trajectory(k_n, state):
    s = cases.lattice_bed(130, 1, 0.01, 0.1, bond_frac=0.05)
    s.k_n = k_n.copy()
    before = s.tobytes()
    rng = numpy.random.default_rng(2)
    x, v = (rng.random((130, 3)), rng.random((130, 3))) if state else (None, None)
    t = Trajectory(s, 5, 4, params=("k_n", "gamma_n", "mu"))
    got = t.image([1.5e6, 2.5, 0.3], x, v)
    want = sim().frombytes(before)
    for name, value in zip(t.params, (1.5e6, 2.5, 0.3)):
        for field in t.ties[name]:
            getattr(want, field)[0] = value
    if state:
        want.x[:, :3], want.vel[:, :3] = x, v
    assert got == want.tobytes()
    assert s.tobytes() == before and s.k_n.dtype == k_n.dtype


@pytest.mark.parametrize("field,value,first", [
    ("k_n", numpy.float64(5.0e5), 5.0e5), ("k_n", numpy.array(5.0e5), 5.0e5),
    ("k_n", 5.0e5, 5.0e5), ("k_n", numpy.array([[5.0e5]]), 5.0e5),
    ("k_n", numpy.array([5.0e5, 7.0]), 5.0e5),
    ("g", numpy.array([[1.0, 2.0, -9.81]]), [1.0, 2.0, -9.81])])
def test_image_of_a_template_with_other_shapes(field, value, first):
    """A parameter the template holds as a number, or in an array of another
    shape than a decoded one: its first entry changes and nothing else."""
    s = cases.lattice_bed(130, 1, 0.01, 0.1)
    want = sim().frombytes(s.tobytes())
    getattr(want, field)[:] = first
    getattr(want, field)[0] = 1.5e6
    setattr(s, field, value)
    t = Trajectory(s, 5, 4, params=("p",), ties={"p": (field,)})
    assert t.image([1.5e6]) == want.tobytes()
    assert getattr(s, field) is value
