"""Requests admitted under different cell scalings served in the same steps: those on unit cells go to one launch of a
step, the others to a second one that shares its buffers.  Each result is that of the request served alone (the masses
are summed in another order: 1e-6 of the largest density covers the FP32 result)."""

import time

import numpy as np
import pytest

import adeco_amd as A
from adeco_amd.lattice import make_lattice

pytestmark = pytest.mark.gpu

# boxes that are no cubes: under the reference's scaling their cells are no unit cells
LONG = ([5.0, 95.0, 10.0, 80.0, 8.0, 90.0], 224)
SHORT = ([20.0, 70.0, 15.0, 55.0, 30.0, 90.0], 96)


@pytest.fixture(autouse=True)
def exact_scaling():
    A.set_cell_scaling(A.SCALING_EXACT)
    yield
    A.set_cell_scaling(A.SCALING_EXACT)


def alone(rl, request, scaling):
    A.set_cell_scaling(scaling)
    with A.Server(rl) as srv:
        return srv.wait(srv.submit(*request), timeout=60)[0]


def admitted(srv):
    for _ in range(20000):
        s = srv.stats()
        if s["active"] or s["requests_done"]:
            return
        time.sleep(1e-4)
    raise AssertionError("not admitted")


@pytest.mark.parametrize("first", [A.SCALING_EXACT, A.SCALING_REFERENCE])
def test_steps_of_both_forms(first):
    other = A.SCALING_REFERENCE if first == A.SCALING_EXACT else A.SCALING_EXACT
    lat = make_lattice(20, 2.0, seed=5)
    with A.ResidentLattice.from_lattice(lat) as rl:
        want = alone(rl, LONG, first), alone(rl, SHORT, other)
        A.set_cell_scaling(first)
        print(f"[serve forms] first {first}", flush=True)
        with A.Server(rl, step_tiles=64) as srv:
            a = srv.submit(*LONG)
            admitted(srv)
            A.set_cell_scaling(other)
            b = srv.submit(*SHORT)
            got_b, info_b = srv.wait(b, timeout=60)
            got_a, info_a = srv.wait(a, timeout=60)
    assert info_a["t_admit"] <= info_b["t_admit"] < info_a["t_done"]  # some steps held both
    for got, w in zip((got_a, got_b), want):
        assert w.max() > 0 and np.abs(got - w).max() <= 1e-6 * w.max()
