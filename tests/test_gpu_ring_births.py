"""The Adams-Bashforth ring of point agents, with and without ones born by divisions, after
a call that ends early at an error: the entry that the steps before the last one do not
carry over is brought along from the failing step, so that history, snapshot and state
equal those of one-step calls bit for bit."""
import numpy as np
import pytest

from cellular_raza_amd import CartesianCuboid, InstanceSpec, MechanicsBackend, MorsePotential, NewtonDamped, SimulationError

pytestmark = pytest.mark.gpu


def make(graph, precision, dim):
    dom = CartesianCuboid.from_boundaries_and_interaction_range([0.0] * dim, [30.0] * dim, 3.0)
    # the velocity of a free agent grows by about a third in every step
    g = MechanicsBackend([InstanceSpec(dom, MorsePotential(0.5, 1.0, 3.0, 0.1), NewtonDamped(-3.0, 1.0))], dt=0.1,
                         mechanics_solver_order=2, graph=graph, precision=precision)
    rng = np.random.default_rng(8)
    g.set_agents(rng.uniform(0.0, 30.0, (2000, dim)), rng.normal(0.0, 0.01, (2000, dim)))
    return g


def same(a, b):
    for x, y in zip(a.get_state(), b.get_state()):
        assert np.array_equal(x, y)
    ha, hb = a.get_history(), b.get_history()
    assert ha[2] == hb[2]
    assert np.array_equal(ha[0], hb[0]) and np.array_equal(ha[1], hb[1])
    sa, sb = a.snapshot(), b.snapshot()
    assert all(np.array_equal(sa[k], sb[k]) for k in sa)
    assert np.array_equal(a.identifiers()["history_held"], b.identifiers()["history_held"])
    assert np.array_equal(a.voxel_order(), b.voxel_order())


@pytest.mark.parametrize("dim,precision", [(2, "fp64"), (3, "mixed")])
@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("births", [False, True])
def test_history_after_an_error(births, graph, dim, precision):
    failed = set()
    for speed in (2.0, 10.0, 150.0, 220.0, 1000.0):
        a, one = make(graph, precision, dim), make(False, precision, dim)
        for g in (a, one):
            g.step(9)
            if births:
                x = g.get_positions()
                mothers = np.arange(0, 2000, 3)
                vel = np.zeros((len(mothers), dim))
                vel[5, 0] = speed  # the daughter that will leave the domain
                g.insert_agents(mothers, x[mothers] * 0.999 + 0.01, daughter_vel=vel)
            g.step(1 if speed < 5.0 else 0)
        steps = 0
        with pytest.raises(SimulationError, match="BoundaryError"):
            for steps in range(60):
                one.step(1)
        with pytest.raises(SimulationError, match="BoundaryError"):
            a.step(60)
        assert a.info().step == one.info().step
        same(a, one)
        failed.add(steps)
        a.close()
        one.close()
    assert max(failed) > 1 and (not births or {0, 1} <= failed), failed
