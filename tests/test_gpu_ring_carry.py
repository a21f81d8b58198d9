"""The Adams-Bashforth ring after calls of several steps.  Steps before the last one of
a long call do not carry over the ring entry that no later step reads; what a caller
sees (get_history, snapshots, the steps after it) equals one-step calls bit for bit, at
call lengths on both sides of the change, in graph replays and single launches, and when
an error ends the call early."""
import numpy as np
import pytest

from cellular_raza_amd import InstanceSpec, MechanicsBackend, RodMechanics, SimulationError, workloads

pytestmark = pytest.mark.gpu


def points(**kw):
    wl = workloads.c2_sorting_3d(n=4000, seed=61)
    g = MechanicsBackend(wl.instances, dt=wl.dt, mechanics_solver_order=2, noise="philox", seed=3, **kw)
    g.set_agents(wl.pos, wl.vel, wl.species)
    return g


def rods(damping=1.5, speed=1.0, **kw):
    wl = workloads.c3_rods_2d(n=300, seed=62)
    m = wl.instances[0].mechanics
    spec = InstanceSpec(wl.instances[0].domain, wl.instances[0].interaction,
                        RodMechanics(n_vertices=8, diffusion_constant=0.0, spring_tension=m.spring_tension,
                                     rigidity=m.rigidity, spring_length=m.spring_length, damping=damping))
    g = MechanicsBackend([spec], dt=wl.dt, mechanics_solver_order=2, **kw)
    vel = np.repeat(np.random.default_rng(63).normal(0.0, speed, (300, 1, 2)), 8, axis=1)
    g.set_agents(wl.pos.reshape(300, -1), vel.reshape(300, -1))
    return g


def same(a, b):
    for x, y in zip(a.get_state(), b.get_state()):
        assert np.array_equal(x, y)
    ha, hb = a.get_history(), b.get_history()
    assert ha[2] == hb[2]
    assert np.array_equal(ha[0], hb[0]) and np.array_equal(ha[1], hb[1])
    sa, sb = a.snapshot(), b.snapshot()
    assert all(np.array_equal(sa[k], sb[k]) for k in sa)


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("make", [points, rods])
def test_history_after_long_calls(make, graph):
    a, one = make(graph=graph), make(graph=False)
    for n in (7, 8, 9, 1, 16, 2, 37):
        a.step(n)
        for _ in range(n):
            one.step(1)
        same(a, one)
    a.close()
    one.close()


@pytest.mark.parametrize("graph", [True, False])
def test_history_after_an_error_in_a_long_call(graph):
    kw = dict(damping=-200.0, speed=2000.0)
    one, steps = rods(graph=False, **kw), 0
    with pytest.raises(SimulationError, match="BoundaryError"):
        for steps in range(40):
            one.step(1)
    assert 1 < steps < 39
    a = rods(graph=graph, **kw)
    with pytest.raises(SimulationError, match="BoundaryError"):
        a.step(40)
    assert a.info().step == one.info().step == steps + 1
    same(a, one)
    a.close()
    one.close()
