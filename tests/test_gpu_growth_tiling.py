"""A population that grows by divisions has the tiling of one that was set up at its size:
the lanes per agent follow the insertions across every change of the default, with the
forces of a fresh context and, where it is small enough, of the CPU oracle (FP64 within
1e-12, mixed within 1e-5), before and after steps in graphs captured for the old tiles."""
import numpy as np
import pytest

from cellular_raza_amd import CartesianCuboid, InstanceSpec, Langevin, MechanicsBackend, SpeciesMorsePotential
from oracle.oracle import OracleSim

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-12, "mixed": 1e-5}
L = 74.0


def rel_err(a, b):
    return np.linalg.norm(a - b, axis=1).max() / np.linalg.norm(b, axis=1).max()


def spec():
    dom = CartesianCuboid.from_boundaries_and_interaction_range([0.0] * 3, [L] * 3, 2.5)
    pot = SpeciesMorsePotential(1.0, 1.0, 2.5, 0.5, [[1.0, 0.2], [0.2, 1.0]])
    return [InstanceSpec(dom, pot, Langevin(1.0, 2.0, 0.01))]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_lanes_follow_a_growing_population(precision):
    rng = np.random.default_rng(5)
    kw = dict(dt=0.005, mechanics_solver_order=2, noise="philox", seed=3, precision=precision)
    g = MechanicsBackend(spec(), **kw)
    pos = rng.uniform(0.0, L, (1100, 3))
    g.set_agents(pos, species=(np.arange(1100) % 2).astype(np.int32))
    species = np.arange(1100) % 2
    seen = [g.tiling()["lanes_per_agent"]]
    while len(pos) < 130000:
        g.step(17)
        pos = g.get_positions()
        n = len(pos)
        g.insert_agents(np.arange(n), rng.uniform(0.0, L, (n, 3)))
        species = np.concatenate([species, species])
        pos = g.get_positions()
        fresh = MechanicsBackend(spec(), **kw)
        fresh.set_agents(pos, species=species.astype(np.int32))
        assert g.tiling() == fresh.tiling()
        seen.append(g.tiling()["lanes_per_agent"])
        f = g.compute_forces()
        assert rel_err(f, fresh.compute_forces()) <= TOL[precision]
        fresh.close()
        if len(pos) < 20000:
            o = OracleSim(spec(), dt=0.005)
            o.set_agents(pos, species=species.astype(np.int32))
            assert rel_err(f, o.compute_forces()) <= TOL[precision]
            o.close()
    g.close()
    assert seen == sorted(seen, reverse=True) and seen[0] == 8 and seen[-1] == 1, seen


def test_a_tuned_tiling_stays():
    """What crm_autotune chose is not chosen again by an insertion."""
    rng = np.random.default_rng(6)
    g = MechanicsBackend(spec(), dt=0.005, autotune=True)
    g.set_agents(rng.uniform(0.0, L, (2000, 3)), species=np.zeros(2000, dtype=np.int32))
    lanes = g.tiling()["lanes_per_agent"]
    while g.n_agents < 64000:
        g.insert_agents(np.arange(g.n_agents), rng.uniform(0.0, L, (g.n_agents, 3)))
        assert g.tiling()["lanes_per_agent"] == lanes
    g.close()
