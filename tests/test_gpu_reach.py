"""The force kernel leaves out stencil columns and rows that an agent's cutoff does not
reach.  Forces against the CPU oracle (FP64 within 1e-12, mixed within 1e-5) where that
can go wrong: voxels as wide as the cutoff, a hair wider and several times wider, boxes
whose voxels differ per axis, agents on and next to voxel borders, pairs at the cutoff
across corners, one- and two-voxel grids, and an agent that keeps a voxel its position
is not in."""
import numpy as np
import pytest

from cellular_raza_amd import CartesianCuboid, InstanceSpec, MechanicsBackend, MorsePotential, NewtonDamped
from oracle.oracle import OracleSim

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-12, "mixed": 1e-5}


def rel_err(a, b):
    return np.linalg.norm(a - b, axis=1).max() / max(np.linalg.norm(b, axis=1).max(), 1e-300)


def compare(dom, pot, pos, precision):
    spec = [InstanceSpec(dom, pot, NewtonDamped(1.0, 1.0))]
    g, o = MechanicsBackend(spec, dt=0.01, precision=precision), OracleSim(spec, dt=0.01)
    for s in (g, o):
        s.set_agents(pos)
    assert rel_err(g.compute_forces(), o.compute_forces()) <= TOL[precision]
    g.close()
    o.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n_voxels", [(1, 1, 1), (2, 1, 3), (5, 5, 5), (4, 9, 6), (11, 3, 7)])
def test_cutoffs_up_to_the_voxel_edge(n_voxels, dim, precision):
    n_voxels = n_voxels[-dim:]
    rng = np.random.default_rng(sum(n_voxels))
    edges = np.array([2.0, 3.1, 2.6])[-dim:]
    dom = CartesianCuboid.from_boundaries_and_n_voxels([-1.0] * dim, list(-1.0 + edges * n_voxels), n_voxels)
    n = 40 * int(np.prod(n_voxels)) if dim == 2 else 15 * int(np.prod(n_voxels))
    pos = -1.0 + rng.uniform(1e-9, 1.0, (n, dim)) * edges * n_voxels
    # agents on voxel borders and within rounding of them
    for a in range(n // 4):
        k = rng.integers(0, dim)
        at = -1.0 + edges[k] * rng.integers(0, n_voxels[k])
        pos[a, k] = at + rng.choice([0.0, 1e-15, -1e-15, 1e-9, -1e-9])
    pos = np.clip(pos, -1.0 + 1e-12, -1.0 + edges * n_voxels - 1e-9)
    for cutoff in (edges.min(), 0.999 * edges.min(), 0.5 * edges.min(), 0.05):
        compare(dom, MorsePotential(0.4, 1.0, float(cutoff), 0.5), pos, precision)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_pairs_at_the_cutoff_across_corners(precision):
    """Pairs whose distance is the cutoff +- 1e-9 along directions through the corners
    and edges of the voxels: the force jumps there, so a lost pair shows."""
    rng = np.random.default_rng(5)
    dom = CartesianCuboid.from_boundaries_and_interaction_range([0.0] * 3, [60.0] * 3, 2.5)
    pos = []
    for i in range(9):
        for j in range(9):
            corner = np.array([5.0 + 5.0 * i, 5.0 + 5.0 * j, 5.0 + 5.0 * ((i + j) % 9)])
            u = rng.normal(size=3) * [rng.choice([0.02, 1.0]), 1.0, 1.0]
            u /= np.linalg.norm(u)
            t, eps = rng.uniform(0.05, 0.95), rng.choice([-1e-9, 1e-9])
            pos += [corner - u * 2.5 * t, corner + u * (2.5 * (1.0 - t) + eps)]
    compare(dom, MorsePotential(1.0, 1.0, 2.5, 0.5), np.array(pos), precision)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_an_agent_outside_its_voxel_keeps_its_pairs(precision):
    """An agent that a step puts exactly on the domain's maximum has no voxel there and
    stays in the old one, several voxels away: pairs of the old voxel's stencil count
    as in the reference, whatever their distance to that voxel's borders."""
    dom = CartesianCuboid.from_boundaries_and_n_voxels([0.0, 0.0], [40.0, 40.0], [4, 4])
    pos = np.array([[32.0, 25.0], [33.0, 25.5], [39.5, 25.2], [20.5, 25.0], [39.0, 11.0]])
    vel = np.zeros_like(pos)
    vel[0, 0] = 8.0  # one Euler step of dt 1: x = 40 = max
    spec = [InstanceSpec(dom, MorsePotential(1.0, 0.5, 4.0, 0.5), NewtonDamped(0.0, 1.0))]
    g = MechanicsBackend(spec, dt=1.0, precision=precision, mechanics_solver_order=0)
    o = OracleSim(spec, dt=1.0, mechanics_solver_order=0)
    for s in (g, o):
        s.set_agents(pos, vel)
        s.step(1)
    assert g.get_state()[0][0, 0] == 40.0
    assert rel_err(g.compute_forces(), o.compute_forces()) <= TOL[precision]
    g.close()
    o.close()
