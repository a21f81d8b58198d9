"""The tiling of contexts that are not tuned, and the tiles' LDS capacities.

Without crm_autotune the lanes per agent follow from the system's size: many for small
systems, one for large ones.  Forces against the CPU oracle (FP64 within 1e-12, mixed
within 1e-5) at sizes on both sides of each change, and on tiles whose staged records
just fit, or just do not fit, into LDS (those read global memory)."""
import numpy as np
import pytest

from cellular_raza_amd import (CartesianCuboid, InstanceSpec, Langevin, MechanicsBackend, MorsePotential,
                               NewtonDamped, SpeciesMorsePotential, workloads)
from oracle.oracle import OracleSim

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-12, "mixed": 1e-5}


def rel_err(a, b):
    den = np.linalg.norm(b, axis=1).max()
    num = np.linalg.norm(a - b, axis=1).max()
    return num / den if den > 0 else num


def check(instances, pos, species, precision):
    g = MechanicsBackend(instances, dt=0.01, precision=precision)
    o = OracleSim(instances, dt=0.01)
    for s in (g, o):
        s.set_agents(pos, species=species)
    assert rel_err(g.compute_forces(), o.compute_forces()) <= TOL[precision]
    lanes = g.tiling()["lanes_per_agent"]
    g.close()
    o.close()
    return lanes


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("dim", [2, 3])
def test_default_lanes_by_size(dim, precision):
    seen = []
    for n in (1, 2, 63, 1000, 12000, 17000, 30000, 45000, 60000, 110000, 160000):
        wl = (workloads.c4_ensemble_2d(n_instances=1, seed=3, n_min=n, n_max=n) if dim == 2 else
              workloads.c2_sorting_3d(n=n, seed=n))
        seen.append(check(wl.instances, wl.pos, wl.species, precision))
    assert seen == sorted(seen, reverse=True) and seen[0] == 8 and seen[-1] == 1, seen


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("over", [-1, 0, 1, 700])
@pytest.mark.parametrize("dim", [2, 3])
def test_tiles_at_their_lds_capacity(dim, over, precision):
    """One 3^dim-voxel domain: the middle plane's tile stages every agent."""
    cap = {(3, "fp64"): 1152, (2, "fp64"): 1600, (3, "mixed"): 1232, (2, "mixed"): 1232}[dim, precision]
    rng = np.random.default_rng(cap + over)
    dom = CartesianCuboid.from_boundaries_and_interaction_range([0.0] * dim, [30.0] * dim, 10.0)
    n = cap + over
    pos = rng.uniform(1e-6, 30.0, (n, dim))
    if dim == 2:
        inst, sp = [InstanceSpec(dom, MorsePotential(1.0, 1.0, 4.0, 0.5), NewtonDamped(1.0, 1.0))], None
    else:
        pot = SpeciesMorsePotential(1.0, 1.0, 6.0, 0.5, [[1.0, 0.2], [0.3, 0.7]])
        inst, sp = [InstanceSpec(dom, pot, Langevin(1.0, 2.0, 0.01))], rng.integers(0, 2, n).astype(np.int32)
    check(inst, pos, sp, precision)
