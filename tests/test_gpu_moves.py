"""The next order of a step against the CPU oracle: agents that stay in a voxel keep their
order, movers are appended by previous voxel and position (update_mechanics.rs:418-513).

Free agents (no interaction) with velocities of about a voxel per step, so that voxel
starts, orders and positions equal the oracle's exactly: voxels with more agents than a
wavefront, instances and grids at the edges of workgroups and scan tiles, grids of more
scan tiles than a workgroup scans one by one, agents binned after the forces, rods.
"""
import numpy as np
import pytest

from cellular_raza_amd import (Brownian, CartesianCuboid, InstanceSpec, MechanicsBackend, NewtonDamped, NoInteraction,
                               workloads)
from oracle.oracle import OracleSim

pytestmark = pytest.mark.gpu


def same_order(g, o):
    assert np.array_equal(g.get_voxels()[1], o.get_voxels()[1])
    assert np.array_equal(g.voxel_order(), o.get_voxels()[2].astype(np.uint32))


# voxels per axis, agents per instance
GRIDS = {
    "one_voxel": ((1, 1), [700]),
    "crowded_pair": ((2, 1), [1500]),
    "crowded_3d": ((2, 2, 2), [1000]),
    "ragged": ((4, 3), [1, 63, 64, 65, 255, 256, 257, 2]),
    "one_scan_tile": ((64, 32), [3000]),
    "one_scan_tile_and_one": ((683, 3), [3000]),
    "three_scan_tiles_3d": ((17, 17, 17), [20011]),
    "as_many_tiles_as_scanned": ((1024, 1024), [2000]),
    "wider_scan_tiles": ((1025, 1025), [2000]),
    "wider_scan_tiles_3d": ((102, 103, 104), [50001]),
}


@pytest.mark.parametrize("mech", ["damped", "brownian"])
@pytest.mark.parametrize("name", sorted(GRIDS))
def test_orders_match_oracle(name, mech):
    n, counts = GRIDS[name]
    rng = np.random.default_rng(len(name))
    dom = CartesianCuboid.from_boundaries_and_interaction_range([0.0] * len(n), [float(k) for k in n], 1.0)
    m = NewtonDamped(damping_constant=0.0, mass=1.0) if mech == "damped" else Brownian(diffusion_constant=0.5, kb_temperature=1.0)
    specs = [InstanceSpec(dom, NoInteraction(), m) for _ in counts]
    total = sum(counts)
    pos = rng.uniform(0.001, 0.999, (total, len(n))) * np.array(n)
    vel = rng.normal(0.0, 0.2, (total, len(n)))
    kw = dict(dt=1.0 if mech == "damped" else 0.05, mechanics_solver_order=0,
              noise="none" if mech == "damped" else "philox", seed=4)
    g, o = MechanicsBackend(specs, **kw), OracleSim(specs, **kw)
    g.set_agents(pos, vel, None, counts)
    o.set_agents(pos, vel, None, counts)
    same_order(g, o)
    for steps in (1, 1, 2, 5):
        g.step(steps)
        o.step(steps)
        same_order(g, o)
        # (the normals may differ in their last bits)
        assert np.abs(g.get_state()[0] - o.get_state()[0]).max() <= (0.0 if mech == "damped" else 1e-11 * max(n))
    g.close()
    o.close()


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("noise", ["none", "buffer"])  # binned ahead, and after the forces
def test_rod_orders_match_oracle(noise, graph):
    wl = workloads.c3_rods_2d(n=700, seed=11)
    vel = np.repeat(np.random.default_rng(12).normal(0.0, 300.0, (700, 1, 2)), 8, axis=1).reshape(700, -1)
    kw = dict(dt=wl.dt, mechanics_solver_order=2, noise=noise)
    g, o = MechanicsBackend(wl.instances, graph=graph, **kw), OracleSim(wl.instances, **kw)
    for x in (g, o):
        x.set_agents(wl.pos.reshape(700, -1), vel)
    for steps in (1, 2, 9):
        z = np.zeros((steps, 700, 16)) if noise == "buffer" else None
        g.step(steps, z)
        o.step(steps, z)
        same_order(g, o)
    g.close()
    o.close()
