"""Read-backs in agent order on every transfer path: rows written to pinned memory by
the gathering kernel (up to 256 KiB), chunks of 256 KiB through host threads, and
chunks of 1 MiB (above 4 MiB), at the sizes next to each limit.  The state read right
after set_agents is the caller's own, bit for bit, although the slots are in voxel
order; the forces of a spring without pair interactions are -k (x - c) in closed form
(one product, so exact; the mixed path rounds them once to float)."""
import numpy as np
import pytest

from cellular_raza_amd import (CartesianCuboid, DomainSpring, InstanceSpec, MechanicsBackend, NewtonDamped,
                               NoInteraction, workloads)

pytestmark = pytest.mark.gpu

# agents of a 3-D system whose positions and velocities (48 bytes) end next to 256 KiB,
# to eight chunks of 256 KiB, to 4 MiB and to 8 MiB
SIZES = [1, 5461, 5462, 43690, 43691, 87381, 87382, 174762, 174763, 400001]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_point_rows_in_agent_order(n, precision):
    rng = np.random.default_rng(n)
    dom = CartesianCuboid.from_boundaries_and_n_voxels([0.0] * 3, [10.0] * 3, [7, 5, 9])
    spring = DomainSpring(strength=[2.0] * 3, center=[4.0] * 3)
    g = MechanicsBackend([InstanceSpec(dom, NoInteraction(), NewtonDamped(1.0, 1.0), spring)], dt=0.01,
                         precision=precision)
    pos, vel = rng.uniform(1e-9, 10.0, (n, 3)), rng.normal(size=(n, 3))
    g.set_agents(pos, vel)
    p, v = g.get_state()
    assert np.array_equal(p, pos) and np.array_equal(v, vel)
    assert np.array_equal(g.get_positions(), pos)
    f = -2.0 * (pos - 4.0)
    assert np.array_equal(g.compute_forces(), f.astype(np.float32) if precision == "mixed" else f)
    p, v = g.get_state()  # the forces were read through the spare state buffer
    assert np.array_equal(p, pos) and np.array_equal(v, vel)
    g.step(1)  # an Euler step (the ring holds one entry): x + dt v, reflected
    x = pos + 0.01 * vel
    x = np.where(x < 0.0, -x, np.where(x > 10.0, 20.0 - x, x))
    np.testing.assert_allclose(g.get_positions(), x, rtol=0.0, atol=1e-14)
    dx, dv, held = g.get_history()
    assert held == 1 and np.array_equal(dx[0], vel)
    g.close()


@pytest.mark.parametrize("n", [3, 1024, 1025, 40000])
def test_rod_rows_in_agent_order(n):
    wl = workloads.c3_rods_2d(n=n, seed=n)
    g = MechanicsBackend(wl.instances, dt=wl.dt)
    vel = np.random.default_rng(n).normal(size=(n, 16))
    g.set_agents(wl.pos.reshape(n, -1), vel)
    p, v = g.get_state()
    assert np.array_equal(p, wl.pos.reshape(n, -1)) and np.array_equal(v, vel)
    g.close()
