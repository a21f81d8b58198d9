"""Read-backs on both sides of every line between their transfer paths: the rows are the
caller's own bit for bit, and one agent more does not make the call jump.  The time that
is compared is the median of many calls into the same memory; the next path may cost
half as much again at the line, where paths that start a thread for a quarter of a
megabyte took two to three times as much as the one below them."""
import time

import numpy as np
import pytest

from cellular_raza_amd import CartesianCuboid, InstanceSpec, MechanicsBackend, NewtonDamped, NoInteraction, _abi

pytestmark = pytest.mark.gpu

KIB = 1024


def context(n):
    dom = CartesianCuboid.from_boundaries_and_n_voxels([0.0] * 3, [10.0] * 3, [7, 5, 9])
    g = MechanicsBackend([InstanceSpec(dom, NoInteraction(), NewtonDamped(1.0, 1.0))], dt=0.01)
    rng = np.random.default_rng(n)
    pos, vel = rng.uniform(1e-9, 10.0, (n, 3)), rng.normal(size=(n, 3))
    g.set_agents(pos, vel)
    return g, pos, vel


# bytes at which a read could change its path, and the parts and threads of one path
LINES = [256 * KIB, 512 * KIB, 1024 * KIB, 1536 * KIB, 2048 * KIB, 3072 * KIB, 4096 * KIB, 8192 * KIB]


@pytest.mark.parametrize("arrays", [1, 2])
@pytest.mark.parametrize("line", LINES)
@pytest.mark.parametrize("over", [0, 1])
def test_rows_at_the_lines(line, over, arrays):
    n = line // (24 * arrays) + over
    g, pos, vel = context(n)
    for _ in range(2):  # the second read finds what the first one left behind
        if arrays == 2:
            p, v = g.get_state()
            assert np.array_equal(v, vel)
        else:
            p = g.get_positions()
        assert np.array_equal(p, pos)
    assert np.array_equal(g.compute_forces(), np.zeros((n, 3)))
    g.close()


@pytest.mark.parametrize("arrays", [1, 2])
@pytest.mark.parametrize("line", LINES)
def test_no_jump_at_the_lines(line, arrays):
    sides = []
    for n in (line // (24 * arrays), line // (24 * arrays) + 1):
        g, pos, _ = context(n)
        out = [np.zeros((n, 3)) for _ in range(2)]
        sides.append((g, pos, out, [x.ctypes.data_as(_abi.DP) for x in out], []))
    for _ in range(60):  # in turn, so that what else the host does falls on both
        for g, _, _, ptr, t in sides:
            t0 = time.perf_counter()
            g._check(g._lib.crm_get_state(g._h, ptr[0], ptr[1] if arrays == 2 else None))
            t.append(time.perf_counter() - t0)
    below, above = (float(np.median(t[10:])) for *_, t in sides)
    for g, pos, out, _, _ in sides:
        assert np.array_equal(out[0], pos)
        g.close()
    assert above <= 1.5 * below + 5e-6, (below, above)
