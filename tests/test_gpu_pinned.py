"""Pinned host memory: calls borrow it from a pool of the process, so that contexts hold
none of their own, and contexts on threads of their own do not see each other's rows."""
import threading

import numpy as np
import pytest

from cellular_raza_amd import CartesianCuboid, InstanceSpec, MechanicsBackend, NewtonDamped, NoInteraction, SimulationError

pytestmark = pytest.mark.gpu


def context(n, seed):
    dom = CartesianCuboid.from_boundaries_and_n_voxels([0.0] * 2, [10.0] * 2, [70, 50])
    g = MechanicsBackend([InstanceSpec(dom, NoInteraction(), NewtonDamped(1.0, 1.0))], dt=0.01)
    rng = np.random.default_rng(seed)
    pos, vel = rng.uniform(1e-9, 10.0, (n, 2)), rng.normal(size=(n, 2))
    g.set_agents(pos, vel)
    return g, pos, vel


def mapped():
    """KiB of address space of this process."""
    with open("/proc/self/status") as f:
        return next(int(line.split()[1]) for line in f if line.startswith("VmSize"))


def test_reads_leave_no_memory_with_the_context():
    """What large reads of 128 contexts add to the address space is less than half of a block
    of 8 MiB for each.  (The first context's have brought the runtime's own; the reading
    threads' heaps, 64 MiB of it each, are at most seven.)"""
    made = [context(140000, k)[0] for k in range(129)]
    for _ in range(3):
        made[0].get_state()
    before = mapped()
    for g in made[1:]:
        g.get_state()
    grown = mapped() - before
    for g in made:
        g.close()
    assert grown < 128 * 4096, grown


def test_reads_on_many_threads():
    """More threads than the pool keeps blocks, in every transfer path."""
    bad = []

    def work(k):
        for n in (1, 5000, 20000, 60000, 140000):
            g, pos, vel = context(n + k, 100 * k + 1)
            for _ in range(3):
                p, v = g.get_state()
                if not (np.array_equal(p, pos) and np.array_equal(v, vel)):
                    bad.append((k, n))
            g.close()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    g, pos, vel = context(50000, 7)  # after the last context's end the pool begins anew
    assert np.array_equal(g.get_state()[0], pos)
    g.close()


def test_steps_and_errors_on_many_threads():
    """Every step reads the control block: more threads than the pool keeps blocks, one of
    them with an agent that leaves the domain."""
    bad = []

    def work(k):
        dom = CartesianCuboid.from_boundaries_and_n_voxels([0.0] * 2, [10.0] * 2, [7, 5])
        g = MechanicsBackend([InstanceSpec(dom, NoInteraction(), NewtonDamped(-5.0 if k == 3 else 0.0, 1.0))], dt=0.1,
                             mechanics_solver_order=0)
        pos, vel = np.full((300, 2), 5.0), np.zeros((300, 2))
        vel[7, 0] = 5.0 if k == 3 else 0.01 * (k + 1)
        g.set_agents(pos, vel)
        done = 0
        try:
            for done in range(60):
                g.step(1)
        except SimulationError as e:
            if k != 3 or e.kind != "BoundaryError":
                bad.append((k, done, str(e)))
            failed.append(done)
        if k != 3:
            want = 5.0
            for _ in range(60):
                want = want + 0.1 * (0.01 * (k + 1))
            if g.info().step != 60 or g.get_positions()[7, 0] != want:
                bad.append((k, done, g.get_positions()[7, 0], want))
        g.close()

    failed = []
    threads = [threading.Thread(target=work, args=(k,)) for k in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad and len(failed) == 1, (bad, failed)
