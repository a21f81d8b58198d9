"""Mie potentials whose exponents are not integers (or beyond the integer powers' range)
run kernels of their own: forces against the CPU oracle (FP64 within 1e-12, mixed within
1e-5) for points and rods, with one exponent or both, and in ensembles where a single
instance has them; and the states after graph steps."""
import numpy as np
import pytest

from cellular_raza_amd import (CartesianCuboid, InstanceSpec, MechanicsBackend, MiePotential, NewtonDamped,
                               RodInteraction, workloads)
from oracle.oracle import OracleSim

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-12, "mixed": 1e-5}
PAIRS = [(11.5, 6.0), (12.0, 5.5), (9.3, 4.7), (7.0, 0.5)]
# en + 1 = 64 is the last integer power and 65 is not one of them (FP64: sixty-four
# rounded factors leave mixed precision less than its 1e-5)
ENDS = [(63.0, 6.0), (64.0, 6.0), (64.0, 63.0)]


def rel_err(a, b):
    return np.linalg.norm(a - b, axis=1).max() / np.linalg.norm(b, axis=1).max()


def spec(dim, side, exponents):
    dom = CartesianCuboid.from_boundaries_and_interaction_range([0.0] * dim, [side] * dim, 2.5)
    return InstanceSpec(dom, MiePotential(1.0, 1.0, 50.0, 2.5, *exponents), NewtonDamped(1.0, 1.0))


def lattice(rng, dim, n):
    """n^dim agents, jittered."""
    x = np.stack(np.meshgrid(*[np.arange(n)] * dim, indexing="ij"), -1).reshape(-1, dim)
    return (x + 0.5) * 2.0 + rng.uniform(-0.4, 0.4, x.shape)


def compare(specs, pos, counts, precision, steps=0, **kw):
    kw = dict(dt=0.001, mechanics_solver_order=2, **kw)
    g, o = MechanicsBackend(specs, precision=precision, **kw), OracleSim(specs, **kw)
    for s in (g, o):
        s.set_agents(pos, None, None, counts)
    assert rel_err(g.compute_forces(), o.compute_forces()) <= TOL[precision]
    if steps:
        g.step(steps)
        o.step(steps)
        assert np.abs(g.get_state()[0] - o.get_state()[0]).max() <= 1e-10
    g.close()
    o.close()


@pytest.mark.parametrize("exponents,precision", [(e, p) for e in PAIRS for p in TOL] + [(e, "fp64") for e in ENDS])
@pytest.mark.parametrize("dim,n", [(2, 3), (2, 40), (3, 9), (3, 40)])
def test_points(dim, n, exponents, precision):
    pos = lattice(np.random.default_rng(n), dim, n)
    compare([spec(dim, 2.0 * n, exponents)], pos, [len(pos)], precision,
            steps=18 if precision == "fp64" and n < 20 else 0)


@pytest.mark.parametrize("precision", sorted(TOL))
@pytest.mark.parametrize("odd_one", [0, 3])
def test_one_instance_of_an_ensemble(odd_one, precision):
    rng = np.random.default_rng(9)
    specs = [spec(2, 2.0 * (6 + k), (11.5, 6.0) if k == odd_one else (12.0, 6.0)) for k in range(5)]
    pos = [lattice(rng, 2, 6 + k) for k in range(5)]
    compare(specs, np.concatenate(pos), [len(x) for x in pos], precision)


@pytest.mark.parametrize("precision", sorted(TOL))
@pytest.mark.parametrize("exponents", PAIRS[:3])
def test_rods(exponents, precision):
    wl = workloads.c3_rods_2d(n=500, seed=4)
    s = wl.instances[0]
    inst = [InstanceSpec(s.domain, RodInteraction(MiePotential(0.4, 0.1, 5.0, 1.5, *exponents)), s.mechanics)]
    compare(inst, wl.pos.reshape(500, -1), [500], precision)
