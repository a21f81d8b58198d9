"""FP64 pair forces are the reference's operations with their IEEE roundings: isolated
pairs, whose only force is one interaction, equal the same expressions in numpy bit for
bit (sqrt and division are correctly rounded there; integer powers by the same
products).  Distances over the whole range, and next to zero where the squared distance
leaves the range of the shared reciprocal."""
import numpy as np
import pytest

from cellular_raza_amd import (BoundLennardJones, CartesianCuboid, CellSpecificInteraction, InstanceSpec,
                               MechanicsBackend, MiePotential, NewtonDamped)

pytestmark = pytest.mark.gpu


def ipow(x, e):
    r, b = np.ones_like(x), x
    while e:
        if e & 1:
            r = r * b
        b, e = b * b, e >> 1
    return r


def mie(z, r, dirs):
    sigma = np.power(6.0 / 12.0, 1.0 / 6.0) * 2.0
    c = 12.0 / 6.0 * np.power(12.0 / 6.0, 6.0 / 6.0)
    sr = sigma / r
    part = 12.0 / sigma * ipow(sr, 13) - 6.0 / sigma * ipow(sr, 7)
    return dirs * np.fmin(c * 1.5 * part, 1e3)[:, None]


def blj(z, r, dirs):
    sr = 1.2 / r
    val = 4.0 * 0.7 / r * (12.0 * ipow(sr, 11) - 6.0 * ipow(sr, 5))
    return -dirs * np.fmin(np.inf / r, val)[:, None]


def sorting(z, r, dirs):
    mrd = 0.3162277660168379
    rr = np.where(r < 0.9 * mrd, 0.9 * mrd, r)
    inv = 1.0 / (rr / 1.8)
    inv2, bound = inv * inv, 4.0 + inv
    s = 2.0 * np.fmax(np.fmin(inv2 - inv2 * inv2, bound), -bound)
    cut = np.where(1.35 * 1.8 - rr >= 0.0, 1.0, 0.0)[:, None]
    return (dirs * np.fmin(s, 0.0)[:, None]) * cut + (dirs * np.fmax(s, 0.0)[:, None]) * cut


CASES = {
    "mie": (MiePotential(1.0, 1.5, 1e3, 2.5, 12.0, 6.0), mie),
    "blj": (BoundLennardJones(0.7, 1.2, np.inf, 2.5), blj),
    "sorting": (CellSpecificInteraction(0.9, 2.0, 1.35), sorting),
}


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("name", sorted(CASES))
def test_isolated_pairs_equal_ieee_arithmetic(name, dim):
    pot, expected = CASES[name]
    m = 24 if dim == 3 else 120  # pairs per axis, too far apart to interact
    rng = np.random.default_rng(dim)
    grid = np.stack(np.meshgrid(*[np.arange(m)] * dim, indexing="ij"), -1).reshape(-1, dim) * 10.0 + 10.0
    u = rng.normal(size=grid.shape)
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    r = rng.uniform(0.3, 2.42, len(grid))
    a = grid + rng.uniform(-1.0, 1.0, grid.shape)
    b = a + u * r[:, None]
    b[:40] = a[:40] + u[:40] * 10.0 ** -rng.uniform(1, 14, (40, 1))  # close pairs
    a[40], b[40] = 10.0, 10.0  # a squared distance below 2^-900, apart from every other pair
    a[40, 0], b[40, 0] = 1e-140, 3e-140
    dom = CartesianCuboid.from_boundaries_and_interaction_range([0.0] * dim, [10.0 * (m + 1)] * dim, 2.5)
    g = MechanicsBackend([InstanceSpec(dom, pot, NewtonDamped(1.0, 1.0))], dt=0.01, weighting="physical")
    pos = np.concatenate([a, b])
    g.set_agents(pos, species=np.zeros(len(pos), dtype=np.int32))
    f = g.compute_forces()
    z = np.concatenate([a - b, b - a])
    d2 = np.zeros(len(z))
    for k in range(dim):
        d2 = d2 + z[:, k] * z[:, k]
    with np.errstate(all="ignore"):
        d = np.sqrt(d2)
        want = expected(z, d, z / d[:, None])
    assert np.array_equal(f, want, equal_nan=True)  # (1e-140 apart: inf * 0)
    g.close()
