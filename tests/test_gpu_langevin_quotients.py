"""The quotients of the Langevin sorting interaction are IEEE divisions for every operand:
isolated FP64 pairs equal the same expressions in numpy bit for bit, so close to contact
that the Gaussian factor is exactly 1, and with attractions that are infinite, that
overflow in the quotient, or that leave the pull below the range of exact remainders."""
import numpy as np
import pytest

from cellular_raza_amd import (CartesianCuboid, CellSpecificInteractionLangevin, InstanceSpec, MechanicsBackend,
                               NewtonDamped)

pytestmark = pytest.mark.gpu

R = 12.0  # contact distance of two cells of radius 6


def pairs(attraction, cutoff, distance):
    """Forces on isolated pairs, and the same in numpy."""
    rng = np.random.default_rng(len(distance))
    m = 9
    grid = (np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3) * 60.0 + 60.0)[:len(distance)]
    u = rng.normal(size=grid.shape)
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    a = grid + rng.uniform(-1.0, 1.0, grid.shape)
    b = a + u * distance[:, None]
    dom = CartesianCuboid.from_boundaries_and_interaction_range([0.0] * 3, [60.0 * (m + 1)] * 3, 30.0)
    pot = CellSpecificInteractionLangevin(cell_radius=R / 2, attraction_rr=attraction, attraction_bb=attraction,
                                          attraction_rb=attraction, repulsion=5.0, cutoff=cutoff)
    g = MechanicsBackend([InstanceSpec(dom, pot, NewtonDamped(1.0, 1.0))], dt=0.01, weighting="physical")
    pos = np.concatenate([a, b])
    g.set_agents(pos, species=np.zeros(len(pos), dtype=np.int32))
    f = g.compute_forces()
    g.close()
    z = np.concatenate([a - b, b - a])
    d2 = np.zeros(len(z))
    for k in range(3):
        d2 = d2 + z[:, k] * z[:, k]
    r = np.sqrt(d2)
    with np.errstate(all="ignore"):
        pull = ((-attraction) * (r - R)) * (cutoff - r)
        sm1 = r / R - 1.0
        gauss = np.where(sm1 < 7.4e-9, 1.0, np.exp(-(sm1 * sm1)))  # 1 - sm1^2 rounds to 1 (numpy's exp may not)
        s = np.where(r <= R, 5.0 * (R - r), np.where(r <= cutoff, (pull / cutoff) * gauss, 0.0))
        return f, -(s[:, None] * (z / r[:, None])), r


@pytest.mark.parametrize("cutoff", [12.5, 20.0, 29.7])
@pytest.mark.parametrize("attraction", [0.015, 1.5, 1e-290, 1e290])
def test_quotients_next_to_contact(attraction, cutoff):
    rng = np.random.default_rng(1)
    f, want, r = pairs(attraction, cutoff, R * (1.0 + rng.uniform(1e-13, 7e-9, 729)))
    assert (r > R).sum() > 1400  # (the factor is exp(-5e-17) there: 1)
    assert np.array_equal(f, want)


@pytest.mark.parametrize("attraction", [np.inf, -np.inf, 1e308, 1e-307])
def test_attractions_at_the_ends_of_the_range(attraction):
    rng = np.random.default_rng(2)
    f, want, r = pairs(attraction, 20.0, rng.uniform(12.5, 19.5, 700))
    if abs(attraction) >= 1e308:
        assert np.isinf(want).any() and not np.isnan(want).any()
    # exp may differ by its last bits; subnormal results are rounded to 4.9e-324 three times
    np.testing.assert_allclose(f, want, rtol=1e-14, atol=3e-323)
