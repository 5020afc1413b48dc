"""The FP64 pair law's square root and divisions (pp64.hip) term by term: boxes
of isolated pairs, each particle's force a single term of its partner's, bit
for bit against the oracle's sqrt and divide.  Separations from far inside the
spline to rcut; masses of random, all-ones and next-to-one mantissas; cubed
distances r2 r next to a power of two on either side, where the reciprocal's
error is largest against its spacing."""
import numpy as np
import pytest

from cuco_amd import engine as E
from cuco_amd import ics

pytestmark = pytest.mark.gpu

M, L = 256, 256.0
RCUT, SOFT = 5.625, 0.05


def pairs(cells, r, rng):
    """Pairs of separation r in random directions, one per block of `cells`
    cells a side (further than rcut from each other)."""
    side = int(M // cells)
    n = min(side ** 3, len(r))
    c = np.stack(np.unravel_index(np.arange(n), (side,) * 3), 1) * float(cells) + 0.3
    d = rng.standard_normal((n, 3))
    d *= (r[:n] / np.linalg.norm(d, axis=1))[:, None]
    # half the separation on either side of a point that leaves rcut to the
    # next block's pair
    mid = c + 0.5 * (RCUT if cells > 9 else 0.7) + rng.random((n, 3)) * 0.05
    pos = np.mod(np.concatenate([mid - 0.5 * d, mid + 0.5 * d]), L)
    pos[pos >= L] = 0.0
    return pos


def masses(n, rng):
    m = rng.uniform(1.0, 2.0, n)
    m[rng.random(n) < 0.2] = 2.0 - 2.0 ** -52
    m[rng.random(n) < 0.2] = 1.0 + 2.0 ** -52
    m[rng.random(n) < 0.1] = 1.0
    return m


def check(orc, pos, mass):
    eng = E.Engine(max_particles=len(pos), pm_grid=M, box_size=L, G=1.0, asmth=1.25, rcut=RCUT,
                   soft_h=SOFT)
    eng.upload(pos, None, mass)
    eng.gravity_linklist(E.FP64)
    got = eng.accelerations(pm=False)
    eng.close()
    p = orc.params(M, L, 1.0, 1.25, RCUT, SOFT)
    ref, _ = orc.pp_force(p, pos, mass)
    assert (ref != 0).any(axis=1).mean() > 0.95
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("seed", range(6))
def test_random_separations(orc, seed):
    rng = np.random.default_rng(seed)
    pos = pairs(7, np.geomspace(1e-4, 0.6, 40000), rng)
    check(orc, pos, masses(len(pos), rng))


@pytest.mark.parametrize("seed", range(6))
def test_up_to_the_cut(orc, seed):
    rng = np.random.default_rng(10 + seed)
    pos = pairs(12, rng.uniform(0.5, 5.6, 9000), rng)
    check(orc, pos, masses(len(pos), rng))


@pytest.mark.parametrize("seed", range(6))
def test_cubes_next_to_a_power_of_two(orc, seed):
    rng = np.random.default_rng(20 + seed)
    n = 40000
    k = rng.integers(-12, -2, n)
    off = rng.choice([-1.0, 1.0], n) * 2.0 ** -rng.integers(20, 52, n).astype(float)
    pos = pairs(7, np.cbrt(2.0 ** k * (1.0 + off)), rng)
    check(orc, pos, masses(len(pos), rng))
