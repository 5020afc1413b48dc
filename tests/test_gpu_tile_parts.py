"""Long tiles of the FP32 pair kernel, each taken by several waves
(pp32.hip): a dense blob of thousands of particles, alone and across the
periodic corner, for every Morton block size, tiles of 64 and 128, common
and per-particle masses, rcut on and off a table bin edge.  Against the FP64
path with the tolerance of the edge cases (2e-5 of the largest force, plus,
per neighbour closer than 2h, the rounding of a coordinate at the tile's
reach times the softened law's largest slope); the same bits on every
evaluation and, in an ensemble, as a single-box handle's."""
import numpy as np
import pytest
from scipy.spatial import cKDTree

from cuco_amd import engine as E
from cuco_amd import ics

from helpers import make_engine

pytestmark = pytest.mark.gpu

BOX = ics.small_box("parts", 16, 64, 80.0, 51)
MASS = float(BOX.mass)


def blob(center, n, rng):
    cell = BOX.L / BOX.M
    pos = np.concatenate([np.mod(center + rng.normal(0.0, 1.6 * cell, (n, 3)), BOX.L),
                          rng.uniform(0, BOX.L, (3000, 3))])
    pos[pos >= BOX.L] = 0.0
    return pos


def tolerance(pos, ref, mass):
    cell = BOX.L / BOX.M
    unit = max(np.linalg.norm(ref, axis=1).max(), ics.G_INTERNAL * mass.max() / cell ** 2)
    h = BOX.soft_h
    # a tile reaches rcut and a super-block of up to 32 cells from its anchor
    delta = 4 * float(np.spacing(np.float32(BOX.rcut + 32 * cell)))
    per_pair = 10.67 * ics.G_INTERNAL * mass.max() * delta / h ** 3
    tree = cKDTree(pos, boxsize=BOX.L)
    close = tree.query_ball_point(pos, 2 * h, return_length=True) - 1
    return 2e-5 * unit + per_pair * close


@pytest.mark.parametrize("masses", ["equal", "unequal"])
@pytest.mark.parametrize("rcut", [1.0, 0.97])
@pytest.mark.parametrize("place", ["middle", "corner"])
def test_split_tiles_match_fp64(place, rcut, masses):
    rng = np.random.default_rng(7)
    pos = blob(np.full(3, 0.37 if place == "middle" else 0.0) * BOX.L, 12000, rng)
    n = pos.shape[0]
    mass = np.full(n, MASS) if masses == "equal" else MASS * rng.uniform(0.5, 1.5, n)
    kw = BOX.engine_kwargs()
    kw["rcut"] *= rcut
    eng = E.Engine(max_particles=n, **kw)
    eng.upload(pos, None, mass)
    eng.gravity_linklist(E.FP64)
    ref = eng.accelerations(pm=False)
    tol = tolerance(pos, ref, mass)
    for shift in (2, 3, 4):
        for wide in (0, 1):
            print(place, rcut, masses, shift, wide, flush=True)
            eng.set_tuning(shift, 8, pp_wide_tiles=wide)
            eng.gravity_linklist(E.FP32)
            a = eng.accelerations(pm=False)
            err = np.abs(a - ref).max(axis=1)
            assert (err <= tol).all(), (shift, wide, err.max(), int(np.argmax(err - tol)))
            eng.compute_accelerations(E.FP32, False)
            assert np.array_equal(eng.accelerations(pm=False), a)
    eng.close()


def test_split_tiles_keep_their_bits_in_an_ensemble():
    rng = np.random.default_rng(8)
    other = ics.small_box("parts_other", 16, 32, 50.0, 52)
    sets = [(other, rng.uniform(0, other.L, (5000, 3))), (BOX, blob(np.full(3, 0.4) * BOX.L, 9000, rng)),
            (BOX, blob(np.zeros(3), 4000, rng))]
    ens = E.Ensemble([b.engine_kwargs() for b, _ in sets], [len(p) for _, p in sets])
    ens.upload(np.concatenate([p for _, p in sets]), uniform_mass=MASS)
    ens.gravity_linklist(E.FP32)
    got = ens.accelerations(pm=False)
    for k, (box, pos) in enumerate(sets):
        one = make_engine(box, capacity=len(pos))
        one.upload(pos, uniform_mass=MASS)
        one.gravity_linklist(E.FP32)
        assert np.array_equal(got[ens.box_slice(k)], one.accelerations(pm=False)), k
        one.close()
    ens.close()


@pytest.mark.parametrize("masses", ["equal", "unequal"])
@pytest.mark.parametrize("rcut", [1.0, 0.97])
def test_small_launches_keep_the_bits_of_large_ones(rcut, masses):
    """A launch of few tiles takes a tile per workgroup, an ensemble's many
    tiles one per wave: the same candidates, chunks and order of every sum.
    Boxes: a lattice in wide tiles of 2x2x2-cell units, a blob whose tiles are
    split into parts, few particles, a mesh that is not a power of two; the
    last box only makes the ensemble's launch large."""
    rng = np.random.default_rng(9)
    lattice = (np.stack(np.meshgrid(*[np.arange(20)] * 3, indexing="ij"), -1).reshape(-1, 3) + 0.5) / 20
    small = ics.small_box("parts_small", 16, 40, 50.0, 53)
    tiny = ics.small_box("parts_tiny", 4, 16, 20.0, 54)
    many = ics.small_box("parts_many", 16, 64, 80.0, 55)
    sets = [(small, np.mod(lattice * small.L + rng.normal(0, 0.2, (8000, 3)) * small.L / 20, small.L)),
            (BOX, blob(np.full(3, 0.4) * BOX.L, 9000, rng)),
            (tiny, rng.uniform(0, tiny.L, (70, 3))),
            (many, rng.uniform(0, many.L, (190000, 3)))]
    for k, (box, pos) in enumerate(sets):
        pos[pos >= box.L] = 0.0
    mass = [np.full(len(p), MASS) if masses == "equal" else MASS * rng.uniform(0.5, 1.5, len(p))
            for _, p in sets]
    kws = []
    for box, _ in sets:
        kw = box.engine_kwargs()
        kw["rcut"] *= rcut
        kws.append(kw)
    ens = E.Ensemble(kws, [len(p) for _, p in sets])
    ens.upload(np.concatenate([p for _, p in sets]), None, np.concatenate(mass))
    ens.gravity_linklist(E.FP32)
    got = ens.accelerations(pm=False)
    for k, (box, pos) in enumerate(sets[:-1]):
        one = E.Engine(max_particles=len(pos), **kws[k])
        one.upload(pos, None, mass[k])
        one.gravity_linklist(E.FP32)
        assert np.array_equal(got[ens.box_slice(k)], one.accelerations(pm=False)), k
        one.close()
    ens.close()
