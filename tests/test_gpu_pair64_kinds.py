"""The FP64 pair force's teams and list (pp64.hip) against the oracle's
sequential loop (gravlist.cpp:216-338), bit for bit -- the sum order is fixed,
so the tolerance is zero.  In small boxes every wave is long against the
evaluation, so dense waves go to teams and the others to the list; the walks
are in test_gpu_pair64_walks.py and test_gpu_pair64_uniform.py.  Cases: dense blobs
across the periodic corner (image pieces on every axis, several batches of
column pieces), sizes around one wave, pairs exactly at rcut on cell edges,
rcut near half the box (per-pair wrapping), and active sets of the integer
timeline from one to all particles."""
import numpy as np
import pytest

from cuco_amd import engine as E
from cuco_amd import ics

from helpers import make_engine, oracle_params

pytestmark = pytest.mark.gpu

BOX = ics.small_box("kinds", 16, 32, 40.0, 31)
MASS = float(BOX.mass)


def blob(rng, n, center, width):
    return np.mod(center + rng.normal(0.0, width, (n, 3)), BOX.L)


def positions(case, rng):
    L, cell = BOX.L, BOX.L / BOX.M
    if case == "corner_blob":
        return np.concatenate([blob(rng, 3000, np.zeros(3), 1.2 * cell),
                               rng.uniform(0, L, (1500, 3))])
    if case.startswith("blob"):
        return blob(rng, int(case[4:]), np.array([0.5, 0.02, 0.98]) * L, 0.8 * cell)
    if case == "two_blobs":
        return np.concatenate([blob(rng, 1700, np.array([0.3, 0.3, 0.3]) * L, 0.7 * cell),
                               blob(rng, 900, np.array([0.3, 0.3, 0.62]) * L, 3.0 * cell),
                               rng.uniform(0, L, (700, 3))])
    if case == "at_rcut":
        # Clusters on cell corners, their partners exactly rcut away along
        # each axis, and one ulp either side.
        base = np.repeat(np.array([[4.0, 9.0, 17.0], [0.0, 31.0, 15.0]]) * cell, 40, axis=0)
        far = []
        for axis in range(3):
            for sign in (-1.0, 1.0):
                for p in base[::8]:
                    q = p.copy()
                    q[axis] = q[axis] + sign * BOX.rcut
                    far += [q, q.copy(), q.copy()]
                    far[-2][axis] = np.nextafter(q[axis], np.inf)
                    far[-1][axis] = np.nextafter(q[axis], -np.inf)
        pos = np.mod(np.concatenate([base, np.array(far)]), L)
        pos[pos >= L] = 0.0
        return pos
    return rng.uniform(0, L, (20000, 3))  # spread


CASES = ["corner_blob", "blob63", "blob64", "blob65", "blob129", "two_blobs", "at_rcut", "spread"]


@pytest.mark.parametrize("masses", ["equal", "unequal"])
@pytest.mark.parametrize("case", CASES)
def test_bit_identical(orc, case, masses):
    rng = np.random.default_rng(500 + CASES.index(case))
    pos = positions(case, rng)
    n = pos.shape[0]
    mass = np.full(n, MASS) if masses == "equal" else MASS * rng.uniform(0.5, 1.5, n)
    eng = make_engine(BOX, capacity=n)
    eng.upload(pos, None, mass)
    eng.gravity_linklist(E.FP64)
    got = eng.accelerations(pm=False)
    ref, pairs = orc.pp_force(oracle_params(BOX), pos, mass)
    assert np.array_equal(got, ref)
    assert eng.count_pairs()[0] == pairs
    eng.close()


def test_bit_identical_when_rcut_nears_half_the_box(orc):
    box = ics.small_box("kinds_wide", 16, 32, 40.0, 31)
    rcut = 14.9 * box.L / box.M  # 2 rcut + 2 cells just below the mesh
    rng = np.random.default_rng(61)
    cell = box.L / box.M
    pos = np.concatenate([np.mod(rng.normal(0.0, 1.0 * cell, (900, 3)), box.L),
                          rng.uniform(0, box.L, (600, 3))])
    mass = MASS * rng.uniform(0.5, 1.5, pos.shape[0])
    kw = box.engine_kwargs()
    kw["rcut"] = rcut
    eng = E.Engine(max_particles=pos.shape[0], **kw)
    eng.upload(pos, None, mass)
    eng.gravity_linklist(E.FP64)
    p = orc.params(box.M, box.L, ics.G_INTERNAL, box.asmth, rcut, box.soft_h)
    ref, _ = orc.pp_force(p, pos, mass)
    assert np.array_equal(eng.accelerations(pm=False), ref)
    eng.close()


def test_active_sets_get_the_whole_evaluations_force(orc):
    """Timeline steps of a clustered box: whatever share is active, an active
    particle's force is the whole evaluation's at the same positions."""
    rng = np.random.default_rng(71)
    pos = positions("two_blobs", rng)
    n = pos.shape[0]
    mass = np.full(n, MASS)
    vel = rng.normal(0.0, 1e-3, (n, 3))
    eng = make_engine(BOX, capacity=n)
    eng.upload(pos, vel, mass)
    eng.timeline_init(time_begin=0.5, time_max=1.0, omega0=ics.OMEGA_M, omega_lambda=ics.OMEGA_L,
                      hubble=ics.HUBBLE_INTERNAL, err_tol_int_accuracy=0.005,
                      max_size_timestep=0.03, min_size_timestep=0.0,
                      softening_halo=BOX.softening, softening_halo_max_phys=BOX.softening)
    shares = set()
    for _ in range(6):
        _, end = eng.timesteps()
        s = eng.timeline_run(E.FP64, max_steps=1)
        active = end == s["ti_current"]
        shares.add(int(active.sum()))
        got = eng.accelerations(pm=False)
        now, _ = eng.download_particles()
        ref, _ = orc.pp_force(oracle_params(BOX), now, mass)
        assert active.any() and np.array_equal(got[active], ref[active])
    assert min(shares) < n == max(shares)  # the first step has every particle
    eng.close()


@pytest.mark.parametrize("mesh", [16, 96, 512])
def test_bit_identical_whatever_the_targets_order(orc, mesh):
    """Target keys two levels below the cells, or one where 32 bits leave no
    more (512); the box's last key shared with inactive targets (16) or not."""
    box = ics.small_box("kinds_order", 16, mesh, 40.0, 31)
    rng = np.random.default_rng(mesh)
    cell = box.L / mesh
    pos = np.concatenate([np.mod(rng.normal(0.0, 1.0 * cell, (2000, 3)), box.L),
                          np.mod(rng.normal(0.999 * box.L, 0.01 * cell, (300, 3)), box.L),
                          rng.uniform(0, box.L, (1000, 3))])
    pos[pos >= box.L] = 0.0
    mass = MASS * rng.uniform(0.5, 1.5, pos.shape[0])
    eng = make_engine(box, capacity=pos.shape[0])
    eng.upload(pos, None, mass)
    eng.gravity_linklist(E.FP64)
    ref, _ = orc.pp_force(oracle_params(box), pos, mass)
    assert np.array_equal(eng.accelerations(pm=False), ref)
    eng.close()
