"""The FP64 pair force's walks under a plan (pp64.hip): in a box whose time a
dense cluster takes, waves of a few candidates stay with one target per lane,
and those of a small clump with the wave-uniform walk.  Bit for bit against
the oracle, with whole-cell images and with per-pair wrapping, over active
sets too.  Before each comparison the test makes sure from counts of
neighbours that the plan's costs (in its SIMD cycles) leave those waves there."""
import numpy as np
import pytest
from scipy.spatial import cKDTree

from cuco_amd import engine as E
from cuco_amd import ics

pytestmark = pytest.mark.gpu

UNIFORM, LANE, LIST_TARGET, CHAIN = 345, 830, 2500, 2500


class Case:
    def __init__(self, M, rcut_cells, cluster, clumps, clump, sparse, center, home, seed):
        """cluster particles at center, the others over the box home[0]..home[1]."""
        rng = np.random.default_rng(seed)
        self.M, self.L = M, float(M)  # a cell is 1
        self.rcut = rcut_cells
        lo, hi = np.array(home[0], float), np.array(home[1], float)
        # Clumps further apart than a wave reaches.
        side = np.maximum(1, ((hi - lo) // 24).astype(int))
        at = lo + 0.5 + 24.0 * np.stack(np.unravel_index(np.arange(clumps), side), 1)
        self.pos = np.concatenate([
            center + rng.uniform(-0.4, 0.4, (cluster, 3)),
            np.repeat(at, clump, axis=0) + rng.uniform(-0.2, 0.2, (clumps * clump, 3)),
            lo + rng.random((sparse, 3)) * (hi - lo)])
        self.pos = np.mod(self.pos, self.L)
        self.pos[self.pos >= self.L] = 0.0
        self.mass = rng.uniform(0.5, 1.5, len(self.pos))
        self.cluster, self.in_clumps, self.clump = cluster, clumps * clump, clump
        self.kw = dict(pm_grid=M, box_size=self.L, G=1.0, asmth=rcut_cells / 4.5, rcut=rcut_cells,
                       soft_h=0.05)

    def oracle(self, orc, pos=None):
        p = orc.params(self.M, self.L, 1.0, self.kw["asmth"], self.rcut, self.kw["soft_h"])
        return orc.pp_force(p, self.pos if pos is None else pos, self.mass)[0]

    def check_kinds(self):
        """The cluster's waves against the longest of the others."""
        total = self.cluster // 64 * self.cluster * UNIFORM  # at least: each meets all of it
        tree = cKDTree(self.pos, boxsize=self.L)
        c = self.cluster
        # Whole cells within reach: at most this far; a clump's wave: of its box.
        near = tree.query_ball_point(self.pos[c:], self.rcut + 3.0, return_length=True)
        assert near.max() * CHAIN <= total >> 13
        clumped, sparse = near[:self.in_clumps], near[self.in_clumps:]
        # Some clump's wave: fewer candidates than its lanes' walks would take.
        assert clumped.min() * UNIFORM < self.clump * LANE < 64 * LIST_TARGET
        # Some sparse wave: its own 64 targets cost the uniform walk more.
        assert np.sort(sparse)[64] * LANE < 64 * UNIFORM


CASES = {
    "images": dict(M=128, rcut_cells=5.625, cluster=30000, clumps=30, clump=128, sparse=3000,
                   center=(20.5, 30.5, 64.5), home=((40, 0, 0), (128, 128, 128)), seed=1),
    "across": dict(M=128, rcut_cells=5.625, cluster=30000, clumps=30, clump=128, sparse=3000,
                   center=(0.0, 0.0, 127.9), home=((20, 0, 0), (108, 128, 128)), seed=2),
    # 2 rcut + 2 cells fill the mesh: images by the reference's per-pair tests.
    "wrap": dict(M=16, rcut_cells=7.0, cluster=40000, clumps=1, clump=128, sparse=10,
                 center=(3.5, 3.5, 3.5), home=((10.5, 10.5, 10.5), (13.0, 13.0, 13.0)), seed=3),
}


@pytest.mark.parametrize("case", CASES)
def test_bit_identical(orc, case):
    c = Case(**CASES[case])
    if case != "wrap":
        c.check_kinds()
    eng = E.Engine(max_particles=len(c.pos), **c.kw)
    eng.upload(c.pos, None, c.mass)
    eng.gravity_linklist(E.FP64)
    assert np.array_equal(eng.accelerations(pm=False), c.oracle(orc))
    eng.close()


def test_active_sets(orc):
    c = Case(**dict(CASES["images"], cluster=20000, clump=80))
    c.check_kinds()
    rng = np.random.default_rng(4)
    eng = E.Engine(max_particles=len(c.pos), **c.kw)
    eng.upload(c.pos, rng.normal(0.0, 1e-3, c.pos.shape), c.mass)
    soft = 0.05 / 2.8
    eng.timeline_init(time_begin=0.5, time_max=1.0, omega0=ics.OMEGA_M, omega_lambda=ics.OMEGA_L,
                      hubble=ics.HUBBLE_INTERNAL, err_tol_int_accuracy=0.005,
                      max_size_timestep=0.03, min_size_timestep=0.0, softening_halo=soft,
                      softening_halo_max_phys=soft)
    shares = set()
    for _ in range(3):
        _, end = eng.timesteps()
        s = eng.timeline_run(E.FP64, max_steps=1)
        active = end == s["ti_current"]
        shares.add(int(active.sum()))
        now, _ = eng.download_particles()
        ref = c.oracle(orc, now)
        assert active.any() and np.array_equal(eng.accelerations(pm=False)[active], ref[active])
    eng.close()
    assert len(shares) > 1, shares
