"""Units of the FP32 mesh deposit (pm.hip): listed by one block up to 1024
bricks, by three launches beyond.  An ensemble of 1024 bricks and one of 1032
give every box the mesh force it has alone, bit for bit, with bricks that are
split into several units and empty ones among them; alone it is the FP64
path's to the FP32 mesh tolerance of the edge cases (2e-5 of the largest)."""
import numpy as np
import pytest

from cuco_amd import engine as E
from cuco_amd import ics

from helpers import make_engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("last", [None, 32])
def test_mesh_force_either_side_of_the_switch(last):
    rng = np.random.default_rng(5)
    meshes = [128, 128] + ([last] if last else [])
    sets = []
    for k, mesh in enumerate(meshes):
        box = ics.small_box(f"bricks{k}", 16, mesh, 50.0 + k, 60 + k)
        pos = np.concatenate([np.mod(0.3 * box.L + rng.normal(0, 0.5 * box.L / mesh, (9000, 3)), box.L),
                              rng.uniform(0, box.L, (2000 + k, 3))])
        pos[pos >= box.L] = 0.0
        sets.append((box, pos))
    mass = float(sets[0][0].mass)
    ens = E.Ensemble([b.engine_kwargs() for b, _ in sets], [len(p) for _, p in sets])
    ens.upload(np.concatenate([p for _, p in sets]), uniform_mass=mass)
    ens.pmforce_periodic(E.FP32)
    got = ens.accelerations(pp=False)
    for k, (box, pos) in enumerate(sets):
        one = make_engine(box, capacity=len(pos))
        one.upload(pos, uniform_mass=mass)
        one.pmforce_periodic(E.FP32)
        a = one.accelerations(pp=False)
        assert np.array_equal(got[ens.box_slice(k)], a), k
        one.pmforce_periodic(E.FP64)
        ref = one.accelerations(pp=False)
        assert np.abs(a - ref).max() <= 2e-5 * np.linalg.norm(ref, axis=1).max()
        one.close()
    ens.close()
