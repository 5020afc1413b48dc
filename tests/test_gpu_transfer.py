"""Particles to the device and back: what goes up comes down unchanged (wrapped
into the box), as arrays and as records, at counts from one particle to some
slots of the pinned ring and for boxes that share a slot (the counts around
each ring's slots: test_gpu_transfer_rings.py).  Everything is compared bit for
bit with the same arithmetic in numpy."""
import numpy as np
import pytest

from cuco_amd import engine as E
from cuco_amd import ics

pytestmark = pytest.mark.gpu

L = 1000.0


def params(size=L, mesh=32):
    asmth = 1.25 * size / mesh
    return dict(pm_grid=mesh, box_size=size, G=ics.G_INTERNAL, asmth=asmth, rcut=4.5 * asmth,
                soft_h=size / 500)


def outside(rng, n, size):
    """Positions up to two boxes out on either side, some on the faces."""
    pos = (rng.random((n, 3)) * 5.0 - 2.0) * size
    pos[rng.random(n) < 0.1] = 0.0
    pos[rng.random(n) < 0.1] = size
    return pos


def wrapped(pos, size):
    x = pos.copy()
    for _ in range(64):
        x = np.where(x < 0, x + size, x)
    for _ in range(64):
        x = np.where(x >= size, x - size, x)
    return x


def as_records(pos, vel, mass):
    P = np.zeros(pos.shape[0], E.PARTICLE_DTYPE)
    P["Pos"], P["Vel"], P["Mass"] = pos, vel, mass
    return P


@pytest.mark.parametrize("n", [1, 2, 63, 17476, 17477, 32769, 43691, 87382, 300007, 800001])
def test_round_trip(n):
    rng = np.random.default_rng(n)
    pos, vel = outside(rng, n, L), rng.standard_normal((n, 3)) * 300.0
    mass = rng.random(n) + 0.5
    eng = E.Engine(max_particles=n, **params())
    eng.upload(pos, vel, mass)
    p, v = eng.download_particles()
    assert np.array_equal(p, wrapped(pos, L)) and np.array_equal(v, vel)
    P = eng.download_records()
    Q = as_records(wrapped(pos, L), vel, mass)
    assert P.tobytes() == Q.tobytes()
    # Forces come down alike as arrays and in records, at either precision.
    for prec in (E.FP64, E.FP32):
        eng.pmforce_periodic(prec)
        apm = eng.accelerations(pp=False)
        P = eng.download_records()
        assert np.array_equal(P["GravPM"], apm.astype(np.float32))
        assert not P["GravAccel"].any()
        if prec == E.FP32:
            assert np.array_equal(apm, apm.astype(np.float32))
    # Records up: their float positions, wrapped in double.
    R = as_records(outside(rng, n, L), vel, mass)
    eng.upload_records(R)
    p, v = eng.download_particles()
    assert np.array_equal(p, wrapped(R["Pos"].astype(np.float64), L))
    assert np.array_equal(v, R["Vel"].astype(np.float64))
    # The drop-in call gives the record its force and keeps the velocities.
    S = R.copy()
    eng.pmforce_particles(S, E.FP32)
    apm = eng.accelerations(pp=False)
    R["GravPM"] = apm
    assert S.tobytes() == R.tobytes()
    assert np.array_equal(eng.download_particles()[1], v)
    eng.upload(pos, uniform_mass=2.0)
    assert not eng.download_particles()[1].any()
    eng.close()


def test_boxes_that_share_slots():
    sizes, counts = [300.0, 1000.0, 50.0, 700.0], [5, 40000, 1, 100003]
    rng = np.random.default_rng(7)
    pos = np.concatenate([outside(rng, n, s) for n, s in zip(counts, sizes)])
    want = np.concatenate([wrapped(p, s) for p, s in
                           zip(np.split(pos, np.cumsum(counts)[:-1]), sizes)])
    vel = rng.standard_normal(pos.shape)
    ens = E.Ensemble([params(s) for s in sizes], counts)
    ens.upload(pos, vel, uniform_mass=1.0)
    p, v = ens.download_particles()
    assert np.array_equal(p, want) and np.array_equal(v, vel)
    ens.close()


def test_refused_particles_leave_the_handle_as_it_was():
    n = 200001
    rng = np.random.default_rng(3)
    pos, vel = rng.random((n, 3)) * L, rng.standard_normal((n, 3))
    eng = E.Engine(max_particles=n, **params())
    eng.upload(pos, vel, uniform_mass=1.0)
    bad = pos[::-1].copy()
    bad[150000, 1] = np.nan
    bad[199999, 0] = np.inf
    with pytest.raises(E.CucoError, match="non-finite position for particle 150000"):
        eng.upload(bad, vel, uniform_mass=1.0)
    bad[70000, 2] = 1e9
    with pytest.raises(E.CucoError, match="cannot be wrapped"):
        eng.upload(bad, vel, uniform_mass=1.0)
    p, v = eng.download_particles()
    assert np.array_equal(p, pos) and np.array_equal(v, vel)
    with pytest.raises(E.CucoError, match="PP force not computed"):
        eng.accelerations()
    eng.close()
