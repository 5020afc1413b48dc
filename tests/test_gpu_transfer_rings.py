"""Bitwise round trips through every ring of a handle (transfer.hip): four
slots of 4 KB to 256 KB up to 21845 particles, eight of 512 KB up to 1000000,
sixteen of 2 MB above; counts one below, at and one above a slot, all slots and
one more, for double4 entries up and for positions, FP32 accelerations and
records down; rings that a closed handle leaves to the next one."""
import numpy as np
import pytest

from cuco_amd import engine as E

from test_gpu_transfer import L, as_records, params

pytestmark = pytest.mark.gpu

ENTRIES = {"up": 32, "positions": 24, "floats": 12, "records": 60}


def ring(capacity):
    """Bytes of a slot, and slots."""
    if capacity > 1000000:
        return 2 << 20, 16
    b = 4096
    while b < 12 * capacity and b < 512 << 10:
        b *= 2
    return b, 4 if b < 512 << 10 else 8


def round_trip(eng, n, seed):
    rng = np.random.default_rng(seed)
    pos, vel, mass = rng.random((n, 3)) * L, rng.standard_normal((n, 3)), rng.random(n) + 0.5
    eng.upload(pos, vel, mass)
    p, v = eng.download_particles()
    assert np.array_equal(p, pos) and np.array_equal(v, vel)
    assert eng.download_records().tobytes() == as_records(pos, vel, mass).tobytes()
    eng.pmforce_periodic(E.FP32)
    apm = eng.accelerations(pp=False)
    P = eng.download_records()
    assert apm.any() and np.array_equal(P["GravPM"], apm.astype(np.float32))
    R = as_records(pos, vel, mass)
    eng.upload_records(R)
    p, v = eng.download_particles()
    assert np.array_equal(p, R["Pos"].astype(np.float64) % L)
    assert np.array_equal(v, R["Vel"].astype(np.float64))
    S = R.copy()
    eng.pmforce_particles(S, E.FP32)
    R["GravPM"] = eng.accelerations(pp=False)
    assert S.tobytes() == R.tobytes()


@pytest.mark.parametrize("capacity", [341, 342, 5461, 21845, 21846, 1000000])
def test_counts_around_the_slots(capacity):
    slot, slots = ring(capacity)
    counts = {1, capacity}
    for entry in ENTRIES.values():
        per = slot // entry
        counts |= {per - 1, per, per + 1, slots * per - 1, slots * per, slots * per + 1}
    eng = E.Engine(max_particles=capacity, **params())
    for n in sorted(c for c in counts if 1 <= c <= capacity):
        print(capacity, n, flush=True)
        round_trip(eng, n, n)
    eng.close()


@pytest.mark.parametrize("n", [87382, 559232, 559233, 1000001, 1048576, 1048577, 1398097])
def test_the_ring_of_large_handles(n):
    eng = E.Engine(max_particles=max(n, 1000001), **params())
    round_trip(eng, n, n)
    eng.close()


def test_rings_that_closed_handles_leave():
    keep = E.Engine(max_particles=30000, **params())
    for capacity in (5000, 5000, 300, 30000, 5000, 1000001, 5000):
        eng = E.Engine(max_particles=capacity, **params())
        round_trip(eng, min(capacity, 40000), capacity)
        eng.close()
        round_trip(keep, 30000, capacity)
    keep.close()
