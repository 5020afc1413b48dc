"""The work a user of the engine has it do, as cases that can be timed.

Every case goes through the Python binding of the C ABI (``cuco_amd.engine``)
the way a simulation or analysis program does.  The kinds:

* ``forces``   -- one complete force evaluation of resident particles (keys,
                  sort, cell table, pair force, mesh force) and the
                  accelerations read back, as a program with its own
                  integrator does every step.
* ``mesh``     -- the long-range force alone, read back.
* ``short``    -- a short run from initial conditions: upload, first forces,
                  KDK steps, final snapshot records.
* ``steps``    -- KDK steps of a resident box, one graph per step, then the
                  particles read back; the state goes on from pass to pass.
* ``ensemble`` -- the same for many boxes of mixed sizes in one handle.
* ``timeline`` -- the reference's integrator: individual power-of-two steps.
* ``records``  -- the drop-in calls on a caller's PARTICLE array.
* ``sort``     -- the key/value radix sort on device arrays.
* ``fft``      -- the 3D real FFT on device arrays, forward and back.

Sizes are those of the package's workloads (32^3 particles on a 64^3 mesh,
128^3 on 256^3, 256^3 on 512^3, ensembles of 32^3..96^3) and ragged ones
between them.  Particles are the same two kinds: a displaced lattice (early
times, nearly uniform) and NFW halos over a uniform background (late times,
strongly clustered).
"""
import ctypes as C
import math

import numpy as np
import torch

from cuco_amd import engine as E
from cuco_amd import ics

DEV = "cuda:0"
SPACING = 1953.125  # kpc/h: 250 Mpc/h over 128 particles
PREC = {"fp32": E.FP32, "fp64": E.FP64}

# Meshes of the draws: register-FFT sizes and the other even products of
# 2, 3 and 5.
MESHES = [32, 36, 40, 48, 50, 60, 64, 72, 80, 90, 96, 100, 108, 120, 128, 144, 150, 160,
          180, 192, 200, 216, 240, 250, 256]


# ------------------------------------------------------------------ cases
def listed():
    return [
        # The smallest box of the package: latency and launches are what a
        # parameter scan or a test run of this size feels.
        dict(name="forces_32_fp32", kind="forces", n=32768, mesh=64, particles="lattice",
             masses="equal", precision="fp32"),
        # A whole short run of that box: initial conditions to snapshot.
        dict(name="short_32_fp32", kind="short", n=32768, mesh=64, particles="lattice",
             masses="equal", precision="fp32", steps=10),
        # A ragged clustered box with a mass per particle (a zoom or a
        # multi-species set-up) on a mesh of mixed factors, plain path.
        dict(name="forces_ragged_fp64", kind="forces", n=100003, mesh=90, particles="halos",
             masses="unequal", precision="fp64"),
        # The same kind of box, larger, on the fast path.
        dict(name="forces_ragged_fp32", kind="forces", n=300007, mesh=150, particles="halos",
             masses="unequal", precision="fp32"),
        # The ordinary production box, fast path and plain path.
        dict(name="forces_128_fp32", kind="forces", n=2097152, mesh=256, particles="halos",
             masses="equal", precision="fp32"),
        dict(name="forces_128_fp64", kind="forces", n=2097152, mesh=256, particles="halos",
             masses="equal", precision="fp64"),
        # The largest: resident steps of the headline box, with the tuning
        # the autotuner settles on there.
        dict(name="steps_256_fp32", kind="steps", n=16777216, mesh=512, particles="halos",
             masses="equal", precision="fp32", steps=12, tuned=True),
        # Many small boxes advanced together (covariance or emulator runs).
        dict(name="ensemble_24_fp32", kind="ensemble", boxes=24, smallest=32, largest=96,
             precision="fp32", steps=16),
        # The reference's own integrator on a clustered box.
        dict(name="timeline_64_fp64", kind="timeline", n=262144, mesh=128, particles="halos",
             masses="equal", precision="fp64", steps=8),
        # The reference's two force calls on a program's P[] array, swapped
        # in unchanged.
        dict(name="records_128_fp32", kind="records", n=2097152, mesh=256, particles="halos",
             masses="equal", precision="fp32"),
        # Sorting particles by cell key, and a spectrum of a density mesh, on
        # a program's own device arrays.
        dict(name="sort_4m", kind="sort", n=4194301, bits=27),
        dict(name="fft_256_fp32", kind="fft", mesh=256, precision="fp32"),
    ]


def _near_mesh(rng, n):
    """A mesh of about two cells per particle spacing."""
    want = 2.0 * n ** (1.0 / 3.0) * rng.uniform(0.85, 1.15)
    return min(MESHES, key=lambda m: abs(math.log(m / want)))


def draw(rng):
    kind = rng.choice(["forces", "forces", "forces", "mesh", "short", "steps", "ensemble",
                       "records", "sort", "fft", "timeline"])

    def logsize(lo, hi):
        return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))

    particles = rng.choice(["lattice", "halos"])
    masses = rng.choice(["equal", "equal", "unequal"])
    precision = rng.choice(["fp32", "fp32", "fp64"])
    if kind == "ensemble":
        return dict(kind=kind, boxes=rng.randint(2, 24), smallest=32,
                    largest=rng.choice([48, 64, 96]), precision="fp32",
                    steps=rng.randint(1, 5))
    if kind == "sort":
        return dict(kind=kind, n=logsize(1000, 1 << 24), bits=rng.choice([12, 18, 24, 27, 32]))
    if kind == "fft":
        return dict(kind=kind, mesh=rng.choice(MESHES), precision=precision)
    if kind == "timeline":
        n = logsize(20000, 300000)
        return dict(kind=kind, n=n, mesh=_near_mesh(rng, n), particles="halos", masses="equal",
                    precision="fp64", steps=rng.randint(2, 10))
    n = logsize(20000, 2200000)
    case = dict(kind=kind, n=n, mesh=_near_mesh(rng, n), particles=particles, masses=masses,
                precision=precision)
    if kind in ("short", "steps"):
        case["n"] = n = min(n, 400000) if precision == "fp64" else n
        case["mesh"] = _near_mesh(rng, n)
        case["steps"] = rng.randint(2, 10)
    if kind == "steps":
        case["tuned"] = precision == "fp32" and rng.random() < 0.5
    return case


# ------------------------------------------------------------------ inputs
def _box(n, mesh):
    """Parameters of a box of n particles at the common mean density."""
    return ics.Box("case", 1, mesh, SPACING * n ** (1.0 / 3.0), 0, "halos")


def _params(n, mesh):
    b = _box(n, mesh)
    soft_h = 2.8 * SPACING / 30.0
    return dict(pm_grid=mesh, box_size=b.L, G=ics.G_INTERNAL, asmth=b.asmth, rcut=b.rcut,
                soft_h=soft_h)


def _lattice(n, L, gen):
    """n particles of a lattice displaced by a smooth random field; the
    lattice is the smallest cube that holds n, its last sites left empty."""
    side = math.ceil(round(n ** (1.0 / 3.0), 9))
    white = torch.randn((side, side, side), generator=gen, device=DEV, dtype=torch.float64)
    wk = torch.fft.rfftn(white)
    k1 = torch.fft.fftfreq(side, d=1.0 / side, device=DEV, dtype=torch.float64)
    kz = torch.fft.rfftfreq(side, d=1.0 / side, device=DEV, dtype=torch.float64)
    K = torch.meshgrid(k1, k1, kz, indexing="ij")
    k2 = K[0] ** 2 + K[1] ** 2 + K[2] ** 2
    k2[0, 0, 0] = 1.0
    delta = wk / torch.sqrt(k2)
    delta[0, 0, 0] = 0.0
    psi = torch.stack([torch.fft.irfftn(1j * k / k2 * delta, s=(side,) * 3).reshape(-1)
                       for k in K], dim=1)
    step = L / side
    psi *= 0.2 * step / torch.sqrt((psi ** 2).sum(1).mean())
    i = torch.arange(n, device=DEV)
    q = torch.stack([i // (side * side), (i // side) % side, i % side], dim=1)
    pos = torch.remainder((q.double() + 0.5) * step + psi[:n], L)
    a = 0.02
    vel = a * a * ics.hubble_a(a) * ics.growth_rate(a) * psi[:n]
    return pos, vel


def _halos(n, L, gen, mass):
    """Half the particles uniform, half in NFW halos (dN/dM ~ M^-1.9 over two
    decades, c = 8, 200 times the mean density), isotropic velocities."""
    n_in = n // 2
    nh = max(8, n // 8000)
    u = torch.rand(nh, generator=gen, device=DEV, dtype=torch.float64)
    m = (1.0 + u * (100.0 ** -0.9 - 1.0)) ** (-1.0 / 0.9)
    edges = torch.round(torch.cumsum(m, 0) / m.sum() * n_in).long()
    counts = torch.diff(edges, prepend=edges.new_zeros(1))
    host = torch.repeat_interleave(torch.arange(nh, device=DEV), counts, output_size=n_in)
    c = counts.clamp(min=1).double()
    r200 = (3.0 * c * L ** 3 / (800.0 * math.pi * n)) ** (1.0 / 3.0)
    v200 = torch.sqrt(ics.G_INTERNAL * c * mass / r200)
    conc = 8.0
    xs = torch.cat([torch.zeros(1, device=DEV, dtype=torch.float64),
                    torch.logspace(-6, math.log10(conc), 20000, device=DEV,
                                   dtype=torch.float64)])
    ms = torch.log1p(xs) - xs / (1.0 + xs)
    w = torch.rand(n_in, generator=gen, device=DEV, dtype=torch.float64) * ms[-1]
    hi = torch.searchsorted(ms, w).clamp(1, xs.numel() - 1)
    t = (w - ms[hi - 1]) / (ms[hi] - ms[hi - 1])
    x = xs[hi - 1] + t * (xs[hi] - xs[hi - 1])
    d = torch.randn((n_in, 3), generator=gen, device=DEV, dtype=torch.float64)
    d /= torch.linalg.vector_norm(d, dim=1, keepdim=True)
    centers = torch.rand((nh, 3), generator=gen, device=DEV, dtype=torch.float64) * L
    inside = centers[host] + (x * r200[host] / conc)[:, None] * d
    outside = torch.rand((n - n_in, 3), generator=gen, device=DEV, dtype=torch.float64) * L
    pos = torch.remainder(torch.cat([inside, outside]), L)
    vel = torch.zeros_like(pos)
    vel[:n_in] = torch.randn((n_in, 3), generator=gen, device=DEV, dtype=torch.float64) * (
        v200[host] * 0.5 / math.sqrt(2.0))[:, None]
    return pos, vel


def _particles(case, seed):
    """Positions, internal velocities and masses (None: all equal), on the GPU."""
    n, b = case["n"], _box(case["n"], case["mesh"])
    gen = torch.Generator(device=DEV).manual_seed(seed * 2654435761 % (1 << 40) + 17)
    unit = _mass()
    make = _lattice if case["particles"] == "lattice" else _halos
    pos, vel = make(n, b.L, gen) if make is _lattice else make(n, b.L, gen, unit)
    pos = torch.where(pos >= b.L, pos - b.L, pos)
    mass = None
    if case["masses"] == "unequal":
        mass = unit * (0.5 + torch.rand(n, generator=gen, device=DEV, dtype=torch.float64))
    return pos, vel, mass


def _mass():
    rho = 3 * ics.HUBBLE_INTERNAL ** 2 / (8 * math.pi * ics.G_INTERNAL)
    return ics.OMEGA_M * rho * SPACING ** 3


def _factors(a, span, steps):
    """KDK factors of `steps` steps over the relative span of a at a."""
    d, k = E.init_drift_table(a, a * 1.5, ics.OMEGA_M, ics.OMEGA_L, ics.HUBBLE_INTERNAL)
    return E.kdk_factors(d, k, a, a * 1.5, a, a * (1.0 + span), steps)


def _host(t):
    return None if t is None else t.cpu().numpy()


def _start_a(case):
    return 0.02 if case.get("particles", "lattice") == "lattice" else 0.5


def prepare(case, seed):
    kind = case["kind"]
    if kind == "sort":
        gen = torch.Generator(device=DEV).manual_seed(seed + 1)
        keys = torch.randint(0, 1 << case["bits"], (case["n"],), generator=gen, device=DEV,
                             dtype=torch.int64).to(torch.int32)
        vals = torch.arange(case["n"], device=DEV, dtype=torch.int32)
        return dict(case=case, keys=keys, vals=vals)
    if kind == "fft":
        gen = torch.Generator(device=DEV).manual_seed(seed + 2)
        M = case["mesh"]
        dt = torch.float32 if case["precision"] == "fp32" else torch.float64
        field = torch.rand((M, M, M), generator=gen, device=DEV, dtype=dt) * 2.0
        return dict(case=case, field=field)
    prec = PREC[case["precision"]]
    if kind == "ensemble":
        return _prepare_ensemble(case, seed)
    pos, vel, mass = (_host(t) for t in _particles(case, seed))
    eng = E.Engine(max_particles=case["n"], **_params(case["n"], case["mesh"]))
    st = dict(case=case, engine=eng, precision=prec)
    if kind == "short":
        st.update(pos=pos, vel=vel, mass=mass, factors=_factors(_start_a(case), 0.1, case["steps"]))
        return st
    if kind == "records":
        P = np.zeros(case["n"], E.PARTICLE_DTYPE)
        P["Pos"], P["Vel"] = pos, vel
        P["Mass"] = _mass() if mass is None else mass
        st["P"] = P
        return st
    if mass is None:
        eng.upload(pos, vel, uniform_mass=_mass())
    else:
        eng.upload(pos, vel, mass)
    if kind == "steps":
        if case["tuned"]:
            # What Engine.autotune picks on a large clustered box.
            eng.set_tuning(3, 4, pm_overlap=1, pp_symmetric=1, pp_wide_tiles=1)
        # Steps far below the crossing time of a halo core, as the innermost
        # steps of a run are: the box stays what it is over many passes.
        st["factors"] = _factors(_start_a(case), 2e-5, case["steps"])
        eng.compute_accelerations(prec, True)
        eng.synchronize()
    if kind == "timeline":
        a = _start_a(case)
        st["timeline"] = dict(
            time_begin=a, time_max=2.0 * a, omega0=ics.OMEGA_M, omega_lambda=ics.OMEGA_L,
            hubble=ics.HUBBLE_INTERNAL, err_tol_int_accuracy=0.025, max_size_timestep=1e-3,
            min_size_timestep=0.0, softening_halo=SPACING / 30.0,
            softening_halo_max_phys=SPACING / 30.0)
    return st


def _prepare_ensemble(case, seed):
    rng = np.random.default_rng(seed)
    choices = [s for s in (32, 48, 64, 80, 96) if case["smallest"] <= s <= case["largest"]]
    # The boxes are part of the case; their particles come from the seed.
    sides = np.random.default_rng(4004).choice(choices, size=case["boxes"])
    boxes, pos, vel = [], [], []
    for side in sides:
        side = int(side)
        one = dict(n=side ** 3, mesh=2 * side, particles="lattice", masses="equal")
        p, v, _ = _particles(one, int(rng.integers(1 << 30)))
        boxes.append(_params(side ** 3, 2 * side))
        pos.append(p)
        vel.append(v)
    counts = [p.shape[0] for p in pos]
    ens = E.Ensemble(boxes, counts)
    ens.upload(_host(torch.cat(pos)), _host(torch.cat(vel)), uniform_mass=_mass())
    prec = PREC[case["precision"]]
    ens.compute_accelerations(prec, True)
    ens.synchronize()
    return dict(case=case, engine=ens, precision=prec, factors=_factors(0.02, 2e-5, case["steps"]))


# ------------------------------------------------------------------ passes
def _own(case, *arrays):
    """The arrays at the precision the path computes in: a program on the
    FP32 path keeps what it reads back in FP32."""
    if case["precision"] == "fp32":
        return tuple(a.astype(np.float32) for a in arrays)
    return arrays


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _ok(status):
    if status:
        raise E.CucoError(status, "case", E.lib().cuco_last_error().decode())


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "sort":
        keys, vals = state["keys"].clone(), state["vals"].clone()
        _ok(E.lib().cuco_radix_sort(_ptr(keys), _ptr(vals), case["n"], case["bits"]))
        return keys, vals
    if kind == "fft":
        M, f = case["mesh"], state["field"]
        prec = PREC[case["precision"]]
        ct = torch.complex64 if case["precision"] == "fp32" else torch.complex128
        spec = torch.empty((M, M, M // 2 + 1), dtype=ct, device=DEV)
        _ok(E.lib().cuco_fft3d_r2c(M, prec, _ptr(f), _ptr(spec)))
        work = spec * (1.0 / M ** 3)
        back = torch.empty_like(f)
        _ok(E.lib().cuco_fft3d_c2r(M, prec, _ptr(work), _ptr(back)))
        return spec, back
    eng, prec = state["engine"], state["precision"]
    if kind == "forces":
        eng.compute_accelerations(prec, True)
        return _own(case, *eng.accelerations())
    if kind == "mesh":
        eng.pmforce_periodic(prec)
        return _own(case, eng.accelerations(pp=False))
    if kind == "short":
        if state["mass"] is None:
            eng.upload(state["pos"], state["vel"], uniform_mass=_mass())
        else:
            eng.upload(state["pos"], state["vel"], state["mass"])
        eng.compute_accelerations(prec, True)
        eng.kdk_steps(state["factors"], prec, use_graph=True)
        P = eng.download_records()
        return P["Pos"], P["Vel"], P["GravAccel"], P["GravPM"]
    if kind in ("steps", "ensemble"):
        eng.kdk_steps(state["factors"], prec, use_graph=True)
        return eng.download_particles()  # the integrator's state is FP64 on either path
    if kind == "timeline":
        eng.timeline_init(**state["timeline"])
        s = eng.timeline_run(prec, max_steps=case["steps"])
        pos, vel = eng.download_particles()
        return pos, vel, s["ti_current"], s["active"]
    if kind == "records":
        eng.pmforce_particles(state["P"], prec)
        eng.gravity_particles(state["P"], prec)
        return state["P"]["GravAccel"], state["P"]["GravPM"]
    raise ValueError(kind)


# ------------------------------------------------------------------ work
def _pair_flops(case):
    """30 flops per ordered pair inside rcut: 93 neighbours per particle in a
    nearly uniform box, about 7000 in a halo box (both at 8 mesh cells per
    particle; the neighbourhood scales with the mesh cell's volume)."""
    per = 93.0 if case["particles"] == "lattice" else 7000.0
    return 30.0 * per * case["n"] * (8.0 * case["n"] / case["mesh"] ** 3)


def _mesh_flops(n, mesh):
    m3 = float(mesh) ** 3
    return 2 * 2.5 * m3 * math.log2(m3) + 150.0 * n


def work(case):
    kind = case["kind"]
    if kind == "sort":
        return dict(bytes=16.0 * case["n"], flops=0.0)
    word = 8.0 if case["precision"] == "fp64" else 4.0
    if kind == "fft":
        m3 = float(case["mesh"]) ** 3
        return dict(bytes=4.0 * word * m3, flops=2 * 2.5 * m3 * math.log2(m3))
    if kind == "ensemble":
        choices = [s for s in (32, 48, 64, 80, 96) if case["smallest"] <= s <= case["largest"]]
        sides = [int(s) for s in np.random.default_rng(4004).choice(choices, size=case["boxes"])]
        n = float(sum(s ** 3 for s in sides))
        fl = sum(30.0 * 93.0 * s ** 3 + _mesh_flops(s ** 3, 2 * s) for s in sides)
        return dict(bytes=96.0 * n, flops=case["steps"] * fl)
    n = float(case["n"])
    evals = {"forces": 1, "mesh": 0, "short": case.get("steps", 0) + 1,
             "steps": case.get("steps", 0), "timeline": case.get("steps", 0), "records": 1}[kind]
    flops = evals * _pair_flops(case) + max(evals, 1) * _mesh_flops(n, case["mesh"])
    per = {"forces": 32 + 6 * word, "mesh": 32 + 3 * word, "short": 56 + 60, "steps": 96,
           "timeline": 96, "records": 2 * (16 + 12)}[kind]
    return dict(bytes=per * n, flops=flops)


# ------------------------------------------------------------------ 64-bit results
def _mesh_force(pos, mass, p):
    """CIC density, Green's function, 4-point gradient and CIC gather."""
    M, L = p["pm_grid"], p["box_size"]
    u = pos * (M / L)
    cell = torch.clamp(u.long(), max=M - 1)
    d = u - cell
    rho = torch.zeros(M ** 3, device=DEV, dtype=torch.float64)
    corners = []
    for c in range(8):
        o = torch.tensor([c >> 2, (c >> 1) & 1, c & 1], device=DEV)
        w = torch.where(o.bool(), d, 1.0 - d).prod(1)
        i = (cell + o) % M
        corners.append(((i[:, 0] * M + i[:, 1]) * M + i[:, 2], w))
        rho.index_add_(0, corners[-1][0], w * mass)
    k = torch.fft.fftfreq(M, d=1.0 / M, device=DEV, dtype=torch.float64).abs()
    one = torch.where(k > 0, (torch.sinc(k / M)) ** -4, torch.ones_like(k))
    one = one * torch.exp(-(k ** 2) * (2.0 * math.pi * p["asmth"] / L) ** 2)
    kz = k[: M // 2 + 1]
    k2 = k[:, None, None] ** 2 + k[None, :, None] ** 2 + kz[None, None, :] ** 2
    k2[0, 0, 0] = 1.0
    green = -one[:, None, None] * one[None, :, None] * one[: M // 2 + 1][None, None, :] / k2
    green[0, 0, 0] = 0.0
    phi = torch.fft.irfftn(torch.fft.rfftn(rho.view(M, M, M)) * green, s=(M, M, M)) * M ** 3
    fac = p["G"] / (math.pi * L) * M / (2.0 * L)
    out = []
    for ax in range(3):
        g = (4.0 / 3.0) * (torch.roll(phi, 1, ax) - torch.roll(phi, -1, ax)) - (1.0 / 6.0) * (
            torch.roll(phi, 2, ax) - torch.roll(phi, -2, ax))
        g = (fac * g).reshape(-1)
        out.append(sum(g[i] * w for i, w in corners))
    return torch.stack(out, 1)


def _pair_force(pos, mass, p):
    """The short-range law (stepped erfc table, spline softening with the
    reference's constants, gravlist.cpp:307-316) over all
    pairs inside rcut, by cells of at least rcut / 2."""
    L, G, rcut, h = p["box_size"], p["G"], p["rcut"], p["soft_h"]
    u = 3.0 / 1000 * (torch.arange(1000, device=DEV, dtype=torch.float64) + 0.5)
    table = (torch.erfc(u) + 2.0 * u / math.sqrt(math.pi) * torch.exp(-u * u)).float().double()
    asmthfac = 0.5 / p["asmth"] * (1000 / 3.0)
    n = pos.shape[0]
    m = max(1, int(math.floor(L / (0.5 * rcut))))
    cell = torch.clamp((pos * (m / L)).long(), max=m - 1)
    key = (cell[:, 0] * m + cell[:, 1]) * m + cell[:, 2]
    key, order = torch.sort(key, stable=True)
    sp, sm, sc = pos[order], mass[order], cell[order]
    start = torch.searchsorted(key, torch.arange(m ** 3 + 1, device=DEV))
    acc = torch.zeros((n, 3), device=DEV, dtype=torch.float64)
    offs = range(-2, 3) if m >= 5 else range(m)
    todo = [(a, b, c) for a in offs for b in offs for c in offs]
    me = torch.arange(n, device=DEV)
    for off in todo:
        q = (sc + torch.tensor(off, device=DEV)) % m
        kq = (q[:, 0] * m + q[:, 1]) * m + q[:, 2]
        first, cnt = start[kq], start[kq + 1] - start[kq]
        total = torch.cumsum(cnt, 0)
        t0 = 0
        while t0 < n:
            done = int(total[t0 - 1]) if t0 else 0
            t1 = max(t0 + 1, int(torch.searchsorted(total, done + 20_000_000)))
            t1 = min(t1, n)
            c = cnt[t0:t1]
            i = torch.repeat_interleave(me[t0:t1], c)
            if i.numel():
                base = torch.cumsum(c, 0) - c
                j = (torch.arange(i.numel(), device=DEV) -
                     torch.repeat_interleave(base - first[t0:t1], c))
                d = sp[j] - sp[i]
                d = d - L * torch.round(d / L)
                r2 = (d * d).sum(1)
                near = torch.nonzero((r2 <= rcut * rcut) & (i != j)).squeeze(1)
                i, j, d, r = i[near], j[near], d[near], torch.sqrt(r2[near])
                x = r / h
                w = torch.where(
                    r >= h, 1.0 / r ** 3,
                    torch.where(x < 0.5, (10.66667 + x * x * (32.0 * x - 38.4)) / h ** 3,
                                (21.33333 - 48.0 * x + 38.4 * x * x -
                                 10.66667 * x ** 3 - 0.06667 / x ** 3) / h ** 3))
                bin_ = (asmthfac * r).long()
                f = torch.where(bin_ < 1000, table[torch.clamp(bin_, max=999)],
                                torch.zeros_like(r))
                f = torch.where(r > 0, G * sm[j] * w * f, torch.zeros_like(r))
                acc.index_add_(0, i, d * f[:, None])
            t0 = t1
    out = torch.empty_like(acc)
    out[order] = acc
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "fft":
        field = prepare(case, seed)["field"].double()
        return torch.fft.rfftn(field), field
    if kind not in ("forces", "mesh", "records", "short"):
        return None
    if kind == "short" and case["n"] * case["steps"] > 400000:
        return None
    pos, vel, mass = _particles(case, seed)
    p = _params(case["n"], case["mesh"])
    if mass is None:
        mass = torch.full((case["n"],), _mass(), device=DEV, dtype=torch.float64)
    if kind == "records":  # the calls see the record's float positions
        pos, mass = pos.float().double(), mass.float().double()
        pos = torch.remainder(pos, p["box_size"])
    pairs = case["n"] <= (400000 if case["particles"] == "halos" else 2000000)
    if kind == "short":
        def forces():
            return _pair_force(pos, mass, p), _mesh_force(pos, mass, p)
        app, apm = forces()
        for k1, dr, k2 in _factors(_start_a(case), 0.1, case["steps"]):
            vel = vel + (app + apm) * float(k1)
            pos = torch.remainder(pos + vel * float(dr), p["box_size"])
            app, apm = forces()
            vel = vel + (app + apm) * float(k2)
        return pos, vel, app, apm
    apm = _mesh_force(pos, mass, p)
    if kind == "mesh":
        return (apm,)
    return (_pair_force(pos, mass, p) if pairs else None), apm
