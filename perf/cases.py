"""The work that users of gazpart_amd have it do, as timed cases.

Every case goes through the public entry points (``gazpart_amd.Context``,
``gazpart_amd.dns.Dns`` and, for a field that is already on the GPU, the
C-ABI's ``gp_bind_field_planar``).  Five kinds of work:

* ``step``    -- a run as the configurations have it: the particles of a
                 restart go in, K pipelined steps (advance + collisions),
                 the particles come back.
* ``host``    -- the drop-in pattern of a host code that owns PART: upload,
                 ADV_PARTICLE_ELLP, COLLISION, download, every cycle.
* ``dns``     -- the spectral fluid solver: K steps, then the velocity.
* ``coupled`` -- fluid and particles together, from a restart's particles:
                 fluid step, CHECK_CFL, the new field and DTIME to the
                 particles, one particle step, K times.
* ``stats``   -- a statistics cycle: the probes' INTERPH of all six fields,
                 STAT_PARTICLE with its PDFs, and STAT_PARTFLUID.

The particles of a case start with the fluid's velocity and half its
vorticity at their place, as in a run that has been going for a while.  Every
pass starts from the same particles (the explicit scheme of the reference
lets thin particles spin up without bound over thousands of steps).
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import gazpart_amd as G
from gazpart_amd import workload as W
from gazpart_amd.dns import Dns

L = 2.0 * math.pi
VISC, RHOF = 0.01, 1.0
MARGIN = 1.0e-9


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _step(name, n, np_, k, *, prec="mixed", scheme=3, kind="spheroids", phi=1e-3, nens=1,
          k0=4.0, graph=2, brick=0):
    c = dict(work="step", n=n, np=np_, k=k, prec=prec, scheme=scheme, kind=kind, phi=phi,
             nens=nens, k0=k0, graph=graph, brick=brick)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest run that is done in earnest, plain FP64: 10,000 equal
        # prolate spheroids on 64^3; a step is launches and latency
        _step("step 64^3 10k fp64", 64, 10_000, 64, prec="fp64", kind="equal", graph=1),
        # the usual run: 256^3, a million spheroids of all aspect ratios and
        # Stokes numbers, in the mixed form
        _step("step 256^3 1M mixed", 256, 1_000_000, 50),
        # and in the form that reproduces the reference's own arithmetic
        _step("step 256^3 1M fp64", 256, 1_000_000, 32, prec="fp64"),
        # its other interpolation scheme, tri-axial particles, sizes that
        # divide by nothing
        _step("step 101^3 123k fp64 lag4", 101, 123_457, 40, prec="fp64", scheme=4,
              kind="triaxial"),
        # a parameter study: 64 ensembles of 1e3 to 5e5 particles on one field
        _step("step 256^3 64 ensembles", 256, 5_700_000, 24, kind="ensembles", nens=64, graph=1,
              brick=2),
        # a dense suspension, 5 % by volume: collisions set the time
        _step("step 256^3 2M dense", 256, 2_000_000, 16, kind="triaxial", phi=0.05, graph=1),
        # the largest: 512^3 and 8 million tri-axial particles
        _step("step 512^3 8M mixed", 512, 8_000_000, 40, kind="triaxial", k0=8.0),
        # a host code that owns the particles and calls the step cycle by cycle
        dict(name="host 100^3 60k fp64", work="host", n=100, np=61_234, k=4, prec="fp64", scheme=3,
             kind="spheroids", phi=1e-3),
        # the fluid alone, small and at the usual run's size
        dict(name="dns 64^3", work="dns", n=64, k=40, k0=4.0),
        dict(name="dns 256^3", work="dns", n=256, k=16, k0=6.0),
        # an evolving, forced fluid with particles in it
        dict(name="coupled 128^3 200k", work="coupled", n=128, np=200_000, k=10, prec="mixed",
             scheme=3, kind="spheroids", phi=1e-3, k0=4.0),
        # a statistics cycle over a run of six particle sizes
        dict(name="stats 128^3 1M", work="stats", n=128, np=1_000_000, probes=100_000, nspec=6,
             prec="fp64", scheme=3),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    work = rng.choice(["step", "step", "step", "step", "host", "dns", "dns", "coupled", "stats"])
    if work == "step":
        kind = rng.choice(["equal", "spheroids", "spheroids", "triaxial", "triaxial", "ensembles"])
        np_ = _log(rng, 3_000, 3_000_000)
        phi = math.exp(rng.uniform(math.log(3e-4), math.log(5e-2))) if kind == "triaxial" else 1e-3
        nens = rng.randint(4, 80) if kind == "ensembles" else 1
        # a grid of 0.03 to 0.6 particles a node, as the configurations have
        n = int(min(320, max(40, round((np_ / math.exp(rng.uniform(math.log(0.03), math.log(0.6))))
                                       ** (1 / 3)))))
        return _step(None, n, np_, max(9, min(40, int(3e7 / np_))),
                     prec=rng.choice(["mixed", "mixed", "fp64"]), scheme=rng.choice([3, 3, 4]),
                     kind=kind, phi=phi, nens=nens, k0=float(rng.choice([4, 6, 8])),
                     graph=rng.choice([1, 2, 2]), brick=rng.choice([0, 0, 2]))
    if work == "host":
        np_ = _log(rng, 2_000, 400_000)
        n = rng.randint(48, 160)
        return dict(work=work, n=n, np=np_, k=rng.randint(1, 4), prec=rng.choice(["mixed", "fp64"]),
                    scheme=rng.choice([3, 4]), kind=rng.choice(["equal", "spheroids"]), phi=1e-3)
    if work == "dns":
        # the solver takes even sizes: powers of two mostly, as here, others too
        n = rng.choice([32, 64, 128, 128, 256, 48, 96, 100, 160, 192])
        k = rng.randint(4, 60) if n <= 128 else rng.randint(4, 16)
        return dict(work=work, n=n, k=k, k0=round(rng.uniform(3.0, 8.0), 3))
    if work == "coupled":
        n = rng.choice([48, 64, 96, 128, 128, 192])
        return dict(work=work, n=n, np=_log(rng, 5_000, 500_000), k=rng.randint(2, 12),
                    prec=rng.choice(["mixed", "fp64"]), scheme=rng.choice([3, 4]),
                    kind=rng.choice(["spheroids", "triaxial"]), phi=1e-3, k0=4.0)
    return dict(work=work, n=rng.randint(40, 160), np=_log(rng, 10_000, 2_000_000),
                probes=_log(rng, 300, 300_000), nspec=rng.choice([1, 2, 4, 6, 12]),
                prec=rng.choice(["mixed", "fp64"]), scheme=rng.choice([3, 4]))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1_000_003 + salt) & 0x7FFFFFFF)
    return g


def _velocity(n, k0, seed):
    """Divergence-free random Fourier velocity with E(k) ~ k^4 exp(-2 (k/k0)^2)
    and unit rms, and its vorticity: (3, n, n, n) each, x fastest."""
    g = _gen(seed, 1)
    o = dict(device="cuda", dtype=torch.float64)
    kz = torch.fft.fftfreq(n, 1.0 / n, **o)[:, None, None]
    ky = torch.fft.fftfreq(n, 1.0 / n, **o)[None, :, None]
    kx = torch.fft.rfftfreq(n, 1.0 / n, **o)[None, None, :]
    k2 = kx * kx + ky * ky + kz * kz
    amp = k2.sqrt() * torch.exp(-k2 / (k0 * k0))
    amp = torch.where((kx.abs() >= n // 2) | (ky.abs() >= n // 2) | (kz.abs() >= n // 2),
                      torch.zeros_like(amp), amp)
    k2[0, 0, 0] = 1.0
    w = [torch.complex(torch.randn(k2.shape, generator=g, **o), torch.randn(k2.shape, generator=g, **o))
         for _ in range(3)]
    div = (kx * w[0] + ky * w[1] + kz * w[2]) / k2
    uh = [amp * (w[0] - kx * div), amp * (w[1] - ky * div), amp * (w[2] - kz * div)]
    del w, div
    u = torch.stack([torch.fft.irfftn(c, s=(n, n, n)) for c in uh])
    s = 1.0 / float((u * u).mean().sqrt())
    om = torch.empty_like(u)
    om[0] = torch.fft.irfftn(1j * (ky * uh[2] - kz * uh[1]), s=(n, n, n))
    om[1] = torch.fft.irfftn(1j * (kz * uh[0] - kx * uh[2]), s=(n, n, n))
    om[2] = torch.fft.irfftn(1j * (kx * uh[1] - ky * uh[0]), s=(n, n, n))
    return u * s, om * s


def _umax(u):
    return float((u * u).sum(0).max().sqrt())


def _species(case, seed, np_):
    """(rows, species of each particle, ensemble of each particle or None)"""
    g = np.random.default_rng(int(seed) * 7919 + 11)
    kind, k0 = case.get("kind", "classes"), case.get("k0", 4.0)
    dx = L / (case["n"] - 1)

    def loguni(lo, hi, m):
        return np.exp(g.uniform(math.log(lo), math.log(hi), m))

    def rhop(st, deq):
        return W.rhop_for_stokes(st, deq, 1.0 / k0, RHOF, VISC)

    if kind == "equal":
        a = 0.2 * dx
        rows = W.species_spheroid(a, 2.0, rhop(1.0, 2.0 * a / 2.0 ** (2 / 3)))[None, :]
        return rows, np.zeros(np_, dtype=np.int32), None
    if kind == "classes":
        m = case["nspec"]
        a, apr = 0.2 * dx * g.uniform(0.5, 1.5, m), g.uniform(1.1, 4.0, m)
        rows = W.species_spheroid(a, apr, rhop(loguni(0.3, 3.0, m), 2.0 * a / apr ** (2 / 3)))
        return np.atleast_2d(rows), g.integers(0, m, np_).astype(np.int32), None
    req = (case["phi"] * L ** 3 * 3.0 / (4.0 * math.pi * np_)) ** (1.0 / 3.0)
    if kind == "triaxial":
        rb, rc = g.uniform(1.0, 4.0, np_), g.uniform(1.0, 4.0, np_)
        a = req * np.cbrt(rb * rc)
        rows = W.species_triaxial(a, a / rb, a / rc, rhop(1.0, np.full(np_, 2.0 * req)))
        return rows, np.arange(np_, dtype=np.int32), None
    if kind == "spheroids":
        apr = loguni(1 / 3, 3.0, np_)
        a = req * apr ** (2 / 3)
        rows = W.species_spheroid(a, apr, rhop(loguni(0.3, 10.0, np_), 2.0 * a / apr ** (2 / 3)))
        return rows, np.arange(np_, dtype=np.int32), None
    # ensembles: sizes spread over a factor of 500 as far as np allows
    m = case["nens"]
    share = loguni(1.0, 500.0, m)
    cnt = np.maximum(1, (share / share.sum() * np_).astype(np.int64))
    cnt[int(cnt.argmax())] += np_ - int(cnt.sum())
    apr = loguni(1 / 3, 3.0, m)
    a = 3.9e-3 * (256.0 / case["n"]) * apr ** (2 / 3)
    rows = W.species_spheroid(a, apr, rhop(loguni(0.3, 10.0, m), 2.0 * a / apr ** (2 / 3)))
    sid = np.repeat(np.arange(m, dtype=np.int32), cnt)
    return np.atleast_2d(rows), sid, sid.copy()


def _particles(np_, reach, u, om, seed):
    """State (13, np) on the host: uniform positions clear of the x walls,
    uniform orientations, the fluid's velocity and half its vorticity."""
    n = u.shape[-1]
    g = _gen(seed, 2)
    o = dict(device="cuda", dtype=torch.float64)
    x = reach + (L - 2.0 * reach) * torch.rand((3, np_), generator=g, **o)
    q = torch.randn((4, np_), generator=g, **o)
    q /= q.norm(dim=0)
    i = (x / (L / (n - 1))).round().long() % n
    at = (i[2] * n + i[1]) * n + i[0]
    v = u.reshape(3, -1)[:, at]
    h = 0.5 * ((n - 1) / n) * om.reshape(3, -1)[:, at]
    # into the body frame: R(q)^T h, as rotation by the conjugate
    a, b = q[0], -q[1:]
    t = 2.0 * torch.cross(b, h, dim=0)
    s = h + a * t + torch.cross(b, t, dim=0)
    return torch.cat([x, v, q, s]).cpu().numpy()


def _bind(ctx, u, om):
    torch.cuda.synchronize()
    n = u.shape[-1]
    ctx._chk(ctx.lib.gp_bind_field_planar(ctx.h, ctypes.c_int(n), ctypes.c_void_p(u.data_ptr()),
                                          ctypes.c_void_p(om.data_ptr()),
                                          ctypes.c_double((n - 1) / n)))


def _context(case, seed, u, om, **kw):
    rows, sid, grp = _species(case, seed, case["np"])
    # CFL 0.1, and no particle moves by more than a quarter of its size
    dt = min(0.1 * L / (case["n"] - 1), 0.25 * float(np.median(rows[:, :3].max(1)))) / _umax(u)
    ctx = G.Context(case["n"], L, VISC, RHOF, dt, scheme=case["scheme"],
                    precision=G.PREC_MIXED if case["prec"] == "mixed" else G.PREC_FP64,
                    dpmax=2.0 * float(max(rows[:, W.SP_EMAJ].max(), rows[:, :3].max())), **kw)
    _bind(ctx, u, om)
    ctx.set_species(rows)
    st = _particles(case["np"], float(rows[:, :3].max()) * (1.0 + MARGIN), u, om, seed)
    ctx.set_particles(st, sid)
    if grp is not None:
        ctx.set_groups(grp)
    return ctx, st, sid, grp


def prepare(case, seed):
    work, n = case["work"], case["n"]
    u, om = _velocity(n, case.get("k0", 4.0), seed)
    s = {"case": case}
    if work == "step":
        s["ctx"], s["state"], s["sid"], s["grp"] = _context(case, seed, u, om,
                                                            graph=case["graph"],
                                                            brick=case["brick"])
    elif work == "host":
        s["ctx"], s["state"], s["sid"], _ = _context(case, seed, u, om)
    elif work == "dns":
        s["dns"] = Dns(n, L, VISC, 0.05 * (L / (n - 1)) / _umax(u))
        s["dns"].set_velocity(u.cpu().numpy())
    elif work == "coupled":
        s["dns"] = Dns(n, L, VISC, 0.05 * (L / (n - 1)) / _umax(u),
                       forcing=dict(kmin=0.5, kmax=2.5, sigma=0.3, tforce=0.2, seed=-1 - seed % 999))
        s["dns"].set_velocity(u.cpu().numpy())
        s["ctx"], s["state"], s["sid"], _ = _context(case, seed, u, om, graph=2)
        s["dt"] = s["ctx"].params.dtime
    else:
        s["ctx"], _, _, _ = _context(case, seed, u, om, keep_fluid=True)
        s["ctx"].adv_particle_ellp()
        s["x"] = _probes(case, seed)
    torch.cuda.synchronize()
    return s


def _probes(case, seed):
    return np.random.default_rng(int(seed) * 31 + 5).uniform(0.0, L, (3, case["probes"]))


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    case = s["case"]
    work = case["work"]
    if work == "step":
        ctx = s["ctx"]
        ctx.set_particles(s["state"], s["sid"])
        if s["grp"] is not None:
            ctx.set_groups(s["grp"])
        ctx.step(case["k"])
        return {"particles": ctx.get_particles()}
    if work == "host":
        ctx, st = s["ctx"], s["state"]
        for c in range(case["k"]):
            ctx.set_particles(st, s["sid"])
            ctx.adv_particle_ellp(c + 1)
            ctx.collision(c + 1)
            st = ctx.get_particles()
        return {"particles": st}
    if work == "dns":
        s["dns"].step(case["k"])
        return {"velocity": s["dns"].velocity()}
    if work == "coupled":
        dns, ctx = s["dns"], s["ctx"]
        ctx.set_particles(s["state"], s["sid"])
        ctx.adv_particle_ellp(0)
        for c in range(case["k"]):
            dns.step(1)
            ctx.set_dtime(dns.cfl(s["dt"]))
            dns.bind(ctx)
            ctx.collision_advance(c + 1)
        return {"particles": ctx.get_particles(), "velocity": dns.velocity()}
    ctx, x = s["ctx"], s["x"]
    return {"probes": np.stack([ctx.interph(case["scheme"], c, x[0], x[1], x[2]) for c in range(6)]),
            "particle": ctx.particle_stats(), "pdf": ctx.particle_pdf(),
            "fluid": ctx.partfluid_stats()}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _stencil(case):
    return (4 if case["scheme"] == 3 else 5) ** 2 * 4


def _particle_step(case):
    """Bytes and operations of one advance with its collision pass: the state
    read and written, its constants read, the field nodes that some stencil
    reaches read once; the six weighted sums and the two Runge-Kutta stages."""
    n3, np_ = case["n"] ** 3, case["np"]
    fp64 = case["prec"] == "fp64"
    state = 2 * (7 * 8 + 6 * (8 if fp64 else 4))
    nodes = n3 * (1.0 - math.exp(-np_ * float((4 if case["scheme"] == 3 else 5) ** 3) / n3))
    by = np_ * (state + 96 + 2 * 16) + 6 * (8 if fp64 else 4) * nodes
    return by, np_ * (6 * 2 * _stencil(case) + 1500.0)


def _fluid_step(n):
    """The velocity read and written once a step, seven transforms of three
    components."""
    n3 = float(n) ** 3
    return 2 * 3 * 8 * n3, 7 * 3 * 2.5 * n3 * 3 * math.log2(n)


def work(case):
    w, n = case["work"], case["n"]
    if w == "dns":
        by, fl = _fluid_step(n)
        return {"bytes": case["k"] * by + 24.0 * n ** 3, "flops": case["k"] * fl}
    if w in ("step", "host"):
        by, fl = _particle_step(case)
        io = 2 * 13 * 8 * case["np"] * (1 if w == "step" else case["k"])
        return {"bytes": case["k"] * by + io, "flops": case["k"] * fl}
    if w == "coupled":
        pb, pf = _particle_step(case)
        fb, ff = _fluid_step(n)
        bind = n ** 3 * (3 * 8 + 6 * (8 if case["prec"] == "fp64" else 4))
        return {"bytes": case["k"] * (pb + fb + bind) + 2 * 13 * 8 * case["np"] + 24.0 * n ** 3,
                "flops": case["k"] * (pf + ff)}
    # statistics: the state once for each of the three, the fluid at the
    # particles, the probes' points and values
    st = 13 * 8 if case["prec"] == "fp64" else 7 * 8 + 6 * 4
    return {"bytes": case["np"] * (3.0 * st + 6 * 8) + case["probes"] * (24.0 + 48.0),
            "flops": case["np"] * 900.0 + case["probes"] * 6 * 2.0 * _stencil(case)}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def exact(case, seed):
    # the particles of a run have no such value: where the contact solve stops
    # short of a root, its iterates decide which pairs collide
    if case["work"] == "dns":
        return {"velocity": _exact_dns(case, seed)}
    if case["work"] == "stats":
        return {"probes": _exact_probes(case, seed), "particle": None, "pdf": None, "fluid": None}
    return None


def _exact_dns(case, seed):
    """The fluid steps with torch's transforms: integrating-factor RK2 of the
    rotational form, projection, cos^4 filter between 8/9 and 1 of pi n / L."""
    n, u = case["n"], _velocity(case["n"], case["k0"], seed)[0]
    dt = 0.05 * (L / (n - 1)) / _umax(u)
    o = dict(device="cuda", dtype=torch.float64)
    k1 = torch.arange(n, **o)
    k1 = torch.where(k1 <= n // 2, k1, k1 - n)
    kx, ky, kz = torch.arange(n // 2 + 1, **o)[None, None, :], k1[None, :, None], k1[:, None, None]
    k2 = kx * kx + ky * ky + kz * kz
    inv = torch.where(k2 > 0, 1.0 / torch.where(k2 > 0, k2, torch.ones_like(k2)),
                      torch.zeros_like(k2))
    r = k2.sqrt() / (math.pi * n / L)
    c = torch.cos((math.pi / 2) * (r - 8.0 / 9.0) / (1.0 - 8.0 / 9.0))
    filt = torch.where(r <= 8.0 / 9.0, torch.ones_like(r), torch.where(r <= 1.0, c ** 4,
                                                                     torch.zeros_like(r)))
    e = torch.exp(-VISC * k2 * dt)

    def back(a):
        return torch.fft.irfftn(torch.fft.ifftn(a, dim=(1, 2), norm="forward"), s=(n,), dim=(3,),
                                norm="forward")

    def rhs(v, V):
        z = back(torch.stack([1j * (ky * V[2] - kz * V[1]), 1j * (kz * V[0] - kx * V[2]),
                              1j * (kx * V[1] - ky * V[0])]))
        T = torch.fft.rfftn(torch.cross(v, z, dim=0), dim=(1, 2, 3), norm="forward")
        d = (kx * T[0] + ky * T[1] + kz * T[2]) * inv
        # the mean has no projection: its T is dropped (a |k|^2 of "infinity")
        T = torch.stack([T[0] - kx * d, T[1] - ky * d, T[2] - kz * d])
        T[:, 0, 0, 0] = 0.0
        return T

    for _ in range(case["k"]):
        U = torch.fft.rfftn(u, dim=(1, 2, 3), norm="forward")
        R = rhs(u, U)
        Un, U = (U + 0.5 * dt * R) * e, (U + dt * R) * e
        U = Un + 0.5 * dt * rhs(back(U), U)
        d = (kx * U[0] + ky * U[1] + kz * U[2]) * inv
        U = torch.stack([U[0] - kx * d, U[1] - ky * d, U[2] - kz * d]) * filt
        u = back(U)
    return u.cpu().numpy()


def _exact_probes(case, seed):
    """Lagrange interpolation on 4 nodes (or 5, with the y row of J + 2 taken
    at J + 1 as the reference's fourth-order routine does)."""
    n = case["n"]
    u, om = _velocity(n, case.get("k0", 4.0), seed)
    f = torch.cat([u, om * ((n - 1) / n)])
    x = torch.from_numpy(_probes(case, seed)).cuda() / (L / (n - 1))
    i0 = x.floor().long()
    off = [-1, 0, 1, 2] if case["scheme"] == 3 else [-2, -1, 0, 1, 2]
    a = x - i0
    wt = []
    for m in off:
        t = torch.ones_like(a)
        for j in off:
            if j != m:
                t = t * (a - j) / (m - j)
        wt.append(t)
    out = torch.zeros((6, x.shape[1]), device="cuda", dtype=torch.float64)
    for kz, mz in enumerate(off):
        for ky, my in enumerate(off):
            jy = (i0[1] + (1 if (case["scheme"] == 4 and my == 2) else my)) % n
            for kx, mx in enumerate(off):
                out += f[:, (i0[2] + mz) % n, jy, (i0[0] + mx) % n] * (wt[kx][0] * wt[ky][1] * wt[kz][2])
    return out.cpu().numpy()
