"""The workloads that this framework's speed is measured on.

Every case advances a dycore state by one large step (three Runge-Kutta stages,
``1 + max(1, ns // 2) + ns`` acoustic substeps) through the public entry points:
``Dycore.step``, ``Dycore.graph_step``, ``Ensemble.step`` (graph and persistent)
and ``step_noalloc``.  The grids are those of the idealized cases, the benchmark
and the ensemble, from an 80 x 1 x 40 slab to 433 x 433 x 50, with the option
sets that are run in earnest: the plain dry dynamics, the mixed-precision form,
constant-K diffusion, the regional set (map factors, rotation, log-pressure
specific volume, 6th-order filter, Smagorinsky diffusion, theta limiter) and
the moist step with transported species.

``listed`` gives the cases, ``draw`` more of the same ranges, ``prepare`` the
seeded state and the handle, ``run`` one pass, ``work`` the bytes and
operations that the pass cannot do without, ``exact`` the same step in plain
64-bit torch.
"""

from __future__ import annotations

import dataclasses
import math

import numpy as np
import torch

from wrf_gpu_amd import ic
from wrf_gpu_amd.dycore import Dycore, Ensemble, step_noalloc
from wrf_gpu_amd.grid import MOIST_FIELDS, STATE_FIELDS, Metrics, Namelist

ENSEMBLE = ((129, 129), (201, 201), (257, 257), (321, 321))


def _case(name, base, nx, ny, nz, ns, options="dry", entry="step", precision="fp64", members=1):
    return {"name": name, "base": base, "nx": nx, "ny": ny, "nz": nz, "ns": ns, "options": options,
            "entry": entry, "precision": precision, "members": members}


def listed():
    return [
        # the 2-D warm bubble slab, stepped 5000 times by its gate: the smallest
        # domain, where launches and latency are all there is
        _case("slab_80x1x40", "slab", 80, 1, 40, 10),
        # the 2-D density current with its constant-K diffusion, replayed from a graph
        _case("slab_500x1x60_constk_graph", "slab", 500, 1, 60, 10, options="constk", entry="graph"),
        # the CPU-sized 3-D warm bubble, stepped eagerly ...
        _case("bubble_64x64x40", "bubble", 64, 64, 40, 6),
        # ... by the persistent step, one launch per large step ...
        _case("bubble_64x64x40_persistent", "bubble", 64, 64, 40, 6, entry="persistent"),
        # ... and moist, without a handle (callers that cannot allocate), on a small odd grid
        _case("bubble_41x37x30_moist_noalloc", "bubble", 41, 37, 30, 6, options="moist", entry="noalloc"),
        # a regional domain with everything a real-data namelist turns on for a dry run
        _case("terrain_141x123x45_regional", "terrain", 141, 123, 45, 4, options="regional"),
        # the adjoint workload's domain, replayed from a graph
        _case("bubble_257x257x50_graph", "bubble", 257, 257, 50, 6, entry="graph"),
        # four ensemble members of uneven sizes, advanced together on the graph's branches ...
        _case("ensemble_4_members_graph", "ensemble", 321, 321, 50, 6, entry="ensemble", members=4),
        # ... and by the persistent step
        _case("ensemble_4_members_persistent", "ensemble", 321, 321, 50, 6, entry="persistent", members=4),
        # the headline workload: stratified flow over a hill
        _case("terrain_433x433x50", "terrain", 433, 433, 50, 6),
        # the same in the mixed-precision form
        _case("terrain_433x433x50_mixed", "terrain", 433, 433, 50, 6, precision="mixed"),
        # the same with the six species coupled and transported (the monotonic limiter)
        _case("terrain_433x433x50_moist", "terrain", 433, 433, 50, 6, options="moist"),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    base = rng.choice(("slab", "bubble", "bubble", "terrain", "terrain", "ensemble"))
    nz = rng.randint(20, 64)
    if base == "slab":
        return _drawn(base, size(40, 600), 1, nz, rng.choice((6, 8, 10)), rng.choice(("dry", "constk")),
                      rng.choice(("step", "graph")), "fp64", 1)
    if base == "ensemble":
        return _drawn(base, size(24, 321), size(24, 321), nz, rng.choice((4, 6)), "dry",
                      rng.choice(("ensemble", "persistent")), rng.choice(("fp64", "fp64", "mixed")), rng.randint(2, 4))
    options = rng.choice(("dry", "dry", "regional", "moist", "constk"))
    precision = "fp64" if options == "moist" else rng.choice(("fp64", "fp64", "mixed"))
    top = 433 if options in ("dry", "moist") and nz <= 50 else 320
    return _drawn(base, size(24, top), size(24, top), nz, rng.choice((4, 6)), options,
                  rng.choice(("step", "graph")), precision, 1)


def _drawn(*fields):
    case = _case("", *fields)
    del case["name"]
    return case


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _members(case):
    """(base, nx, ny) of each domain of the case; an ensemble's members shrink
    from the largest as the 32-member ensemble's do."""

    if case["base"] != "ensemble":
        return [(case["base"], case["nx"], case["ny"])]
    scale = [n / ENSEMBLE[-1][0] for n, _ in ENSEMBLE][-case["members"]:]
    return [("ensemble", max(8, round(case["nx"] * s)), max(8, round(case["ny"] * s))) for s in scale]


def _noise(shape, length, sigma, gen, dev):
    """Gaussian noise of standard deviation sigma, correlated over `length` cells."""

    white = torch.randn(shape, generator=gen, device=dev, dtype=torch.float64)
    kx = torch.fft.fftfreq(shape[-1], device=dev, dtype=torch.float64) * (2 * math.pi * length)
    ky = torch.fft.fftfreq(shape[-2], device=dev, dtype=torch.float64) * (2 * math.pi * length)
    damp = torch.exp(-0.5 * (kx[None, :] ** 2 + ky[:, None] ** 2))
    out = torch.fft.ifft2(torch.fft.fft2(white) * damp).real
    return out * (sigma / out.std())


def _domain(base, nx, ny, nz, ns, options, gen):
    """Metrics, namelist and seeded initial state (device tensors) of one domain:
    hydrostatically balanced columns, as the idealized cases build them."""

    dev = str(gen.device)
    f64 = {"device": dev, "dtype": torch.float64}
    p_top = 5000.0
    if base == "slab":  # dx = 250 m, or the density current's 100 m; uniform layers of that depth
        dx = 100.0 if options == "constk" else 250.0
        depth = min(dx, 12000.0 / nz)
        eta, _, _, mass = ic.uniform_z_hydrostatic_base(np.arange(nz + 1) * depth, ic.THETA0)
        p_top, dt, zdamp = ic.P0 - mass, 0.1, 0.25 * nz * depth
    elif base == "terrain":  # stretched levels
        eta = 1.0 - (np.arange(nz + 1) / nz) ** 1.4
        dx, dt, zdamp = 3000.0, 3.0 * ns, 5000.0
    else:
        eta = np.linspace(1.0, 0.0, nz + 1)
        dx, dt, zdamp = 1000.0, 1.0 * ns, 5000.0
    m = Metrics.flat(nx=nx, ny=ny, nz=nz, dx=dx, dy=dx, eta=eta, p_top=p_top)
    nl = Namelist(dt_s=dt, acoustic_substeps=ns, zdamp=zdamp)
    if options == "constk":
        nl = nl.replace(const_nu_m2_s=75.0)
    elif options == "moist":
        nl = nl.replace(moist=True, moist_adv_opt=2)
    elif options == "regional":
        nl = nl.replace(diff_6th_opt=2, diff_opt=1, km_opt=4, scalar_adv_opt=2, hypsometric_opt=2)
        m = _regional(m)

    x = (torch.arange(nx, **f64) + 0.5) * dx
    y = (torch.arange(ny, **f64) + 0.5) * dx
    r2 = (x[None, :] - 0.5 * nx * dx) ** 2 + ((y[:, None] - 0.5 * ny * dx) ** 2 if ny > 1 else 0.0)
    kappa = ic.R_DRY / ic.CP_DRY
    if base == "terrain":
        n2, theta_s = 1.0e-4, 288.0
        height = 1000.0 / (1.0 + r2 / 1.0e8)
        exner = 1.0 - ic.GRAVITY ** 2 / (ic.CP_DRY * theta_s * n2) * (1.0 - torch.exp(-n2 * height / ic.GRAVITY))
        mub = ic.P0 * exner ** (1.0 / kappa) - p_top

        def theta_base(z):
            return theta_s * torch.exp(n2 * z / ic.GRAVITY)
    else:
        height = torch.zeros((ny, nx), **f64)
        mub = torch.full((ny, nx), ic.P0 - p_top, **f64)

        def theta_base(z):
            return torch.full_like(z, ic.THETA0)

    def alpha(theta, p):
        return (ic.R_DRY / ic.P0) * theta * (p / ic.P0) ** (kappa - 1.0)

    znw = torch.tensor(m.eta, **f64)
    dnw = (znw[1:] - znw[:-1])[:, None, None]
    pb = 0.5 * (znw[1:] + znw[:-1])[:, None, None] * mub + p_top
    phb0 = ic.GRAVITY * height[None]

    def faces(alt):
        return torch.cat([phb0, phb0 - torch.cumsum(dnw * mub * alt, 0)])

    z = height + 7000.0 * torch.log(pb[:1] / pb)
    for _ in range(4):
        phb = faces(alpha(theta_base(z), pb))
        z = 0.5 * (phb[1:] + phb[:-1]) / ic.GRAVITY
    alb = alpha(theta_base(z), pb)
    phb = faces(alb)
    if base == "slab":
        amp, rx, zc = (-15.0, 4000.0, 3000.0) if options == "constk" else (2.0, 2000.0, 2000.0)
        r = torch.sqrt(r2 / rx ** 2 + ((z - zc) / 2000.0) ** 2)
        tp = amp * torch.where(r <= 1.0, 0.5 * (1.0 + torch.cos(math.pi * r)), torch.zeros_like(r))
        tp = tp + 0.01 * (2.0 * torch.rand(z.shape, generator=gen, **f64) - 1.0)
    elif base == "bubble":
        r = torch.sqrt(r2 / 4.0e6 + ((z - 2000.0) / 2000.0) ** 2)
        tp = 2.0 * torch.where(r <= 1.0, 0.5 * (1.0 + torch.cos(math.pi * r)), torch.zeros_like(r))
        tp = tp + 0.01 * (2.0 * torch.rand(z.shape, generator=gen, **f64) - 1.0)
    else:
        tp = _noise((nz, ny, nx), 20000.0 / dx, 0.5 if base == "ensemble" else 0.1, gen, dev)
    theta = theta_base(z) + tp
    al = alpha(theta, pb) - alb
    php = torch.cat([torch.zeros_like(phb0), -torch.cumsum(dnw * mub * al, 0)])
    alt = alb - (php[1:] - php[:-1]) / dnw / mub
    p_full = ic.P0 * ((ic.R_DRY * theta) / (ic.P0 * alt)) ** (1.0 / (1.0 - kappa))
    u = torch.full((nz, ny, nx + 1), 0.0 if base == "slab" else 10.0, **f64)
    v = torch.zeros((nz, ny + 1, nx), **f64)
    if base in ("ensemble", "terrain"):
        u += _noise(u.shape, 20000.0 / dx, 1.0, gen, dev)
        v += _noise(v.shape, 20000.0 / dx, 1.0, gen, dev)
    s = {"u": u, "v": v, "w": torch.zeros((nz + 1, ny, nx), **f64),
         "theta": theta, "p_total": p_full, "p_perturbation": p_full - pb, "ph_total": phb + php,
         "ph_perturbation": php, "mu_total": mub.clone(), "mu_perturbation": torch.zeros((ny, nx), **f64),
         "mudf": torch.zeros((ny, nx), **f64)}
    if nl.moist:
        zz = (z - z[:1]).clamp_min(0.0)
        s["qv"] = 0.012 * torch.exp(-zz / 2500.0) * (1.0 + 0.1 * (torch.rand(z.shape, generator=gen, **f64) - 0.5))
        for q, amp, at in (("qc", 1.0e-3, 0.3), ("qr", 4.0e-4, 0.2), ("qi", 2.0e-4, 0.7), ("qs", 1.0e-4, 0.6),
                           ("qg", 1.5e-4, 0.4)):
            level = torch.exp(-((torch.arange(nz, **f64) - at * nz) / 3.0) ** 2)[:, None, None]
            s[q] = amp * level * _noise((1, ny, nx), 4.0, 1.0, gen, dev).clamp_min(0.0)
    return m, nl, {k: v.contiguous() for k, v in s.items()}


def _regional(m):
    """The metrics of a mid-latitude projection: map factors and rotation, and
    the dry-pressure coefficients that the log-pressure specific volume reads."""

    def factor(ny, nx, sj, si):
        j, i = np.meshgrid((np.arange(ny) + sj) / max(m.ny, 1), (np.arange(nx) + si) / m.nx, indexing="ij")
        return 1.0 + 0.02 * np.cos(2 * np.pi * j) + 0.01 * np.cos(2 * np.pi * i)

    msft = factor(m.ny, m.nx, 0.5, 0.5)
    msfu, msfv = factor(m.ny, m.nx + 1, 0.5, 0.0), factor(m.ny + 1, m.nx, 0.0, 0.5)
    lat = np.deg2rad(40.0 + 5.0 * (np.arange(m.ny) / m.ny - 0.5))[:, None] * np.ones((1, m.nx))
    turn = np.deg2rad(4.0) * (np.arange(m.nx) / m.nx - 0.5)[None, :] * np.ones((m.ny, 1))
    return dataclasses.replace(m, c3h=0.5 * (m.eta[1:] + m.eta[:-1]), c3f=m.eta.copy(), msftx=msft, msfty=msft, msfux=msfu, msfuy=msfu, msfvx=msfv, msfvy=msfv,
                               f=1.4584e-4 * np.sin(lat), e=1.4584e-4 * np.cos(lat), sina=np.sin(turn),
                               cosa=np.cos(turn))


def _inputs(case, seed):
    gen = torch.Generator(device=_device())
    gen.manual_seed(int(seed))
    return [_domain(base, nx, ny, case["nz"], case["ns"], case["options"], gen)
            for base, nx, ny in _members(case)]


# --------------------------------------------------------------------------
# One pass
# --------------------------------------------------------------------------
def prepare(case, seed):
    domains = _inputs(case, seed)
    state = {"entry": case["entry"], "fields": [s for _, _, s in domains]}
    if case["entry"] == "noalloc":
        state["metrics"], state["namelist"] = domains[0][0], domains[0][1]
        return state
    state["dycores"] = [Dycore(m, nl, precision=case["precision"]) for m, nl, _ in domains]
    if case["entry"] == "graph":
        state["dycores"][0].capture_graph(state["fields"][0])
    elif case["entry"] in ("ensemble", "persistent"):
        state["ensemble"] = Ensemble(list(zip(state["dycores"], state["fields"])),
                                     persistent=case["entry"] == "persistent")
    return state


def run(state):
    fields = state["fields"]
    if state["entry"] == "step":
        state["dycores"][0].step(fields[0])
    elif state["entry"] == "graph":
        state["dycores"][0].graph_step()
    elif state["entry"] == "noalloc":
        step_noalloc(fields[0], state["namelist"], state["metrics"])
    else:
        state["ensemble"].step()
    return fields


# Operations per cell of one stage's setup and finish, and of one acoustic
# substep (a divide counted as one, a pow as 60), from the expressions.
_STAGE_FLOPS, _SUBSTEP_FLOPS, _SPECIES_FLOPS = 520, 170, 400


def work(case):
    """The state read and written once; the operations of its stages and substeps."""

    n_fields = 8 + (len(MOIST_FIELDS) if case["options"] == "moist" else 0)
    ns = case["ns"]
    substeps = 1 + max(1, ns // 2) + ns
    cells = sum(nx * ny * case["nz"] for _, nx, ny in _members(case))
    flops = 3 * _STAGE_FLOPS + substeps * _SUBSTEP_FLOPS
    if case["options"] == "moist":
        flops += len(MOIST_FIELDS) * _SPECIES_FLOPS
    return {"bytes": 2 * 8 * n_fields * cells, "flops": flops * cells}


# --------------------------------------------------------------------------
# The same large step in plain 64-bit torch
# --------------------------------------------------------------------------
def exact(case, seed):
    return [_large_step(m, nl, s) for m, nl, s in _inputs(case, seed)]


RD, G, T0 = 287.0, 9.81, 300.0
CP = 7.0 * RD / 2.0
CPOVCV, CVPM = CP / (CP - RD), -(CP - RD) / CP
P0 = 100000.0


def _x(q, d):
    return torch.roll(q, -d, -1)


def _y(q, d):
    return torch.roll(q, -d, -2)


def _flux5(q, vel, sh):
    """The upwind-biased fifth-order flux through each point's minus face."""

    a, b, c, d, e, f = (sh(q, n) for n in (-3, -2, -1, 0, 1, 2))
    f6 = (37.0 * (d + c) - 8.0 * (e + b) + (f + a)) / 60.0
    return vel * (f6 - torch.sign(vel) * ((f - a) - 5.0 * (e - b) + 10.0 * (d - c)) / 60.0)


def _flux3(q, vel):
    """The third-order vertical flux vel * F through faces 2 .. n-2 of n levels."""

    a, b, c, d = q[:-3], q[1:-2], q[2:-1], q[3:]
    return vel * ((7.0 * (c + b) - (d + a)) / 12.0 + torch.sign(-vel) * ((d - a) - 3.0 * (c - b)) / 12.0)


def _edge_x(q):
    """Mass points averaged to the u faces, edge values at the ends."""

    return torch.cat([q[..., :1], 0.5 * (q[..., 1:] + q[..., :-1]), q[..., -1:]], -1)


def _edge_y(q):
    return torch.cat([q[..., :1, :], 0.5 * (q[..., 1:, :] + q[..., :-1, :]), q[..., -1:, :]], -2)


def _pad_x(q):
    return torch.cat([q[..., :1], q, q[..., -1:]], -1)


def _pad_y(q):
    return torch.cat([q[..., :1, :], q, q[..., -1:, :]], -2)


class _Grid:
    """Metrics as tensors: vertical ones (n, 1, 1), map factors (ny, nx)."""

    def __init__(self, m, dev):
        def t(a):
            return torch.tensor(np.asarray(a), device=dev, dtype=torch.float64)

        for k in ("c1h", "c2h", "c1f", "c2f", "dnw", "rdnw", "dn", "rdn", "fnm", "fnp", "c3h", "c4h", "c3f", "c4f"):
            setattr(self, k, t(getattr(m, k))[:, None, None])
        for k in ("msftx", "msfty", "msfux", "msfuy", "msfvx", "msfvy", "f", "e", "sina", "cosa"):
            setattr(self, k, t(getattr(m, k)))
        self.nx, self.ny, self.nz, self.dx, self.dy = m.nx, m.ny, m.nz, m.dx, m.dy
        self.rdx, self.rdy, self.p_top, self.rotating = 1.0 / m.dx, 1.0 / m.dy, m.p_top, m.rotating
        self.cf = (m.cf1, m.cf2, m.cf3)
        dn = m.dn[-1] if abs(m.dn[-1]) > 1e-30 else 1.0
        self.cfn, self.cfn1 = (0.5 * m.dnw[-1] + m.dn[-1]) / dn, -0.5 * m.dnw[-1] / dn

    def mh(self, mu):
        return self.c1h * mu + self.c2h

    def mf(self, mu):
        return self.c1f * mu + self.c2f

    def to_faces(self, q):
        """Mass levels interpolated to the interior w faces 1 .. nz-1."""

        return self.fnm[1:] * q[1:] + self.fnp[1:] * q[:-1]


def _log_alpha(g, dph, mass):
    pf = g.c3f * mass + g.c4f + g.p_top
    return dph / (g.c3h * mass + g.c4h + g.p_top) / torch.log(pf[:-1] / pf[1:])


def _vertical(g, q, r):
    """The vertical flux through the w faces: 2nd order next to the lids, 3rd inside."""

    out = torch.zeros_like(r)
    out[1] = r[1] * (g.fnm[1] * q[1] + g.fnp[1] * q[0])
    out[-2] = r[-2] * (g.fnm[-1] * q[-1] + g.fnp[-1] * q[-2])
    out[2:-2] = _flux3(q, r[2:-2])
    return out


def _advect(g, q, ru, rv, rom):
    fx, fy, fz = _flux5(q, ru, _x), _flux5(q, rv, _y), _vertical(g, q, rom)
    t = -g.msftx * g.rdx * (_x(fx, 1) - fx) - g.msftx * g.rdy * (_y(fy, 1) - fy)
    return t - g.rdnw * (fz[1:] - fz[:-1])


def _limited(g, opt, q, q0, mu, mu0, ru, rv, rom, dt):
    """Flux-limited advection from the step origin q0 (1 positive-definite, 2 monotonic)."""

    def upwind(qm, qp, vel, mass, width):
        cr = vel * dt / width / mass
        return mass * (width / dt) * (0.5 * (cr + cr.abs()).clamp_max(1.0) * qm
                                      + 0.5 * (cr - cr.abs()).clamp_min(-1.0) * qp)

    lx = upwind(_x(q0, -1), q0, ru, g.mh(0.5 * (mu + _x(mu, -1))), g.dx)
    ly = upwind(_y(q0, -1), q0, rv, g.mh(0.5 * (mu + _y(mu, -1))), g.dy)
    lz = torch.zeros_like(rom)
    mh = g.mh(mu).expand(q.shape)
    dz = 2.0 / (g.rdnw[1:] + g.rdnw[:-1])
    lz[1:-1] = upwind(q0[:-1], q0[1:], rom[1:-1], 0.5 * (mh[1:] + mh[:-1]), dz)
    ax, ay, az = _flux5(q, ru, _x) - lx, _flux5(q, rv, _y) - ly, _vertical(g, q, rom) - lz

    def pos(a):
        return a.clamp_min(0.0)

    def neg(a):
        return a.clamp_max(0.0)

    m2 = g.msftx * g.msftx
    ax1, ay1, lx1, ly1 = _x(ax, 1), _y(ay, 1), _x(lx, 1), _y(ly, 1)
    low = g.mh(mu0) * q0 - dt * (m2 * (g.rdx * (lx1 - lx) + g.rdy * (ly1 - ly)) + g.msftx * g.rdnw * (lz[1:] - lz[:-1]))
    out = dt * (m2 * (g.rdx * (pos(ax1) - neg(ax)) + g.rdy * (pos(ay1) - neg(ay)))
                + g.msftx * g.rdnw * (neg(az[1:]) - pos(az[:-1])))

    def scale(flux, room):
        return torch.where(flux > room, (room / (flux + 1.0e-20)).clamp_min(0.0), torch.ones_like(flux))

    if opt == 1:
        s = scale(out, low)
        sx = torch.where(ax > 0.0, _x(s, -1), s)
        sy = torch.where(ay > 0.0, _y(s, -1), s)
        sz = torch.where(az[1:-1] < 0.0, s[:-1], s[1:])
    else:
        up, dn = torch.cat([q0[1:], q0[-1:]]), torch.cat([q0[:1], q0[:-1]])
        around = torch.stack([q0, _x(q0, 1), _x(q0, -1), _y(q0, 1), _y(q0, -1), up, dn])
        into = -dt * (m2 * (g.rdx * (neg(ax1) - pos(ax)) + g.rdy * (neg(ay1) - pos(ay)))
                      + g.msftx * g.rdnw * (pos(az[1:]) - neg(az[:-1])))
        sa = scale(into, around.amax(0) * g.mh(mu0) - low)
        sb = scale(out, low - around.amin(0) * g.mh(mu0))
        sx = torch.where(ax > 0.0, torch.minimum(sa, _x(sb, -1)), torch.minimum(sb, _x(sa, -1)))
        sy = torch.where(ay > 0.0, torch.minimum(sa, _y(sb, -1)), torch.minimum(sb, _y(sa, -1)))
        sz = torch.where(az[1:-1] < 0.0, torch.minimum(sa[1:], sb[:-1]), torch.minimum(sb[1:], sa[:-1]))
    fx, fy = sx * ax + lx, sy * ay + ly
    fz = torch.zeros_like(lz)
    fz[1:-1] = sz * az[1:-1] + lz[1:-1]
    return (-g.msftx * g.rdx * (_x(fx, 1) - fx) - g.msftx * g.rdy * (_y(fy, 1) - fy)
            - g.rdnw * (fz[1:] - fz[:-1]))


def _diffusion(g, nl, s):
    """The explicit diffusion tendencies of u, v, w, theta."""

    mu = s["mu_total"]
    fields = [(s["u"], g.mh(_edge_x(mu))), (s["v"], g.mh(_edge_y(mu))), (s["w"], g.mf(mu)), (s["theta"], g.mh(mu))]
    total = [torch.zeros_like(f) for f, _ in fields]
    if nl.diff_6th_opt:
        coef = nl.diff_6th_factor * 0.015625 / (2.0 * nl.dt_s)
        for n, (f, mass) in enumerate(fields):
            line = torch.zeros_like(f)
            for sh in (_x, _y)[: 2 if f.shape[-2] > 1 else 1]:
                d = 10.0 * (f - sh(f, -1)) - 5.0 * (sh(f, 1) - sh(f, -2)) + (sh(f, 2) - sh(f, -3))
                d = torch.where(d * (f - sh(f, -1)) <= 0.0, torch.zeros_like(d), d)
                line = line + coef * (sh(d, 1) - d)
            total[n] += mass * line
    if nl.const_nu_m2_s > 0.0:
        ph = s["ph_total"]
        dz = max(float(((ph[1:] - ph[:-1]) / G).mean()), 1.0)
        for n, (f, mass) in enumerate(fields):
            mass = mass.expand(f.shape)
            t = torch.zeros_like(f)
            for sh, d in ((_x, g.dx), (_y, g.dy))[: 2 if f.shape[-2] > 1 else 1]:
                flux = 0.5 * (mass + sh(mass, -1)) * nl.const_nu_m2_s * (f - sh(f, -1)) / d
                t = t + (sh(flux, 1) - flux) / d
            flux = 0.5 * (mass[1:] + mass[:-1]) * nl.const_nu_m2_s * (f[1:] - f[:-1]) / dz
            t[:-1] += flux / dz
            t[1:] -= flux / dz
            total[n] += t
    if nl.diff_opt == 1:
        u, v = s["u"][..., :-1], s["v"][:, :-1]
        d12 = (u - _y(u, -1)) * g.rdy + (v - _x(v, -1)) * g.rdx
        d11, d22 = 2.0 * (_x(u, 1) - u) * g.rdx, 2.0 * (_y(v, 1) - v) * g.rdy
        corner = 0.25 * (d12 + _y(d12, 1) + _x(d12, 1) + _y(_x(d12, 1), 1))
        mlen = math.sqrt(g.dx * g.dy)
        km = (nl.c_s ** 2 * mlen * mlen * torch.sqrt(0.25 * (d11 - d22) ** 2 + corner ** 2)).clamp_max(10.0 * mlen)
        km_w = torch.cat([km[:1], 0.5 * (km[1:] + km[:-1]), km[-1:]])
        for n, (f, k) in enumerate(((u, km), (v, km), (s["w"], km_w), (s["theta"] - T0, 3.0 * km))):
            mass = fields[n][1][..., : g.ny, : g.nx]
            t = torch.zeros_like(f)
            for sh, rd in ((_x, g.rdx), (_y, g.rdy))[: 2 if g.ny > 1 else 1]:
                flux = 0.5 * (k + sh(k, -1)) * (0.5 * (mass + sh(mass, -1))) * rd * (f - sh(f, -1))
                t = t + rd * (sh(flux, 1) - flux)
            t = torch.cat([t, t[..., :1]], -1) if n == 0 else torch.cat([t, t[:, :1]], 1) if n == 1 else t
            total[n] += t
    return total


def _large_step(m, nl, s):
    g = _Grid(m, s["u"].device)
    s = dict(s)
    origin = dict(s)
    dt, ns = nl.dt_s, nl.acoustic_substeps
    for rk, dts, nsub, dt_rk in ((1, dt / 3.0, 1, dt / 3.0), (2, dt / ns, max(1, ns // 2), 0.5 * dt), (3, dt / ns, ns, dt)):
        _stage(g, nl, s, origin, rk, dts, nsub, dt_rk)
    return {k: s[k].contiguous() for k in STATE_FIELDS + (MOIST_FIELDS if nl.moist else ())}


def _stage(g, nl, s, origin, rk, dts, nsub, dt_rk):
    nx, ny, nz = g.nx, g.ny, g.nz
    cf1, cf2, cf3 = g.cf
    u, v, w, th = s["u"], s["v"], s["w"], s["theta"]
    p, pp, ph, php = s["p_total"], s["p_perturbation"], s["ph_total"], s["ph_perturbation"]
    mu_t, mu_p = s["mu_total"], s["mu_perturbation"]
    mub, phb, pb = mu_t - mu_p, ph - php, p - pp
    mut = mub + mu_p
    mu_work = torch.zeros_like(mu_p) if rk == 1 else origin["mu_perturbation"] - mu_p
    muts, mu_c = mut + mu_work, mu_p + mu_work
    muu, muus, muv, muvs = _edge_x(mut), _edge_x(muts), _edge_y(mut), _edge_y(muts)

    # transport velocities
    ru = g.mh(0.5 * (mu_t + _x(mu_t, -1))) * u[..., :-1] / g.msfuy[:, :-1]
    rv = g.mh(0.5 * (mu_t + _y(mu_t, -1))) * v[:, :-1] / g.msfvx[:-1]
    div = g.dnw * g.msftx * (g.rdx * (_x(ru, 1) - ru) + g.rdy * (_y(rv, 1) - rv))
    rom = torch.zeros((nz + 1, ny, nx), device=u.device, dtype=u.dtype)
    rom[1:-1] = torch.cumsum(-g.dnw * g.c1h * div.sum(0) - div, 0)[:-1]

    # stage diagnostics
    alt_raw = (RD / P0) * th * (p.clamp_min(1.0) / P0) ** CVPM
    if nl.hypsometric_opt == 2:
        al_ls = _log_alpha(g, ph[1:] - ph[:-1], mu_t) - _log_alpha(g, phb[1:] - phb[:-1], mub)
    else:
        alb = -g.rdnw * (phb[1:] - phb[:-1]) / g.mh(mub)
        al_ls = -(alb * g.c1h * mu_p + g.rdnw * (php[1:] - php[:-1])) / g.mh(mu_t + mu_p)
    php_ls = 0.5 * (ph[1:] + ph[:-1])
    alt = alt_raw.clamp_min(0.1)
    c2a = CPOVCV * (pb + pp) / alt

    # moisture factors
    cqu, cqv, cq1, cq2 = 1.0, 1.0, 1.0, 0.0
    if nl.moist:
        qtot = sum(s[q] for q in MOIST_FIELDS)
        cqu, cqv = 1.0 / (1.0 + _edge_x(qtot)), 1.0 / (1.0 + _edge_y(qtot))
        cqw = 0.5 * (qtot[1:] + qtot[:-1])
        cq1, cq2 = 1.0 / (1.0 + cqw), cqw / (1.0 + cqw)

    # advective tendencies
    diff = _diffusion(g, nl, s)
    rom_u = 0.5 * (rom + _x(rom, -1))
    uu, vx = u[..., :-1], 0.5 * (ru + _x(ru, -1))
    fx = _flux5(uu, _x(vx, 1), lambda q, n: _x(q, n + 1))  # through the face east of each u point
    ut = -g.msfux[:, :-1] * g.rdx * (fx - _x(fx, -1))
    if ny > 1:
        fy = _flux5(uu, 0.5 * (rv + _x(rv, -1)), _y)
        ut = ut - g.msfux[:, :-1] * g.rdy * (_y(fy, 1) - fy)
    fz = _vertical(g, uu, rom_u)
    ut = ut - g.rdnw * (fz[1:] - fz[:-1])
    ut = torch.cat([ut, ut[..., :1]], -1) + diff[0]
    vv = v[:, :-1]
    fx = _flux5(vv, 0.5 * (ru + _y(ru, -1)), _x)
    fy = _flux5(vv, 0.5 * (_y(rv, 1) + rv), lambda q, n: _y(q, n + 1))
    fz = _vertical(g, vv, 0.5 * (rom + _y(rom, -1)))
    vt = -g.msfvy[:-1] * (g.rdx * (_x(fx, 1) - fx) + g.rdy * (fy - _y(fy, -1)))
    vt = vt - g.msfvy[:-1] / g.msfvx[:-1] * g.rdnw * (fz[1:] - fz[:-1])
    vt = torch.cat([vt, vt[:, :1]], 1) + diff[1]
    ruf, rvf = torch.cat([ru[:1], g.to_faces(ru), ru[-1:]]), torch.cat([rv[:1], g.to_faces(rv), rv[-1:]])
    fx = _flux5(w, ruf, _x)
    wt = -g.msftx * g.rdx * (_x(fx, 1) - fx)
    if ny > 1:
        fy = _flux5(w, rvf, _y)
        wt = wt - g.msftx * g.rdy * (_y(fy, 1) - fy)
    fz = torch.zeros_like(w)  # fz[f]: the flux between the w faces f-1 and f
    vel = 0.5 * (rom[1:] + rom[:-1])
    fz[1] = vel[0] * 0.5 * (w[1] + w[0])
    fz[2:-1] = _flux3(w, vel[1:-1])
    wt[1:-1] -= g.rdn[1:] * (fz[2:] - fz[1:-1])
    wt = wt + diff[2]
    limit = rk == 3 and nl.scalar_adv_opt
    if limit:
        tt = _limited(g, nl.scalar_adv_opt, th - T0, origin["theta"] - T0, mu_t, origin["mu_total"], ru, rv, rom, nl.dt_s)
    else:
        tt = _advect(g, th - T0, ru, rv, rom)
    tt = tt + diff[3]
    qt = {}
    if nl.moist and nl.moist_adv_opt:
        for q in MOIST_FIELDS:
            if rk == 3:
                qt[q] = _limited(g, nl.moist_adv_opt, s[q], origin[q], mu_t, origin["mu_total"], ru, rv, rom, nl.dt_s)
            else:
                qt[q] = _advect(g, s[q], ru, rv, rom)

    # large-step pressure gradient
    def large_pgf(pad, dim, msf, rd, mass):
        def lr(q):
            q = pad(q)
            return q.narrow(dim, 0, q.shape[dim] - 1), q.narrow(dim, 1, q.shape[dim] - 1)

        (ppl, ppr), (phl, phr), (al, ar), (bl, br) = lr(pp), lr(php), lr(alt_raw), lr(al_ls)
        (pbl, pbr), (hl, hr), (ml, mr) = lr(pb), lr(php_ls), lr(mu_p)
        ps = ppl + ppr
        dpn = torch.cat([0.5 * (cf1 * ps[:1] + cf2 * ps[1:2] + cf3 * ps[2:3]), 0.5 * g.to_faces(ps),
                         0.5 * (g.cfn * ps[-1:] + g.cfn1 * ps[-2:-1])])
        d = phr - phl
        grad = msf * 0.5 * rd * mass * ((d[1:] + d[:-1]) + (al + ar) * (ppr - ppl) + (bl + br) * (pbr - pbl))
        return grad + msf * rd * (hr - hl) * (g.rdnw * (dpn[1:] - dpn[:-1]) - 0.5 * g.c1h * (ml + mr))

    msf_u, msf_v = g.msfux / g.msfuy, g.msfvy / g.msfvx

    def mean2(q, dim):
        return 0.5 * (q.narrow(dim, 0, q.shape[dim] - 1) + q.narrow(dim, 1, q.shape[dim] - 1))

    ut = ut - cqu * large_pgf(_pad_x, -1, msf_u, g.rdx, g.mh(mean2(_pad_x(mut), -1)))
    vt = vt - cqv * large_pgf(_pad_y, -2, msf_v, g.rdy, g.mh(mean2(_pad_y(mut), -2)))
    if g.rotating:
        ru_e = u * g.mh(mean2(_pad_x(mu_t), -1)) / g.msfuy
        rv_e = v * g.mh(mean2(_pad_y(mu_t), -2)) / g.msfvx
        rw = w * g.mf(mu_t) / g.msfty
        rw = 0.5 * (rw[1:] + rw[:-1])
        ut = ut + msf_u * mean2(_pad_x(g.f), -1) * mean2(_pad_x(mean2(rv_e, -2)), -1)
        ut = ut - mean2(_pad_x(g.e), -1) * mean2(_pad_x(g.cosa), -1) * mean2(_pad_x(rw), -1)
        vt = vt - msf_v * mean2(_pad_y(g.f), -2) * mean2(_pad_y(mean2(ru_e, -1)), -2)
        vt = vt + msf_v * mean2(_pad_y(g.e), -2) * mean2(_pad_y(g.sina), -2) * mean2(_pad_y(rw), -2)

    # small-step work variables
    uw = (g.mh(muus) * origin["u"] - g.mh(muu) * u) / g.msfuy
    vw = (g.mh(muvs) * origin["v"] - g.mh(muv) * v) / g.msfvx
    ww = (g.mf(muts) * origin["w"] - g.mf(mut) * w) / g.msfty
    tw = g.mh(muts) * (origin["theta"] - T0) - g.mh(mut) * (th - T0)
    phw = origin["ph_perturbation"] - php
    ph1 = origin["ph_perturbation"] + phb
    php_h = 0.5 * (phb[:-1] + phb[1:] + php[:-1] + php[1:])

    def p_rho(mw, mass, t1, tw, phw):
        al = -(alt * g.c1h * mw + g.rdnw * (phw[1:] - phw[:-1])) / mass
        return al, c2a * (alt * (tw - g.c1h * mw * t1) / (mass * (T0 + t1)) - al)

    al, pw = p_rho(mu_work, g.mh(muts), origin["theta"] - T0, tw, phw)
    pm1 = pw

    # column setup: rw_tend, ph_tend and the implicit coefficients
    mx = g.msftx / g.msfty
    ru_f, rv_f = g.mh(muu) * u / g.msfuy, g.mh(muv) * v / g.msfvx
    ru_m, u_m, rv_m, v_m = (g.to_faces(mean2(q, d)) for q, d in ((ru_f, -1), (u, -1), (rv_f, -2), (v, -2)))
    rw_t = wt.clone()
    curv = (ru_m * u_m + mx * rv_m * v_m) / 6370.0e3
    if g.rotating:
        curv = curv + g.e * (g.cosa * ru_m - mx * g.sina * rv_m)
    mp = mut - mub
    rw_t[1:-1] += (G / g.msfty) * (cq1 * g.rdn[1:] * (pp[1:] - pp[:-1]) - g.c1f[1:-1] * mp - cq2 * g.mf(mub)[1:-1]) + curv
    c1t, c2t = (cq1[-1], cq2[-1]) if nl.moist else (1.0, 0.0)
    rw_t[-1] += (G / g.msfty) * (-c1t * 2.0 * g.rdnw[-1] * pp[-1] - g.c1f[-1] * mp - c2t * g.mf(mub)[-1])
    ph_t = torch.zeros_like(w)
    wd = 0.5 * (rom[1:] + rom[:-1]) * g.rdnw * (ph[1:] - ph[:-1])
    t = -g.to_faces(wd) + g.mf(mut)[1:-1] * G * w[1:-1] / g.msfty
    fi = ph[1:-1]
    gy = g.mf(muv)[1:-1] * (v[1:] + v[:-1])
    gx = g.mf(muu)[1:-1] * (u[1:] + u[:-1])
    t = t - 0.25 * g.rdy / g.msfty * (gy[:, 1:] * (_y(fi, 1) - fi) + gy[:, :-1] * (fi - _y(fi, -1)))
    t = t - 0.25 * g.rdx / g.msfty * (gx[..., 1:] * (_x(fi, 1) - fi) + gx[..., :-1] * (fi - _x(fi, -1)))
    ph_t[1:-1] = t
    cof = (0.5 * dts * G * (1.0 + nl.epssm)) ** 2
    mh, mf = g.mh(mut).expand(th.shape), g.mf(mut).expand(w.shape)
    a = torch.zeros_like(w)
    a[2:-1] = (-cq1 * cof * g.rdn[1:] * g.rdnw[:-1] * c2a[:-1] / (mh[:-1] * mf[:-2]))[1:]
    b = 1.0 + cq1 * cof * g.rdn[1:] * (g.rdnw[1:] * c2a[1:] / (mh[1:] * mf[1:-1]) + g.rdnw[:-1] * c2a[:-1] / (mh[:-1] * mf[1:-1]))
    c = -cq1 * cof * g.rdn[1:] * g.rdnw[1:] * c2a[1:] / (mh[1:] * mf[2:])
    gamma = torch.zeros_like(w)
    alpha = torch.ones_like(w)
    for k in range(1, nz):
        alpha[k] = 1.0 / (b[k - 1] - a[k] * gamma[k - 1])
        gamma[k] = c[k - 1] * alpha[k]
    top = 2.0 * cof * g.rdnw[-1] ** 2 * c2a[-1] / (mh[-1] * mf[-1])
    alpha[nz] = 1.0 / (1.0 + top)
    omega = rom.clone()  # carried ends

    # acoustic substeps
    mudf = s["mudf"]
    t2 = torch.zeros_like(th)
    ep, em = 1.0 + nl.epssm, 1.0 - nl.epssm
    ht = phb[0] / G

    def terrain(q, dim, face, msf, rd):
        hp = torch.cat([q.narrow(dim, 0, 1), q, q.narrow(dim, q.shape[dim] - 1, 1)], dim)
        d = hp.narrow(dim, 1, hp.shape[dim] - 1) - hp.narrow(dim, 0, hp.shape[dim] - 1)
        low = cf1 * face[0] + cf2 * face[1] + cf3 * face[2]
        flux = d * low
        return msf * 0.5 * rd * (flux.narrow(dim, 1, flux.shape[dim] - 1) + flux.narrow(dim, 0, flux.shape[dim] - 1))

    w_sfc = terrain(ht, -2, v, g.msfty, g.rdy) + terrain(ht, -1, u, g.msftx, g.rdx)
    theta1 = th - T0
    for _ in range(nsub):
        def pgf(pad, dim, msf, rd, mass):
            def lr(q):
                q = pad(q)
                return q.narrow(dim, 0, q.shape[dim] - 1), q.narrow(dim, 1, q.shape[dim] - 1)

            (pl, pr), (hl, hr), (tl, tr), (al_, ar_) = lr(pw), lr(phw), lr(alt), lr(al)
            (bl, br), (fl, fr), (ml, mr) = lr(pb), lr(php_h), lr(muts - mut)
            ps = pl + pr
            dpn = torch.cat([0.5 * (cf1 * ps[:1] + cf2 * ps[1:2] + cf3 * ps[2:3]), 0.5 * g.to_faces(ps),
                             0.5 * (cf1 * ps[-1:] + cf2 * ps[-2:-1] + cf3 * ps[-3:-2])])
            d = hr - hl
            grad = msf * 0.5 * rd * mass * ((d[1:] + d[:-1]) + (tl + tr) * (pr - pl) + (al_ + ar_) * (br - bl))
            return grad + msf * rd * (fr - fl) * (g.rdnw * (dpn[1:] - dpn[:-1]) - 0.5 * g.c1h * (ml + mr))

        dm = _pad_x(mudf)
        uw = uw + dts * ut - dts * cqu * pgf(_pad_x, -1, msf_u, g.rdx, g.mh(muu)) + g.c1h * (-0.01 * g.dx * (dm[:, 1:] - dm[:, :-1]) / g.msfuy)
        dm = _pad_y(mudf)
        vw = vw + dts * vt - dts * cqv * pgf(_pad_y, -2, msf_v, g.rdy, g.mh(muv)) + g.c1h * (-0.01 * g.dy * (dm[1:] - dm[:-1]) / g.msfvx)
        # mass, omega, theta
        uf, vf = uw + g.mh(muu) * u / g.msfuy, vw + g.mh(muv) * v / g.msfvx
        dv = g.msftx * g.msfty * (g.rdy * (vf[:, 1:] - vf[:, :-1]) + g.rdx * (uf[..., 1:] - uf[..., :-1]))
        dmdt = (g.dnw * dv).sum(0)
        mw_old = muts - mut
        mw = mw_old + dts * dmdt
        mu_c = mu_c - mw_old + mw
        mudf, muts = dmdt, mut + mw
        muave = 0.5 * (ep * mw + em * mw_old)
        run_ = omega[0] - torch.cumsum(g.dnw * (g.c1h * dmdt + dv) / g.msfty, 0)
        omega = torch.cat([(omega[0] - rom[0])[None], run_[:-1] - rom[1:-1], omega[-1:]])
        wd = torch.zeros_like(w)
        wd[1:-1] = omega[1:-1] * g.to_faces(theta1)
        v_fl = vw[:, 1:] * (_y(theta1, 1) + theta1) - vw[:, :-1] * (theta1 + _y(theta1, -1))
        u_fl = uw[..., 1:] * (_x(theta1, 1) + theta1) - uw[..., :-1] * (theta1 + _x(theta1, -1))
        tend = g.msftx * (0.5 * g.rdy * v_fl + 0.5 * g.rdx * u_fl) + g.rdnw * (wd[1:] - wd[:-1])
        tw = tw + g.msfty * dts * tt - dts * g.msfty * tend
        t2 = (0.5 * (ep * tw + em * t2) + g.c1h * muave * T0) / (g.mh(muts) * th)
        # implicit w and phi
        rhs = torch.zeros_like(w)
        om = 0.5 * (omega[1:] + omega[:-1]) * g.rdnw * (ph1[1:] - ph1[:-1])
        rr = dts * (ph_t + 0.5 * G * em * ww)
        rr[1:-1] -= dts * g.to_faces(om)
        rhs[1:-1] = phw[1:-1] + g.msfty * rr[1:-1] / mf[1:-1]
        x = torch.zeros_like(w)
        x[0] = w_sfc
        rw = rw_t[1:-1]
        if nl.w_damping == 1:
            cfl = (omega[1:-1] / mf[1:-1] * g.rdnw[1:] * dts).abs()
            rw = rw + torch.where(cfl > 1.0, -torch.sign(ww[1:-1]) * 0.3 * (cfl - 1.0) * mf[1:-1], torch.zeros_like(cfl))
        coef = c2a * g.rdnw / mh
        ta = coef * (ep * (rhs[1:] - rhs[:-1]) + em * (phw[1:] - phw[:-1]))
        buoy = c2a * alt * t2
        x[1:-1] = (ww[1:-1] + dts * rw + cq1 / g.msfty * 0.5 * dts * G * g.rdn[1:] * (ta[1:] - ta[:-1])
                   + dts * G / g.msfty * (g.rdn[1:] * (buoy[1:] - buoy[:-1]) - g.c1f[1:-1] * muave))
        for k in range(1, nz + 1):
            x[k] = (x[k] - a[k] * x[k - 1]) * alpha[k]
        for k in range(nz - 1, 0, -1):
            x[k] = x[k] - gamma[k] * x[k + 1]
        if nl.damp_opt == 3 and nl.dampcoef > 0.0:
            hk = ph1 / G
            bottom = hk[-1] - nl.zdamp
            wgt = torch.where(hk >= bottom, dts * nl.dampcoef * torch.sin(0.5 * math.pi * (hk - bottom) / nl.zdamp) ** 2,
                              torch.zeros_like(hk))
            x[1:] = ((x - wgt * mf * w) / (1.0 + wgt))[1:]
        mft = g.mf(muts)
        phw = torch.cat([phw[:1], (rhs + g.msfty * 0.5 * dts * G * ep * x / mft)[1:]])
        ww = x
        al, pnew = p_rho(muts - mut, g.mh(muts), theta1, tw, phw)
        pw = pnew + 0.1 * (pnew - pm1)
        pm1 = pnew

    # finish
    s["u"] = (g.msfuy * uw + u * g.mh(muu)) / g.mh(muus)
    s["v"] = (g.msfvx * vw + v * g.mh(muv)) / g.mh(muvs)
    s["w"] = (g.msfty * ww + w * g.mf(mut)) / g.mf(muts)
    php = php + phw
    s["ph_perturbation"], s["ph_total"] = php, phb + php
    th = (tw + theta1 * g.mh(mut)) / g.mh(muts) + T0
    if nl.hypsometric_opt == 2:
        spec = _log_alpha(g, s["ph_total"][1:] - s["ph_total"][:-1], mub + mu_c)
    else:
        alb = -(phb[1:] - phb[:-1]) / (g.dnw * g.mh(mub))
        spec = alb - (alb * g.c1h * mu_c + g.rdnw * (php[1:] - php[:-1])) / g.mh(mub + mu_c)
    total = P0 * (RD * th / (P0 * spec)) ** CPOVCV
    s["theta"], s["p_perturbation"], s["p_total"] = th, total - pb, pb + (total - pb)
    s["mu_perturbation"], s["mu_total"], s["mudf"] = mu_c, mub + mu_c, mudf
    for q, tend in qt.items():
        s[q] = (g.mh(origin["mu_total"]) * origin[q] + dt_rk * tend) / g.mh(s["mu_total"])
