"""The work that users of penguin_amd have it do, as cases to be timed.

A case is one pass through the public entry points (``Disk``, ``Batch``): a
number of steps from the present state, then the state read back, which is
what a program does between two output frames; or the gradient of a loss on
the final state.  Frames are kept in the disk's own storage precision, as an
FP32 disk holds no more.  Sizes are those of the repository's configurations
and tests, and generic ones between and around them.

``exact`` integrates the two-dimensional disk in 64-bit torch, written from
the equations of the scheme, with the arithmetic of this file alone.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from penguin_amd import Batch, Disk, batch_configs, disk2d, disk3d


# ------------------------------------------------------------------- cases
def listed():
    return [
        # the smallest grids (parameter scans, tests): launches and latency only
        dict(name="small-64x128", kind="run", nr=64, nphi=128, precision=4, dust=False, kill=False, visc=True,
             graph=True, steps=400),
        # the plain method on its small disk, 256 x 512 gas
        dict(name="gas-256x512", kind="run", nr=256, nphi=512, precision=4, dust=False, kill=False, visc=True,
             graph=True, steps=400),
        # the same disk driven from the host as the reference's main loop
        # drives it: global_dt, solve, one call each per step
        dict(name="hostloop-256x512", kind="host", nr=256, nphi=512, precision=4, dust=False, kill=False, visc=True,
             steps=40),
        # odd and ragged in both directions, reference precision, no captured step
        dict(name="odd-333x777-fp64", kind="run", nr=333, nphi=777, precision=8, dust=True, kill=False, visc=True,
             graph=False, steps=100),
        # an inviscid disk (the other sequence of passes), ragged
        dict(name="inviscid-500x1300", kind="run", nr=500, nphi=1300, precision=4, dust=False, kill=True, visc=False,
             graph=True, steps=200),
        # the benchmark's disk: gas and dust, wave killing
        dict(name="gasdust-1024x3072", kind="run", nr=1024, nphi=3072, precision=4, dust=True, kill=True, visc=True,
             graph=True, steps=400),
        # and the same at the reference's precision
        dict(name="gasdust-1024x3072-fp64", kind="run", nr=1024, nphi=3072, precision=8, dust=True, kill=True,
             visc=True, graph=True, steps=150),
        # many uneven disks advanced together
        dict(name="batch-24", kind="batch", disks=24, precision=4, steps=300),
        # gradient of the gap-opening loss, checkpoints every 20 steps (FP64,
        # the precision in which gradients are held to finite differences)
        dict(name="adjoint-512x1024", kind="adjoint", nr=512, nphi=1024, precision=8, steps=60, ckpt=20),
        # the three-dimensional disk: its full size, an ordinary one, a small
        # one with the other reconstruction at the reference's precision
        dict(name="sph-384x1536x64", kind="sph", nr=384, nphi=1536, ntheta=64, precision=4, recon=5, steps=60),
        dict(name="sph-96x384x64", kind="sph", nr=96, nphi=384, ntheta=64, precision=4, recon=5, steps=60),
        dict(name="sph-40x64x16-fp64", kind="sph", nr=40, nphi=64, ntheta=16, precision=8, recon=6, steps=60),
    ]


def _spread(rng, lo, hi):
    """A whole number between lo and hi, even in its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run"] * 5 + ["host", "batch", "adjoint", "sph", "sph"])
    precision = rng.choice([4, 4, 8])
    if kind in ("run", "host"):
        dust = rng.random() < 0.5
        c = dict(kind=kind, nr=_spread(rng, 48, 1100), nphi=_spread(rng, 64, 3000), precision=precision, dust=dust,
                 kill=rng.random() < 0.5, visc=rng.random() < 0.8)
        if kind == "run":
            c.update(graph=rng.random() < 0.7, steps=_spread(rng, 60, 300))
        else:
            c.update(steps=_spread(rng, 10, 60))
        return c
    if kind == "batch":
        return dict(kind=kind, disks=_spread(rng, 3, 20), precision=precision, steps=_spread(rng, 30, 200))
    if kind == "adjoint":
        return dict(kind=kind, nr=_spread(rng, 64, 512), nphi=_spread(rng, 96, 1024), precision=8,
                    steps=_spread(rng, 20, 60), ckpt=rng.choice([0, 10, 20]))
    return dict(kind=kind, nr=_spread(rng, 24, 200), nphi=_spread(rng, 48, 512), ntheta=_spread(rng, 8, 72),
                precision=precision, recon=rng.choice([5, 5, 6]), steps=_spread(rng, 10, 60))


def _physics(seed):
    """Planet mass, viscosity and aspect ratio of a case's disk, from the seed
    (the ranges of the batched workload)."""
    rng = np.random.default_rng(seed)
    return dict(planet_mass=float(10.0 ** rng.uniform(-4.5, -3.3)), ss_alpha=float(10.0 ** rng.uniform(-3.5, -2.5)),
                sc_h=float(rng.uniform(0.04, 0.07)), seed=int(seed))


def _params(case, seed):
    if case["kind"] == "sph":
        kw = _physics(seed)
        kw["ss_alpha"] *= 0.1
        h = kw["sc_h"]
        return disk3d(case["nr"], case["nphi"], case["ntheta"], precision=case["precision"], recon_flag=case["recon"],
                      zmin=0.5 * math.pi - 3.0 * h, zmax=0.5 * math.pi + 3.0 * h, **kw)
    p = disk2d(case["nr"], case["nphi"], precision=case["precision"], **_physics(seed))
    p.dust_flag = int(case.get("dust", False))
    p.kill_flag = int(case.get("kill", False))
    p.visc_flag = int(case.get("visc", True))
    p.noise_vr = 1.0e-4 if p.dust_flag else 0.0
    return p


def _batch_params(case, seed):
    """The batched workload's uneven grids, with physics and noise from the seed."""
    own = batch_configs(case["disks"], seed=seed)
    return [p.replace(planet_mass=q.planet_mass, ss_alpha=q.ss_alpha, sc_h=q.sc_h, seed=q.seed)
            for p, q in zip(batch_configs(case["disks"], seed=1, precision=case["precision"]), own)]


def _gap_target(p):
    """Radial density profile with a Gaussian gap at the planet."""
    i = np.arange(p.xres + 1, dtype=np.float64)
    xa = p.xmin * np.exp(np.log(p.xmax / p.xmin) * i / p.xres)
    r = 0.5 * (xa[1:] + xa[:-1])
    return r ** (-p.p_alpha) * (1.0 - 0.5 * np.exp(-((r - 1.0) ** 2) / (2.0 * (2.0 * p.sc_h) ** 2)))


# ----------------------------------------------------------- prepare and run
def prepare(case, seed):
    """The disk (or batch) a program holds: created with its seeded initial state."""
    s = dict(case=case)
    if case["kind"] == "batch":
        s["batch"] = Batch(_batch_params(case, seed))
        return s
    p = _params(case, seed)
    s["disk"] = Disk(p)
    if case["kind"] == "adjoint":
        s["target"] = _gap_target(p)
    return s


def _kept(a, precision):
    """An array as a program keeps it: in the disk's storage precision."""
    t = torch.from_numpy(np.asarray(a, dtype=np.float64))
    return t.to(torch.float32) if precision == 4 else t


def run(s):
    case = s["case"]
    prec = case["precision"]
    kind = case["kind"]
    if kind == "batch":
        b = s["batch"]
        dts = b.run(case["steps"])
        gas = [_kept(b.get_state(k)[0], prec).reshape(5, -1) for k in range(b.n)]
        return dict(dts=_kept(dts, prec), gas=torch.cat(gas, dim=1))
    d = s["disk"]
    if kind == "adjoint":
        dts = d.adjoint_forward(case["steps"], case["ckpt"])
        gas, _ = d.get_state()
        dL = np.zeros_like(gas)
        dL[0] = 2.0 * (gas[0].mean(axis=0) - s["target"]) / d.ny
        dq, dalpha, d0 = d.adjoint_backward(dL)
        return dict(dts=_kept(dts, prec), gas=_kept(gas, prec), dq=_kept(dq, prec), dalpha=_kept(dalpha, prec),
                    dstate0=_kept(d0, prec))
    if kind == "host":
        dts = np.array([d.step_host() for _ in range(case["steps"])])
    else:
        dts = d.run(case["steps"], use_graph=bool(case.get("graph", False)))
    gas, dust = d.get_state()
    out = dict(dts=_kept(dts, prec), gas=_kept(gas, prec))
    if dust is not None:
        out["dust"] = _kept(dust, prec)
    return out


# --------------------------------------------------------------------- work
def work(case):
    """State read and written once a step (the adjoint: the forward step, its
    recompute and the transposed step) and the frame returned; operations
    counted from the scheme's formulas per cell and step (gas 2D 900, dust
    350, viscosity 200, transposed step 2500, 3D step 2600)."""
    word = case["precision"]
    if case["kind"] == "batch":
        cells, fields, out, flops = _batch_cells(case), 3, 5, 1100
    elif case["kind"] == "sph":
        cells, fields, out, flops = case["nr"] * case["nphi"] * case["ntheta"], 5, 5, 2600
    else:
        cells = case["nr"] * case["nphi"]
        fields, out, flops = 3, 5, 900 + (200 if case.get("visc", True) else 0)
        if case.get("dust"):
            fields, out, flops = 6, 9, flops + 350
        if case["kind"] == "adjoint":
            fields, out, flops = 3 * fields, 10, 2 * flops + 2500
    return {"bytes": float(cells) * (2 * fields * word * case["steps"] + out * 8),
            "flops": float(cells) * flops * case["steps"]}


def _batch_cells(case):
    return sum(int(p.xres) * int(p.yres) for p in _batch_params(case, 1))


# -------------------------------------------------------------------- exact
def exact(case, seed):
    """What run returns, from the 64-bit integration below; None for the
    three-dimensional disk (no such integration here), for gradients, and
    where the steps would take too long."""
    if case["kind"] == "sph":
        return None
    if not torch.cuda.is_available():
        return None
    if case["kind"] == "batch":
        ps = _batch_params(case, seed)
        if case["disks"] * case["steps"] > 3000:
            return None
        dts, gas = [], []
        for p in ps:
            dt, g, _ = _integrate(p, case["steps"])
            dts.append(dt)
            gas.append(g.reshape(5, -1))
        return dict(dts=torch.stack(dts), gas=torch.cat(gas, dim=1))
    dts, gas, dust = _integrate(_params(case, seed), case["steps"])
    out = dict(dts=dts, gas=gas)
    if dust is not None:
        out["dust"] = dust
    if case["kind"] == "adjoint":
        out.update(dq=None, dalpha=None, dstate0=None)
    return out


def _unit(seed, field, ny, nx):
    """Uniform numbers keyed by (seed, field, cell): SplitMix64."""
    def mix(x):
        x = x + np.uint64(0x9E3779B97F4A7C15)
        x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return x ^ (x >> np.uint64(31))

    with np.errstate(over="ignore"):
        j, i = np.meshgrid(np.arange(ny, dtype=np.uint64), np.arange(nx, dtype=np.uint64), indexing="ij")
        key = mix(np.full(1, seed, dtype=np.uint64)) ^ mix((np.uint64(field) << np.uint64(48)) ^ (j << np.uint64(24)) ^ i)
        return (mix(key) >> np.uint64(11)).astype(np.float64) / 9007199254740992.0


def _weights(edges, radial):
    """Slopes (mean - left value, right value - mean) of the middle one of
    five cells as linear maps of their mean differences: the cubic through
    the means of four cells, in lengths of the middle cell about its centre."""
    h = edges[3] - edges[2]
    x0 = 0.5 * (edges[2] + edges[3])
    y = (np.asarray(edges) - x0) / h
    a = x0 / h if radial else None

    def integral(k, v):   # of y^k, weighted by the radius if radial
        return v ** (k + 1) / (k + 1) if a is None else v ** (k + 2) / (k + 2) + a * v ** (k + 1) / (k + 1)

    mean = np.array([[(integral(k, y[c + 1]) - integral(k, y[c])) / (integral(0, y[c + 1]) - integral(0, y[c]))
                      for k in (1, 2, 3)] for c in range(5)])
    left = np.array([y[2], y[2] ** 2, y[2] ** 3])
    right = np.array([y[3], y[3] ** 2, y[3] ** 3])
    lo = np.linalg.inv(mean[1:4] - mean[0:3])
    hi = np.linalg.inv(mean[2:5] - mean[1:4])
    return (mean[2] - left) @ lo, (right - mean[2]) @ hi


def _slopes(d0, d1, d2, d3, wl, wr, flat):
    l = wl[0] * d0 + wl[1] * d1 + wl[2] * d2
    r = wr[0] * d1 + wr[1] * d2 + wr[2] * d3
    l = torch.copysign(torch.minimum(l.abs(), d1.abs()), d1)
    r = torch.copysign(torch.minimum(r.abs(), d2.abs()), d2)
    off = (r * l <= 0) * 1.0
    l, r = l * (1.0 - off) * (1.0 - flat), r * (1.0 - off) * (1.0 - flat)
    t2, t1 = (l + r) ** 2, 3.0 * (l + r) * (l - r)
    return torch.where(t2 < t1, 2.0 * r, l), torch.where((t2 >= t1) & (t2 < -t1), 2.0 * l, r)


def _flat(p, u, ax):
    """Flattening of cells 2 .. n-3 along axis ax."""
    n = p.shape[ax]
    at = lambda f, k: f.narrow(ax, 2 + k, n - 4)  # noqa: E731
    fb, ff = at(p, 0) - at(p, -1), at(p, 1) - at(p, 0)
    wb, wf = at(p, 1) - at(p, -2), at(p, 2) - at(p, -1)
    on = ((at(u, 0) - at(u, 1) > 0) | (at(u, -1) - at(u, 0) > 0)) & (wf != 0) & (wb != 0)
    steep = lambda a, b: 10.0 * ((a / b - 0.5).abs() - 0.25).clamp(min=0.0)  # noqa: E731
    f = torch.maximum(steep(ff, wf), steep(fb, wb)) * torch.maximum(ff.abs(), fb.abs()) / at(p, 0)
    return torch.where(on, f.clamp(max=0.5), torch.zeros_like(f))


def _parabola(f, ax, wl, wr, flat):
    """(mean - left, mean, right - mean) of cells 2 .. n-3 along axis ax."""
    n = f.shape[ax]
    d = f.narrow(ax, 1, n - 1) - f.narrow(ax, 0, n - 1)
    dd = [d.narrow(ax, k, n - 4) for k in range(4)]
    l, r = _slopes(*dd, wl, wr, flat)
    return l, f.narrow(ax, 2, n - 4), r


def _avg_l(q, P):   # mean over the cell's first fraction q
    l, a, r = P
    return (a - l) + q * ((2.0 * l - r) - q * (l - r))


def _avg_r(q, P):   # mean over its last fraction q
    l, a, r = P
    return (a + r) + q * ((l - 2.0 * r) - q * (l - r))


def _trace(avg, sign, c, dti, R, P, U, V):
    """Half-step state at a cell's edge: sign -1 its left edge, +1 its right."""
    q = ((sign * U[1]).clamp(min=0.0) + c) * dti
    w = (sign * avg(q.clamp(0.0, 1.0), U)).clamp(min=0.0)
    q = (w * dti).clamp(0.0, 1.0)
    r0, p0, u0 = avg(q, R), avg(q, P), avg(q, U)
    cs = (p0 / r0).sqrt()
    q = ((w + cs) * dti).clamp(0.0, 1.0)
    du, dp = (avg(q, U) - u0) * sign / cs, avg(q, P) - p0
    e = (1.0 + du).clamp(min=1.0e-6)
    return r0 * e, p0 * e, u0 + sign * dp / (cs * r0), avg(q, V)


def _hllc(L, R):
    (rl, pl, ul, vl), (rr, pr, ur, vr) = L, R
    cl, cr = (pl / rl).sqrt(), (pr / rr).sqrt()
    pm = 0.5 * (pl + pr) * (1.0 + (ul - ur) / (cl + cr)).clamp(min=1.0e-6)
    sl_, sr_ = rl.sqrt(), rr.sqrt()
    iss = 1.0 / (sl_ + sr_)
    ub = (sl_ * ul + sr_ * ur) * iss
    cb = ((cl * cl * sl_ + cr * cr * sr_) * iss + 0.5 * sl_ * sr_ * iss * iss * (ur - ul) ** 2).sqrt()
    sl, sr = ub - cb, ub + cb
    sm = (rl * ul * cl + rr * ur * cr) / (rl * cl + rr * cr) + 2.0 * (pl - pr) / ((cl + cr) * (rl + rr))
    left = (sl >= 0) | ((sr >= 0) & (sm >= 0))
    pick = lambda a, b: torch.where(left, a, b)  # noqa: E731
    r, p, u, v, s = pick(rl, rr), pick(pl, pr), pick(ul, ur), pick(vl, vr), pick(sl, sr)
    sup = (sl >= 0) | (sr < 0)
    F = torch.where(sup, u * r, sm * r * (s - u) / (s - sm))
    return F, u * F, v * F, torch.where(sup, p, (s * pm - sm * p) / (s - sm))


def _dust_flux(dtl, dtr, L, R):
    """Pressureless flux from the parabolas (density, normal, transverse) of
    the cells left and right of an interface; dt over the cell widths."""
    def side(avg, sign, dti, P):
        edge = P[1][1] + (P[1][2] if sign > 0 else -P[1][0])
        y = (sign * edge).clamp(min=0.0) * dti
        un = avg(y.clamp(0.0, 1.0), P[1])
        e = (1.0 + sign * dti * (P[1][1] - un) / (1.0 - y)).clamp(min=1.0e-6)
        q = ((sign * un).clamp(min=0.0) * dti).clamp(0.0, 1.0)
        r, u, v = avg(q, P[0]) * e, avg(q, P[1]), avg(q, P[2])
        return sign * torch.minimum(P[0][1] * dti, (sign * u * r).clamp(min=0.0)), u, v

    a, ul, vl = side(_avg_r, 1.0, dtl, L)
    b, ur, vr = side(_avg_l, -1.0, dtr, R)
    return a + b, a * ul + b * ur, a * vl + b * vr


class _Grid:
    """Radial tables with three ghost cells a side, and the azimuthal grid."""

    def __init__(self, p, dev):
        nx, ny = int(p.xres), int(p.yres)
        self.nx, self.ny, self.p, self.dev = nx, ny, p, dev
        xa = p.xmin * np.exp(np.log(p.xmax / p.xmin) * (np.arange(nx + 7) - 3.0) / nx)
        x = 0.5 * (xa[1:] + xa[:-1])
        rp, a = p.planet_radius, p.p_alpha
        cs2 = lambda r: p.sc_h**2 / rp * (r / rp) ** (-p.p_beta)  # noqa: E731
        rho = lambda r: (r / rp) ** (-a)  # noqa: E731
        nu = np.zeros_like(x)
        if p.visc_flag:
            nu = p.ss_alpha * math.sqrt(cs2(rp)) * math.sqrt(cs2(rp) * rp**3) * (x / rp) ** a
        dr = 1.1514178e-7
        dpdr = (cs2(x + dr) * rho(x + dr) - cs2(x - dr) * rho(x - dr)) / (2.0 * dr)
        v = np.sqrt(1.0 / x + x / rho(x) * dpdr)
        up = lambda z: torch.tensor(z, dtype=torch.float64, device=dev)  # noqa: E731
        self.xa, self.x, self.cs2, self.c = up(xa), up(x), up(cs2(x)), up(np.sqrt(cs2(x)))
        self.vol, self.dx = up(0.5 * (xa[1:] ** 2 - xa[:-1] ** 2)), up(xa[1:] - xa[:-1])
        self.v, self.nu, self.rho, self.u = up(v), up(nu), up(rho(x)), up(-1.5 * nu / x)
        w = [_weights(xa[c - 2:c + 4], True) for c in range(2, nx + 4)]
        self.wl, self.wr = up(np.array([q[0] for q in w]).T.copy()), up(np.array([q[1] for q in w]).T.copy())
        self.yl, self.yr = _weights(np.arange(6.0), False)
        self.dy = (p.ymax - p.ymin) / ny
        self.phi = up(((np.arange(ny) + 0.5) * self.dy + p.ymin)[:, None])
        self.R = self.x[3:-3]
        self.rot = self.v[3:-3] - self.R * p.frame_omega
        self.ts = p.Stokes * p.sc_h / self.c[3:-3]
        self.ghost_gas = (self.rho, self.u, self.v)
        if p.dust_flag:
            St = p.Stokes
            fg = v / np.sqrt(1.0 / x)
            b = St * St * fg
            L = (1.0 + b) / b * (1.0 - np.sqrt(1.0 - 2.0 * b * (1.0 - fg) / (1.0 + b) ** 2))
            u0 = St * (L * L - 2.0 * L)
            w_ = (1.0 - np.sqrt(1.0 - 2.0 * St * u0)) / St
            L = (1.0 - fg + St * w_ / 2.0) / (1.0 + St * w_ / 2.0)
            u0 = St * (L * L - 2.0 * L)
            w_ = (1.0 - np.sqrt(1.0 - 2.0 * St * u0)) / St
            self.ghost_dust = (up(p.D_G_ratio * rho(x)), up(w_ * np.sqrt(1.0 / x)), up(np.sqrt(1.0 / x)))
        kill = np.zeros(nx)
        if p.kill_flag:
            h = lambda r: math.sqrt(cs2(r) * r**3)  # noqa: E731
            di, do = h(p.xmin) * p.kill_width, h(p.xmax) * p.kill_width
            d = np.maximum((p.xmin + di - x[3:-3]) / di, (x[3:-3] - (p.xmax - do)) / do)
            kill = np.where(d > 0, np.sin((0.5 * np.pi * d).astype(np.float32)).astype(np.float64) ** 2, 0.0)
            kill = kill / x[3:-3] ** 1.5
        self.kill = up(kill)

    def pad(self, S, ghost):
        """Radial ghosts: the initial disk."""
        g = [f.expand(self.ny, -1) for f in ghost]
        return [torch.cat((q[:, :3], f, q[:, -3:]), dim=1) for f, q in zip(S, g)]

    def planet(self, t):
        """Planet pull on every cell (radial, azimuthal) at time t: circular
        orbit in the rotating frame, its mass ramped, with the indirect term."""
        p = self.p
        if p.n_planet == 0:
            return 0.0, 0.0
        m = p.planet_mass * (math.sin(0.5 * math.pi * t / p.ramp_time) if t < p.ramp_time else 1.0)
        a, rs = p.planet_radius, p.rs_fac * p.sc_h * p.planet_radius
        ang = math.fmod(math.sqrt(1.0 / a**3) * t, 2 * math.pi) - math.fmod(p.frame_omega * t, 2 * math.pi) + math.pi
        s, c = torch.sin(self.phi - ang), torch.cos(self.phi - ang)
        k = ((self.R - a) ** 2 + 4.0 * a * self.R * torch.sin(0.5 * (self.phi - ang)) ** 2 + rs**2) ** -1.5
        return -m * (self.R - a * c) * k - c * m / a**2, -m * a * s * k + s * m / a**2

    def viscous(self, S):
        """Divergence of the viscous stress, radial and azimuthal."""
        r, u, v = [f[:, 2:-2] for f in self.pad(S, self.ghost_gas)]
        n = r * self.nu[2:-2]
        x = self.x[2:-2]
        i20, i21, i10 = 1.0 / (x[2:] - x[:-2]), 1.0 / (x[2:] - x[1:-1]), 1.0 / (x[1:-1] - x[:-2])
        R, dy = self.R, self.dy
        mid = lambda f: f[:, 1:-1]  # noqa: E731
        d1 = lambda f: (f[:, 2:] - f[:, :-2]) * i20  # noqa: E731
        d2 = lambda f: ((f[:, 2:] - mid(f)) * i21 - (mid(f) - f[:, :-2]) * i10) * 2.0 * i20  # noqa: E731
        e1 = lambda f: (f.roll(-1, 0) - f.roll(1, 0)) / (2.0 * dy)  # noqa: E731
        e2 = lambda f: (f.roll(-1, 0) - 2.0 * f + f.roll(1, 0)) / dy**2  # noqa: E731
        n1, u1, v1 = mid(n), mid(u), mid(v)
        ux, uy, uxx, uyy, uxy = d1(u), mid(e1(u)) / R, d2(u), mid(e2(u)) / R**2, d1(e1(u)) / R
        vx, vy, vxx, vyy, vxy = d1(v), mid(e1(v)) / R, d2(v), mid(e2(v)) / R**2, d1(e1(v)) / R
        nx_, ny_ = d1(n), mid(e1(n)) / R
        t = uy + vx - v1 / R
        fx = 2 * nx_ * ux + 2 * n1 * uxx + ny_ * t + n1 * (uyy + vxy) + (2 * n1 * ux - n1 * vy - 2 * n1 * (vy + u1 / R)) / R
        fy = (2 * ny_ * (vy + u1 / R) + 2 * n1 * vyy + nx_ * t + n1 * (uxy + vxx) +
              (2 * n1 * uy - n1 * vx + n1 * v1 / R + 2 * n1 * t) / R)
        return fx, fy

    def kick(self, S, D, V, pull, h, middle):
        """Source terms over h; with `middle` the forces at the state predicted over h."""
        r, u, v = S
        px, py = pull
        vx, vy = (V[0] / r, V[1] / r) if V is not None else (0.0, 0.0)
        acc = lambda w: w * w / self.R - 1.0 / self.R**2 + px  # noqa: E731
        tu, tv = u, v
        if middle:
            tu, tv = u + (acc(v) + vx) * h, v + (vy + py) * h
        new = [r, u + (acc(tv) + vx) * h, v + (vy + py) * h]
        if D is None:
            return new, None
        q, du, dv = D
        ts = self.ts / r
        k = -torch.expm1(-h / ts)
        dm = dv + (v - dv + py * ts) * k if middle else dv
        return new, [q, du + (acc(dm) * ts + tu - du) * k, dv + (tv - dv + py * ts) * k]

    def sweep_x(self, S, dt):
        r, u, v = self.pad(S, self.ghost_gas)
        p, L = r * self.cs2, v * self.x
        f = _flat(p, u, 1)
        P = [_parabola(q, 1, self.wl, self.wr, f) for q in (r, p, u, L)]
        lo = [tuple(z[:, :-1] for z in q) for q in P]
        hi = [tuple(z[:, 1:] for z in q) for q in P]
        c, dti = self.c[2:-2], dt / self.dx[2:-2]
        F, Fu, FL, ps = _hllc(_trace(_avg_r, 1.0, c[:-1], dti[:-1], *lo), _trace(_avg_l, -1.0, c[1:], dti[1:], *hi))
        g = self.xa[3:-3]
        dif = lambda a: (a[:, :-1] - a[:, 1:]) * dt / self.vol[3:-3]  # noqa: E731
        D = dif(F * g)
        Du = dif(Fu * g) + 0.5 * (g[:-1] + g[1:]) * dif(ps)
        r0, u0, v0 = r[:, 3:-3], u[:, 3:-3], v[:, 3:-3]
        rn = r0 + D
        return [rn, (r0 * u0 + Du) / rn, (r0 * v0 + dif(FL * g) / self.R) / rn]

    def sweep_x_dust(self, S, dt):
        r, u, v = self.pad(S, self.ghost_dust)
        P = [_parabola(q, 1, self.wl, self.wr, 0.0) for q in (r, u, v * self.x)]
        lo = [tuple(z[:, :-1] for z in q) for q in P]
        hi = [tuple(z[:, 1:] for z in q) for q in P]
        dti = dt / self.dx[2:-2]
        g = self.xa[3:-3]
        D, Du, DL = [(a[:, :-1] - a[:, 1:]) * dt / self.vol[3:-3]
                     for a in (f * g for f in _dust_flux(dti[:-1], dti[1:], lo, hi))]
        r0, u0, v0 = r[:, 3:-3], u[:, 3:-3], v[:, 3:-3]
        rn = r0 + D
        return [rn, (r0 * u0 + Du) / rn, (r0 * v0 + DL / self.R) / rn]

    def wrap(self, f, k):
        j = torch.arange(-k, self.ny + k, device=self.dev) % self.ny
        return f[j]

    def sweep_y(self, S, dt, dust):
        vb = self.v[3:-3]
        r, u, w = [self.wrap(f, 3) for f in (S[0], S[1], S[2] - vb)]
        cs2 = self.cs2[3:-3]
        f = 0.0 if dust else _flat(r, w, 0)
        P = [_parabola(q, 0, self.yl, self.yr, f) for q in (r, w, u)]
        lo = [tuple(z[:-1] for z in q) for q in P]
        hi = [tuple(z[1:] for z in q) for q in P]
        dti = dt / (self.R * self.dy)
        dif = lambda a: (a[:-1] - a[1:]) * dti  # noqa: E731
        if dust:
            D, Dw, Du = [dif(q) for q in _dust_flux(dti, dti, lo, hi)]
        else:
            pl, ph = tuple(cs2 * z for z in lo[0]), tuple(cs2 * z for z in hi[0])
            c = self.c[3:-3]
            F, Fw, Fu, ps = _hllc(_trace(_avg_r, 1.0, c, dti, lo[0], pl, lo[1], lo[2]),
                                  _trace(_avg_l, -1.0, c, dti, hi[0], ph, hi[1], hi[2]))
            D, Dw, Du = dif(F), dif(Fw) + dif(ps), dif(Fu)
        r0, u0, w0 = r[3:-3], u[3:-3], w[3:-3]
        rn = r0 + D
        return [rn, (r0 * u0 + Du) / rn, (r0 * w0 + Dw) / rn + vb]

    def advect(self, S, dt):
        """Orbital advection: the whole-cell shift, then the residual."""
        arc = self.R * self.dy
        shift = torch.floor(self.rot * dt / arc + 0.5)
        speed = self.rot - shift * arc / dt
        j = (torch.arange(self.ny, device=self.dev)[:, None] - shift.long()[None, :]) % self.ny
        vb = self.v[3:-3]
        r, u, w = [self.wrap(f.gather(0, j), 3) for f in (S[0], S[1], S[2] - vb)]
        P = [_parabola(q, 0, self.yl, self.yr, 0.0) for q in (r, u, w)]
        q = (speed.abs() * dt / arc).clamp(0.0, 1.0)
        m = [torch.where(speed > 0, _avg_r(q, tuple(z[:-1] for z in f)), _avg_l(q, tuple(z[1:] for z in f))) for f in P]
        D, Du, Dw = [(a[:-1] - a[1:]) * (speed * dt / arc) for a in (m[0], m[1] * m[0], m[2] * m[0])]
        r0, u0, w0 = r[3:-3], u[3:-3], w[3:-3]
        rn = r0 + D
        return [rn, (r0 * u0 + Du) / rn, (r0 * w0 + Dw) / rn + vb]

    def rate(self, S, D):
        c, vb = self.c[3:-3], self.v[3:-3]
        sx, sy = S[1].abs() + c, (S[2] - vb).abs() + c
        if D is not None:
            sx, sy = torch.maximum(sx, D[1].abs()), torch.maximum(sy, (D[2] - vb).abs())
        return float(torch.maximum(sx / self.dx[3:-3], sy / (self.R * self.dy)).max())


def _integrate(p, steps):
    """`steps` CFL steps of the disk p from its initial state: step sizes, gas, dust."""
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    G = _Grid(p, dev)
    nx, ny = G.nx, G.ny
    S = [f[3:-3].expand(ny, nx).clone() for f in G.ghost_gas]
    if p.noise_rho:
        S[0] = S[0] * (1.0 + p.noise_rho * (2.0 * torch.tensor(_unit(p.seed, 0, ny, nx), device=dev) - 1.0))
    if p.noise_vr:
        S[1] = S[1] + p.noise_vr * G.c[3:-3] * (2.0 * torch.tensor(_unit(p.seed, 1, ny, nx), device=dev) - 1.0)
    D = [f[3:-3].expand(ny, nx).clone() for f in G.ghost_dust] if p.dust_flag else None
    t, dt, dts = 0.0, float(p.end_time), []
    for _ in range(steps):
        dt = min(p.CFL / G.rate(S, D), 1.1 * dt)
        dts.append(dt)
        h = 0.5 * dt
        V = G.viscous(S) if p.visc_flag else None
        S, D = G.kick(S, D, V, G.planet(t), h, False)
        S = G.advect(G.sweep_y(G.sweep_x(S, dt), dt, False), dt)
        if D is not None:
            D = G.advect(G.sweep_y(G.sweep_x_dust(D, dt), dt, True), dt)
        pull = G.planet(t + dt)
        if p.visc_flag:
            V = G.viscous(G.kick(S, None, V, pull, h, True)[0])
        S, D = G.kick(S, D, V, pull, h, True)
        if p.kill_flag:
            S = [f + G.kill * dt * (g[3:-3] - f) for f, g in zip(S, G.ghost_gas)]
        t += dt
    z = torch.zeros_like(S[0])
    gas = torch.stack((S[0], S[0] * G.cs2[3:-3], S[1], S[2], z))
    dust = torch.stack((D[0], D[1], D[2], z)) if D is not None else None
    return torch.tensor(dts, dtype=torch.float64, device=dev), gas, dust
