"""Timed calls of the solver: what a program that runs flow solves has it do.

A case is one output interval of a running solve (advance ``steps`` time
steps, read the progress row and the field), or one batch of requests through
the server.  The solver handle is created, loaded and started in ``prepare``,
as a program keeps it for the whole run; ``run`` continues from where the
last call stopped.  Sizes and parameters are those of this repository's
workloads, tests and decks, or reduced and ragged versions of them.

``exact`` integrates the same channel in 64 bits with plain torch array
operations (no code of this package), for the channels small enough to take
a few seconds.
"""
import math
import os
import sys

import numpy as np
import torch

if os.path.abspath("streams-2_amd") not in sys.path:
    sys.path.insert(0, os.path.abspath("streams-2_amd"))

from streams_mi355x import PREC_FP64, PREC_MIXED, make_channel  # noqa: E402
from streams_mi355x.cases import bl_recycling_case, shock_angle_from_deflection  # noqa: E402
from streams_mi355x.serve import Server  # noqa: E402
from streams_mi355x.solver import ChannelSolver  # noqa: E402


def _channel(nx, ny, nz, steps, **kw):
    return dict({"kind": "channel", "nx": nx, "ny": ny, "nz": nz, "steps": steps, "mach": 1.5, "retau": 220.0,
                 "mixed": False, "conservative": False, "bulk_t": False, "uniform_y": False}, **kw)


def listed():
    return [
        # the smoke-test grid: a user's first run, all latency and launches
        dict(_channel(32, 24, 16, 50), name="channel_32x24x16"),
        # a slice of a tuning study: thin, ragged, uniform rows, bulk-temperature control
        dict(_channel(45, 33, 21, 50, uniform_y=True, bulk_t=True), name="channel_45x33x21_bulk_t"),
        # the subsonic channel deck: conservative viscous form, Sutherland, no WENO faces
        dict(_channel(80, 60, 80, 50, mach=0.2, retau=180.0, conservative=True), name="deck_subsonic_80x60x80"),
        # the test suite's supersonic channel
        dict(_channel(128, 96, 64, 50), name="channel_128x96x64"),
        # extents that fill no tile, row or workgroup
        dict(_channel(211, 118, 77, 50, retau=180.0), name="channel_211x118x77"),
        # an ordinary supersonic production channel
        dict(_channel(256, 128, 128, 50, retau=300.0), name="channel_256x128x128"),
        # the benchmark's channel
        dict(_channel(512, 256, 256, 60, retau=550.0), name="channel_512x256x256"),
        # the mixed-precision form at a production size
        dict(_channel(256, 192, 128, 60, retau=300.0, mixed=True), name="channel_mixed_256x192x128"),
        # turbulent boundary layer with recycling inflow, spanwise statistics sampled once per interval
        {"kind": "bl", "nx": 256, "ny": 96, "nz": 64, "steps": 50, "shock": False, "mixed": False,
         "name": "boundary_layer_256x96x64"},
        # shock / boundary-layer interaction: WENO faces along the shock in every stage
        {"kind": "bl", "nx": 384, "ny": 128, "nz": 96, "steps": 40, "shock": True, "mixed": False,
         "name": "sbli_384x128x96"},
        # a burst of small independent solves through the batching server
        {"kind": "serve", "requests": 16, "side_lo": 32, "side_hi": 64, "steps": 40, "lanes": 2,
         "name": "serve_16_small"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["channel", "channel", "channel", "channel", "mixed", "conservative", "bl", "serve"])
    if kind == "serve":
        lo = rng.randrange(24, 49, 8)
        return {"kind": "serve", "requests": rng.randrange(4, 25), "side_lo": lo, "side_hi": lo + rng.randrange(16, 41, 8),
                "steps": rng.randrange(20, 61, 10), "lanes": rng.choice([0, 1, 2])}
    if kind == "bl":
        return {"kind": "bl", "nx": rng.randrange(150, 420), "ny": rng.randrange(64, 160), "nz": rng.randrange(24, 97),
                "steps": rng.randrange(20, 51), "shock": rng.random() < 0.5, "mixed": rng.random() < 0.25}
    nx, nz = _log_int(rng, 24, 400), _log_int(rng, 12, 160)
    uniform = rng.random() < 0.25
    ny = _log_int(rng, 20, 200) if uniform else 2 * _log_int(rng, 10, 100)  # the stretched grid has an even row count
    c = _channel(nx, ny, nz, rng.randrange(20, 61), retau=180.0 if ny < 64 else 220.0, uniform_y=uniform)
    if kind == "mixed":
        c["mixed"] = True
    elif kind == "conservative":
        c.update(conservative=True, mach=rng.choice([0.2, 0.5]), retau=180.0)
    else:
        c["bulk_t"] = rng.random() < 0.25
    return c


# ------------------------------------------------------------------ inputs
def _channel_case(c, seed):
    """Grid, parameters and initial field of a channel: laminar profile plus
    seeded velocity noise (10 % of the bulk velocity, 2 % in the subsonic
    deck's form)."""
    kw = dict(nx=c["nx"], ny=c["ny"], nz=c["nz"], mach=c["mach"], retau=c["retau"], seed=seed, noise_source="pcg",
              uniform_y=c["uniform_y"], precision=PREC_MIXED if c["mixed"] else PREC_FP64)
    if c["bulk_t"]:
        kw.update(theta_wall=1.0)
    if c["conservative"]:
        kw.update(conservative_viscous=1, visc_model=2, s_suth=110.4, t_ref=220.0, sensor_threshold=1.01,
                  lx=12.0, lz=6.0, dyptarget=0.7, noise=0.02, theta_wall=-2.5)
    return make_channel(**kw)


def _requests(c, seed):
    """The grids belong to the case, the flows on them to the seed."""
    shapes, rng = np.random.default_rng(c["requests"]), np.random.default_rng(seed)
    out = []
    for r in range(c["requests"]):
        side = [2 * int(shapes.integers(c["side_lo"] // 2, c["side_hi"] // 2 + 1)) for _ in range(3)]
        out.append(make_channel(nx=side[0], ny=side[1], nz=side[2], mach=float(rng.uniform(0.3, 1.5)),
                                retau=float(rng.uniform(100.0, 220.0)), seed=1000 * seed + r, noise_source="pcg"))
    return out


def prepare(case, seed):
    if case["kind"] == "serve":
        # 8 GiB hold every request of the largest burst at once
        return {"case": case, "requests": _requests(case, seed),
                "server": Server(8 << 30, max_slots=32, steps_per_graph=10, autotune=False, batch=case["lanes"])}
    if case["kind"] == "bl":
        kw = dict(shock_angle_deg=shock_angle_from_deflection(2.0, 8.0), developed_shock=True) if case["shock"] else {}
        lx = 70.0 * case["nx"] / 1024.0 if not case["shock"] else 105.0 * case["nx"] / 1536.0
        lx = max(lx, 16.0)
        c, rc = bl_recycling_case(case["nx"], case["ny"], case["nz"], lx=lx, lz=6.5 * case["nz"] / 192.0,
                                  x_recyc=0.3 * lx, xshock_imp=0.6 * lx, seed=seed,
                                  precision=PREC_MIXED if case["mixed"] else PREC_FP64, **kw)
        s = ChannelSolver(c.params, c.grid)
        s.set_recycling(rc)
    else:
        c = _channel_case(case, seed)
        s = ChannelSolver(c.params, c.grid)
    s.copy_from_field(c.w0)
    s.init_run()
    s.synchronize()
    return {"case": case, "solver": s, "samples": 0}


# -------------------------------------------------------------------- calls
def _interior(w, ng=3):
    return w[:, ng:-ng, ng:-ng, ng:-ng]


def run(state):
    case = state["case"]
    if case["kind"] == "serve":
        sv = state["server"]
        tickets = [sv.submit(r.params, r.grid, r.w0, case["steps"]) for r in state["requests"]]
        return [_interior(sv.wait(t, 300.0)[0]) for t in tickets]
    s = state["solver"]
    s.advance(case["steps"])
    if case["mixed"]:
        # single-precision fluxes: the snapshot is kept in single precision too
        return {"w": _interior(s.copy_to_field()).astype(np.float32)}
    if case["kind"] == "bl":
        # one sample of the running statistics per output interval
        s.compute_stats(state["samples"])
        state["samples"] += 1
        return {"progress": s.compute_residual(), "w": _interior(s.copy_to_field()), "w_stat": s.get_stats()}
    return {"progress": s.compute_residual(), "w": _interior(s.copy_to_field())}


def work(case):
    """Bytes and operations of one pass that no arrangement of the scheme
    avoids.  Per cell and stage: the state read and written (80 B), and the
    right-hand side carried from stages 1 and 2 to the next one (written and
    read, 40 or 20 B a time).  Operations per cell and stage: the split form of
    the convective fluxes at ~80 operations a direction, ~260 of the viscous
    terms, ~60 of the primitives and the update; WENO faces come on top and
    are not counted.  The field read back is one more pass over the state."""
    f = 20.0 if case.get("mixed") else 40.0
    per_stage = 80.0 + 2.0 * 2.0 / 3.0 * f
    if case["kind"] == "serve":
        mid = 0.5 * (case["side_lo"] + case["side_hi"])
        cells, back = case["requests"] * mid ** 3, 80.0  # each request's field goes in and comes out
    else:
        cells, back = float(case["nx"] * case["ny"] * case["nz"]), 40.0
    stages = 3.0 * case["steps"]
    return {"bytes": cells * (stages * per_stage + back), "flops": cells * stages * 560.0}


# -------------------------------------------------- the same in plain torch
C1 = (0.75, -0.15, 1.0 / 60.0)                           # 6th-order first-derivative weights
C2 = (-245.0 / 90.0, 1.5, -0.15, 1.0 / 90.0)             # 6th-order second-derivative weights
CTAB = ((0.5, 0.0, 0.0), (2.0 / 3.0, -1.0 / 12.0, 0.0), C1)  # by half width 1, 2, 3


class _PlainChannel:
    """The channel of one case: 6th-order KEEP split with WENO5 (Roe
    characteristic split, Jiang-Shu) where the Ducros sensor exceeds the
    threshold, viscous terms in Laplacian or second-order conservative form,
    Wray RK3, constant flow rate and optional bulk-temperature control.
    Arrays are [k, j, i] with three ghost points on each side."""

    def __init__(self, c):
        p, g = c.params, c.grid
        self.p, self.dev = p, "cuda" if torch.cuda.is_available() else "cpu"
        t = lambda a: torch.from_numpy(np.array(a, dtype=np.float64)).to(self.dev)  # noqa: E731
        self.n = (p.nx, p.ny, p.nz)
        self.w = [t(c.w0[m]) for m in range(5)]
        shape = {0: (1, 1, -1), 1: (1, -1, 1), 2: (-1, 1, 1)}
        m1 = (g.dcsidx, g.detady, g.dzitdz)
        ms = (g.dcsidxs, g.detadys, g.dzitdzs)
        m2 = (g.dcsidx2, g.detady2, g.dzitdz2)
        self.m1 = [t(m1[d]).reshape(shape[d]) for d in range(3)]
        self.ms = [t(ms[d]).reshape(shape[d]) for d in range(3)]
        self.m2 = [t(m2[d]).reshape(shape[d]) for d in range(3)]
        self.xc = [t(a).reshape(shape[d]) for d, a in enumerate((g.x, g.y, g.z))]
        yn = t(g.yn)
        self.dy = (yn[1:] - yn[:-1]).reshape(1, -1, 1)
        self.cp, self.cv = p.cp_coeff[0], p.cv_coeff[0]
        self.gam = self.cp / (self.cp - p.rgas0)
        self.fl = None
        self.sensor = torch.zeros_like(self.w[0])
        self.time = 0.0

    # ---- ghosts and views
    def inner(self, a, d=None, o=0):
        s = [slice(3, 3 + m) for m in reversed(self.n)]
        if d is not None:
            q = 2 - d
            s[q] = slice(3 + o, 3 + o + self.n[d])
        return a[tuple(s)]

    def wrap(self, a):
        for q in (0, 2):
            m = a.shape[q] - 6
            if q == 0:
                a[:3] = a[m:m + 3]
                a[m + 3:] = a[3:6]
            else:
                a[:, :, :3] = a[:, :, m:m + 3]
                a[:, :, m + 3:] = a[:, :, 3:6]
        return a

    def temperature(self, w):
        ri = 1.0 / w[0]
        u, v, ww = w[1] * ri, w[2] * ri, w[3] * ri
        q = 0.5 * (u * u + v * v + ww * ww)
        ee = w[4] / w[0] - q
        return u, v, ww, q, self.p.t0 + (ee - self.p.cv_coeff[1] * self.p.t0) / self.cv

    def energy(self, t):
        return (self.p.cv_coeff[1] + self.cv * (t / self.p.t0 - 1.0)) * self.p.t0

    def walls(self):
        p, ny = self.p, self.n[1]
        for l in range(1, 4):
            for src, dst in ((l + 2, 3 - l), (ny + 3 - l, ny + 2 + l)):
                row = [a[:, src] for a in self.w]
                u, v, ww, q, t = self.temperature(row)
                pp = row[0] * t * p.rgas0
                t = 2.0 * p.t_wall - t
                rho = pp / t / p.rgas0
                for a, b in zip(self.w, (rho, -rho * u, -rho * v, -rho * ww, rho * (self.energy(t) + q))):
                    a[:, dst] = b

    def primitives(self):
        p = self.p
        for a in self.w:
            self.wrap(a)
        u, v, w, _, t = self.temperature(self.w)
        rho = self.w[0]
        pp = rho * t * p.rgas0
        r = t / p.t0
        if p.visc_model == 1:
            mu = p.mu0 * r ** p.powerlaw_vtexp
        else:
            s = p.sutherland_s / p.t_ref_dim
            mu = p.mu0 * r ** 1.5 * (1.0 + s) / (r + s)
        return {"r": rho, "u": u, "v": v, "w": w, "h": (self.w[4] + pp) / rho, "t": t, "mu": mu, "p": pp}

    def dt(self):
        p = self.p
        a = {k: self.inner(x) for k, x in self.primitives().items()}
        cs = torch.sqrt(self.gam * p.rgas0 * a["t"])
        nu = a["mu"] / a["r"]
        mx = 0.0
        for d, vel in enumerate(("u", "v", "w")):
            mx = max(mx, float(((a[vel].abs() + cs) * self.m1[d]).max()),
                     float((nu * self.ms[d]).max()), float((nu / p.prandtl * self.ms[d]).max()))
        return p.cfl / mx

    # ---- convective fluxes of direction d, added to fl
    def convect(self, a, fl, d):
        p, n = self.p, self.n[d]
        q = 2 - d

        def span(x, lo, m):  # m points from lo (0 = first ghost) along d, interior elsewhere
            s = [slice(3, 3 + z) for z in reversed(self.n)]
            s[q] = slice(lo, lo + m)
            return x[tuple(s)]

        names = ("r", "u", "v", "w", "p")
        e = a["h"] - a["p"] / a["r"] - 0.5 * (a["u"] ** 2 + a["v"] ** 2 + a["w"] ** 2)
        nf = n + 1
        order = torch.full((nf,), 3, dtype=torch.int64)
        if d == 1:  # the staggered walls lower the stencil order of the faces beside them
            for f, o in ((0, 1), (1, 1), (2, 2)):
                order[f] = min(int(order[f]), o)
                order[n - f] = min(int(order[n - f]), o)
        order = order.to(self.dev)
        shape = [1, 1, 1]
        shape[q] = nf
        vn = ("u", "v", "w")[d]
        acc = [0.0] * 6
        for l in range(1, 4):
            cl = torch.tensor([CTAB[o - 1][l - 1] for o in (1, 2, 3)], device=self.dev, dtype=torch.float64)[order - 1].reshape(shape)
            part = [0.0] * 6
            for m in range(l):  # pairs (f - m, f - m + l); face f lies between cells f and f + 1
                A = {k: span(a[k], 2 - m, nf) for k in names}
                B = {k: span(a[k], 2 - m + l, nf) for k in names}
                eA, eB = span(e, 2 - m, nf), span(e, 2 - m + l, nf)
                uv = (A[vn] + B[vn]) * (A["r"] + B["r"])
                part[0] = part[0] + 2.0 * uv
                for x, k in enumerate(("u", "v", "w")):
                    part[1 + x] = part[1 + x] + uv * (A[k] + B[k])
                part[4] = part[4] + uv * (eA + eB) + uv * (A["u"] * B["u"] + A["v"] * B["v"] + A["w"] * B["w"]) \
                    + 4.0 * (A[vn] * B["p"] + B[vn] * A["p"])
                part[5] = part[5] + 2.0 * (A["p"] + B["p"])
            acc = [x + cl * y for x, y in zip(acc, part)]
        f = [0.25 * x for x in acc[:5]]
        if d == 1:
            for x in f:
                x[:, 0] = 0.0
                x[:, n] = 0.0
        f[1 + d] = f[1 + d] + 0.5 * acc[5]
        hot = span(self.sensor, 0, nf) > p.sensor_threshold
        for s in range(1, 6):
            hot = hot | (span(self.sensor, s, nf) > p.sensor_threshold)
        at = hot.nonzero(as_tuple=True)
        if len(at[0]):
            lab = [at[0] + 3, at[1] + 3, at[2] + 3]
            base = lab[q] - 3  # first window point of the face along d
            win = []
            for s in range(6):
                ix = list(lab)
                ix[q] = base + s
                win.append({k: a[k][tuple(ix)] for k in ("r", "u", "v", "w", "h", "t")})
            fw = self.weno(win, d, order[at[q]])
            for m in range(5):
                f[m][at] = fw[m]
        for m in range(5):
            lo, hi = [slice(None)] * 3, [slice(None)] * 3
            lo[q], hi[q] = slice(0, n), slice(1, n + 1)
            fl[m] = fl[m] + (f[m][tuple(hi)] - f[m][tuple(lo)]) * self.m1[d]

    def weno(self, win, d, order):
        p, gam = self.p, self.gam
        A, B = win[2], win[3]
        r = torch.sqrt(B["r"] / A["r"])
        rho, rp1 = r * A["r"], 1.0 / (r + 1.0)
        u, v, w, h = ((r * B[k] + A[k]) * rp1 for k in ("u", "v", "w", "h"))
        qq = 0.5 * (u * u + v * v + w * w)
        tt = p.t0 + (h - qq - p.cp_coeff[1] * p.t0) / self.cp
        cc = gam * tt * p.rgas0
        c = torch.sqrt(cc)
        p_rho, p_e, etot = tt * p.rgas0, rho * (gam - 1.0), h - tt * p.rgas0
        b3 = etot - rho * p_rho / p_e
        b2 = p_e / (rho * cc)
        b1 = p_rho / cc - b2 * (etot - 2.0 * qq)
        vel = (u, v, w)
        un = vel[d]
        tang = [x for x in range(3) if x != d]
        one, zero = torch.ones_like(un), torch.zeros_like(un)
        left, right = [[None] * 5 for _ in range(5)], [[None] * 5 for _ in range(5)]
        for m, sg in ((0, 1.0), (4, -1.0)):
            left[m][0] = 0.5 * (b1 + sg * un / c)
            for x in range(3):
                left[m][1 + x] = -0.5 * (b2 * vel[x] + (sg / c if x == d else 0.0))
            left[m][4] = 0.5 * b2
            right[m] = [one] + [vel[x] - sg * c if x == d else vel[x] for x in range(3)] + [h - sg * un * c]
        left[1] = [1.0 - b1, b2 * u, b2 * v, b2 * w, -b2]
        right[1] = [one, u, v, w, b3]
        for m, x in ((2, tang[0]), (3, tang[1])):
            left[m] = [-vel[x]] + [one if y == x else zero for y in range(3)] + [zero]
            right[m] = [zero] + [one if y == x else zero for y in range(3)] + [vel[x]]
        ev, cons, flux = [-1.0] * 3, [], []
        for q in win:
            vq = (q["u"], q["v"], q["w"])
            cq, pq, ru = torch.sqrt(gam * p.rgas0 * q["t"]), q["r"] * q["t"] * p.rgas0, q["r"] * vq[d]
            for x, z in enumerate(((vq[d] - cq).abs(), vq[d].abs(), (vq[d] + cq).abs())):
                ev[x] = z if isinstance(ev[x], float) else torch.maximum(ev[x], z)
            cons.append([q["r"]] + [q["r"] * x for x in vq] + [q["r"] * q["h"] - pq])
            flux.append([ru] + [x * ru + (pq if y == d else 0.0) for y, x in enumerate(vq)] + [q["h"] * ru])
        out = [0.0] * 5
        s2 = p.rho0 * p.rho0 * p.u0 * p.u0
        for m in range(5):
            lam = ev[0] if m == 0 else (ev[2] if m == 4 else ev[1])
            vp, vm = [], []
            for q in range(6):
                wc = sum(left[m][x] * cons[q][x] for x in range(5))
                gc = sum(left[m][x] * flux[q][x] for x in range(5))
                x = 0.5 * (gc + lam * wc)
                vp.append(x)
                vm.append(gc - x)
            scale = 1.0 / (s2 * p.u0 * p.u0) if m in (2, 3) else 1.0 / s2
            fi = self.side(vp[:5], order, scale) + self.side(vm[:0:-1], order, scale)
            out = [o + right[m][x] * fi for x, o in enumerate(out)]
        return out

    @staticmethod
    def side(v, order, scale):
        """Upwind reconstruction from five points, v[2] the upwind cell."""
        a, b, c, d, e = v
        ind = (13.0 / 12.0 * (c - 2 * b + a) ** 2 + 0.25 * (3 * c - 4 * b + a) ** 2,
               13.0 / 12.0 * (b - 2 * c + d) ** 2 + 0.25 * (b - d) ** 2,
               13.0 / 12.0 * (c - 2 * d + e) ** 2 + 0.25 * (3 * c - 4 * d + e) ** 2)
        wt = [g / (1e-6 + scale * x) ** 2 for g, x in zip((0.1, 0.6, 0.3), ind)]
        cand = ((2 * a - 7 * b + 11 * c) / 6, (-b + 5 * c + 2 * d) / 6, (2 * c + 5 * d - e) / 6)
        r5 = sum(x * y for x, y in zip(wt, cand)) / sum(wt)
        w0, w1 = ((1.0 / 3.0) / (1e-6 + scale * (c - b) ** 2) ** 2, (2.0 / 3.0) / (1e-6 + scale * (d - c) ** 2) ** 2)
        r3 = 0.5 * (w0 * (3 * c - b) + w1 * (c + d)) / (w0 + w1)
        return torch.where(order >= 3, r5, torch.where(order == 2, r3, c))

    # ---- viscous terms; leaves div/3 and |omega| for the caller
    def viscous(self, a, fl):
        p = self.p
        cpr = self.cp / p.prandtl
        I = self.inner
        f = {"u": a["u"], "v": a["v"], "w": a["w"], "t": a["t"], "m": a["mu"]}
        mu, vel = I(f["m"]), [I(f[k]) for k in "uvw"]
        g = {}
        if p.conservative_viscous:
            for d in range(3):
                h = self.span_c(d, 1) - self.span_c(d, -1)
                for k in f:
                    g[k, d] = (I(f[k], d, 1) - I(f[k], d, -1)) / h
        else:
            lap = {k: 0.0 for k in "uvwt"}
            for d in range(3):
                for k in f:
                    s = sum(C1[l - 1] * (I(f[k], d, l) - I(f[k], d, -l)) for l in (1, 2, 3))
                    g[k, d] = s * self.m1[d]
                    if k != "m":
                        s2 = C2[0] * I(f[k]) + sum(C2[l] * (I(f[k], d, l) + I(f[k], d, -l)) for l in (1, 2, 3))
                        lap[k] = lap[k] + s2 * self.ms[d] + g[k, d] * self.m2[d]
        div = g["u", 0] + g["v", 1] + g["w", 2]
        om2 = (g["w", 1] - g["v", 2]) ** 2 + (g["u", 2] - g["w", 0]) ** 2 + (g["v", 0] - g["u", 1]) ** 2
        sig = [[None] * 3 for _ in range(3)]
        for x, kx in enumerate("uvw"):
            for y, ky in enumerate("uvw"):
                sig[x][y] = g[kx, y] + g[ky, x]
            sig[x][x] = sig[x][x] - 2.0 * div / 3.0
        if p.conservative_viscous:
            # mu-gradient part: s[x][y] = d(u_y)/dx_x multiplies d(mu)/dx_y in momentum x
            s = [[g["uvw"[y], x] - (2.0 * div / 3.0 if x == y else 0.0) for y in range(3)] for x in range(3)]
            sm = [sum(g["m", y] * s[x][y] for y in range(3)) for x in range(3)]
            diss = sum(s[x][y] * g["uvw"[x], y] for x in range(3) for y in range(3)) * mu
            e = sum(sm[x] * vel[x] for x in range(3)) + diss
            qq = 0.5 * (f["u"] ** 2 + f["v"] ** 2 + f["w"] ** 2)
            for d in range(3):
                h = 2.0 / (self.span_c(d, 1) - self.span_c(d, -1))
                for sg, lo, hi in ((1.0, 0, 1), (-1.0, -1, 0)):
                    muf = 0.5 * (I(f["m"], d, lo) + I(f["m"], d, hi)) / (self.span_c(d, hi) - self.span_c(d, lo))
                    for x, k in enumerate("uvw"):
                        sm[x] = sm[x] + sg * h * muf * (I(f[k], d, hi) - I(f[k], d, lo))
                    e = e + sg * h * muf * (cpr * (I(f["t"], d, hi) - I(f["t"], d, lo)) + I(qq, d, hi) - I(qq, d, lo))
        else:
            sm = [sum(g["m", y] * sig[x][y] for y in range(3)) + mu * lap["uvw"[x]] for x in range(3)]
            heat = (sum(g["m", y] * g["t", y] for y in range(3)) + mu * lap["t"]) * cpr
            diss = sum(sig[x][y] * g["uvw"[x], y] for x in range(3) for y in range(3)) * mu
            e = sum(sm[x] * vel[x] for x in range(3)) + diss + heat
        if fl is not None:
            for x in range(3):
                fl[1 + x] = fl[1 + x] - sm[x]
            fl[4] = fl[4] - e
        return div / 3.0, torch.sqrt(om2)

    def span_c(self, d, o):
        x, n = self.xc[d], self.n[d]
        s = [slice(None)] * 3
        s[2 - d] = slice(3 + o, 3 + o + n)
        return x[tuple(s)]

    def dilatation(self, a, fl, d3):
        """The grad(div/3) terms."""
        p = self.p
        full = torch.zeros_like(self.w[0])
        self.inner(full).copy_(d3)
        for l in range(3):
            full[:, l] = full[:, 3]
            full[:, 3 + self.n[1] + l] = full[:, 2 + self.n[1]]
        self.wrap(full)
        mu = self.inner(a["mu"])
        e = 0.0
        for d, k in enumerate("uvw"):
            if p.conservative_viscous:
                s = mu * (self.inner(full, d, 1) - self.inner(full, d, -1)) / (self.span_c(d, 1) - self.span_c(d, -1))
            else:
                s = mu * sum(C1[l - 1] * (self.inner(full, d, l) - self.inner(full, d, -l)) for l in (1, 2, 3)) * self.m1[d]
            fl[1 + d] = fl[1 + d] - s
            e = e + s * self.inner(a[k])
        fl[4] = fl[4] - e

    def set_sensor(self, d3, om):
        div, ul = 3.0 * d3, self.p.u0 / self.p.l0
        s = torch.clamp(-div / torch.sqrt(om * om + div * div + ul * ul), min=0.0) ** 2
        self.sensor.zero_()
        self.inner(self.sensor).copy_(s)
        self.wrap(self.sensor)

    def solve(self, steps):
        p, dy = self.p, self.dy
        self.walls()
        self.set_sensor(*self.viscous(self.primitives(), None))
        prev = None
        for _ in range(steps):
            dt = self.dt()
            dpdx = 0.0
            for s, (rk, gk) in enumerate(((0.0, 8.0 / 15.0), (-17.0 / 60.0, 5.0 / 12.0), (-5.0 / 12.0, 3.0 / 4.0))):
                a = self.primitives()
                fl = [0.0] * 5
                for d in range(3):
                    self.convect(a, fl, d)
                d3, om = self.viscous(a, fl)
                if s == 2:
                    self.set_sensor(d3, om)
                self.dilatation(a, fl, d3)
                inc = [-gk * dt * x for x in fl]
                if s:
                    inc = [x - rk * dt * y for x, y in zip(inc, prev)]
                prev = fl
                rho, ru, t = self.inner(self.w[0]), self.inner(self.w[1]), self.inner(a["t"])
                b1, b2 = (float((x * dy).sum()) / p.volchan for x in inc[:2])
                rhob = float((rho * dy).sum()) / p.volchan
                ub = float((ru * dy).sum()) / p.volchan / rhob
                tb = float((ru * dy * t).sum()) / p.volchan / rhob / ub
                dpdx += b2
                stage_rho = rho.clone()
                inc[0] = inc[0] - b1
                inc[1] = inc[1] - b2
                inc[4] = inc[4] - self.inner(a["u"]) * b2
                for x, y in zip(self.w, inc):
                    self.inner(x).add_(y)
                if p.theta_wall >= -1.0:
                    wi = [self.inner(x) for x in self.w]
                    tn = self.temperature(wi)[4]
                    shift = p.t_bulk_target - float((wi[1] * tn * dy).sum()) / p.volchan / rhob / ub
                    wi[4].copy_(wi[0] * self.energy(tn + shift) + 0.5 * (wi[1] ** 2 + wi[2] ** 2 + wi[3] ** 2) / wi[0])
                    last_t = tn
                else:
                    last_t = t
                self.walls()
                last = (stage_rho, last_t, inc[1])
            self.time += dt
        rho, t, inc1 = last
        pp = rho * t * p.rgas0
        # the residual takes the forced increment of the last stage
        res = math.sqrt(float(((inc1 / dt) ** 2).sum()) / rho.numel())
        return {"dt": dt, "time": self.time, "dpdx": dpdx, "rhobulk": rhob, "ubulk": ub, "tbulk": tb,
                "residual_rhou": res, "icyc": steps,
                "rhomin": float(rho.min()), "rhomax": float(rho.max()), "tmin": float(t.min()),
                "tmax": float(t.max()), "pmin": float(pp.min()), "pmax": float(pp.max())}


def _plain(c, steps):
    s = _PlainChannel(c)
    progress = s.solve(steps)
    return progress, torch.stack([s.inner(x) for x in s.w]).cpu().numpy()


def exact(case, seed):
    if case["kind"] == "serve":
        return [_plain(r, case["steps"])[1] for r in _requests(case, seed)]
    # the recycling inflow feeds on the C library's random stream; the largest channels take too long this way
    if case["kind"] == "bl" or case["nx"] * case["ny"] * case["nz"] * case["steps"] > 400e6:
        return None
    progress, w = _plain(_channel_case(case, seed), case["steps"])
    return {"w": w} if case["mixed"] else {"progress": progress, "w": w}
