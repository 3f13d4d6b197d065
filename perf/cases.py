"""Performance cases of the pseudo-time path.

A case is a resident solve: the grid, metrics and kernel choice are what a
program keeps, and one pass is what it does with a new state -- upload it,
run a number of multigrid cycles through ``Solve``, and read the solution
and the residual history back.  Pinned host buffers, as for checkpoints.

The listed cases cover what the repository's benchmark, tests and serving
program run: steady Euler from one 16^3-cell block to 48 uneven blocks, the
NACA 0012 O-grid, harmonic balance, Wilcox k-omega and SST, dual time
stepping, batched and concurrent serving, every smoothing family in use and
the FP64, FP32-residual and contracted precision modes.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from cosa_amd import _lib
from cosa_amd import case as cases
from cosa_amd import serve
from cosa_amd.config import kw_turbulence
from cosa_amd.solver import Solve

# flow and scheme settings shared by the cases of one kind
EULER = dict(ilimf=4, epslimf=1e-6, nl_crs=2, ncycle=100000)
KOMEGA = dict(tu=1e-4, mutfar=1e-2, stemp=110.4 / 288.15, ifixq=1, lim_prodtke=1, prdlim=20.0)


def listed():
    return [
        # one small block on one level, smoothed step by step by a driver that
        # waits for every cycle: launches and latency
        dict(name="tiny_block", kind="channel", dims="17x17x17", nlevel=1, irsop=1, cycles=20, drive="steps"),
        # odd extents that no tile divides, variable-coefficient smoothing
        # (cirs_v1), two blocks of different shape, one level
        dict(name="ragged_cirs_v1", kind="channel", dims="74x39x28,46x60x23", nlevel=1, irsop=2, cycles=6,
             drive="steps"),
        # the same kind of blocks with the FP32 residual and constant coefficients
        dict(name="ragged_f32", kind="channel", dims="99x36x29,50x52x41", nlevel=1, irsop=1, cycles=6,
             drive="graph", precision=1),
        # the aerofoil O-grid with its seam cut, three levels
        dict(name="naca_o193", kind="naca", ni=193, nj=49, nk=9, nlevel=3, irsop=1, cycles=10, drive="graph",
             autotune=1),
        # harmonic balance, N = 4, pitching aerofoil (moving metrics), two levels
        dict(name="naca_hb4", kind="hb", ni=385, nj=97, nk=5, nharms=4, nlevel=2, irsop=1, cycles=6, drive="graph",
             autotune=1),
        # batched serving: 16 requests of one grid as the blocks of one solve,
        # each with its own freestream, cirs_v2 smoothing, norms and forces per block
        dict(name="serve_batch16", kind="batch", grid="small", slots=16, nlevel=2, irsop=3, cycles=10, drive="graph"),
        # concurrent serving: resident solves of different size and physics,
        # each on its own stream with one cycle in flight
        dict(name="serve_mix", kind="mix", cycles=8, drive="graph"),
        # dual time stepping with the implicit physical-time term: one physical step
        dict(name="dual_step", kind="channel", dims="97x49x49", nlevel=2, irsop=1, cycles=8, drive="dual"),
        # RANS on an aerofoil O-grid, Menter SST, two levels
        dict(name="naca_sst", kind="sst", ni=257, nj=65, nk=9, nlevel=2, irsop=2, cycles=6, drive="graph"),
        # RANS wing, Wilcox k-omega, four blocks with cuts, three levels
        dict(name="wing_komega", kind="wing", ni=257, nj=65, nk=33, nblocks=4, nlevel=3, irsop=1, cycles=4,
             drive="graph", autotune=1),
        # uneven multiblock channels in the contracted FP64 mode
        dict(name="uneven16_fp64c", kind="uneven", nblocks=16, nlevel=3, irsop=1, cycles=8, drive="graph",
             precision=3, autotune=1),
        # uneven multiblock channels, the benchmark's headline kind
        dict(name="uneven48", kind="uneven", nblocks=48, nlevel=3, irsop=1, cycles=8, drive="graph", autotune=1),
    ]


def draw(rng):
    """Another case of the same kinds, sizes over the whole range."""
    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["channel", "channel", "naca", "hb", "sst", "wing", "uneven"])
    c = dict(kind=kind, cycles=rng.randint(3, 6), drive=rng.choice(["graph", "graph", "steps"]),
             irsop=rng.choice([1, 1, 1, 2, 3]), autotune=rng.randint(0, 1))
    if kind == "channel":
        # one level with any extents, or two / three levels on multiples of 4 / 8 cells
        c["nlevel"] = rng.choice([1, 1, 2, 3])
        m = 1 if c["nlevel"] == 1 else 2 ** c["nlevel"]
        dims = []
        for _ in range(rng.randint(1, 4)):
            dims.append("x".join(str(max(2 if m > 1 else 9, logint(9, 140) // m) * m + 1) for _ in range(3)))
        c["dims"] = ",".join(dims)
        c["precision"] = rng.choice([0, 0, 1, 3])
    elif kind == "uneven":
        c.update(nblocks=rng.randint(4, 16), nlevel=3, irsop=1, precision=rng.choice([0, 0, 1, 3]))
    elif kind == "wing":
        c.update(ni=8 * logint(8, 24) + 1, nj=8 * logint(3, 8) + 1, nk=8 * logint(2, 4) + 1, nblocks=rng.randint(1, 4),
                 nlevel=rng.choice([2, 3]), irsop=1, precision=rng.choice([0, 0, 1]))
    else:
        c.update(ni=8 * logint(6, 48) + 1, nj=4 * logint(5, 24) + 1, nk=4 * rng.randint(1, 3) + 1, nlevel=2)
        if kind == "naca":
            c["precision"] = rng.choice([0, 0, 1, 3])
        elif kind == "hb":
            c.update(nharms=rng.randint(1, 4), irsop=1)
        else:
            c.update(irsop=rng.choice([1, 2]), nj=4 * logint(8, 16) + 1)
    return c


# ---------------------------------------------------------------------------
# building the solves

def _dims(c):
    if c["kind"] == "uneven":
        return [tuple(d) for d in cases.uneven_dims(c["nblocks"], seed=0)]
    return [tuple(int(v) for v in t.split("x")) for t in c["dims"].split(",")]


def _irs(c):
    irs = {1: dict(irsop=1, cfl=2.0, cfl_irs=4.0), 2: dict(irsop=2, cfl=2.0, cfl_irs=4.0),
           3: dict(irsop=3, psirs=0.125, cfl=2.0, cfl_irs=5.0)}
    return irs[c["irsop"]]


def _mix():
    """The resident solves of serve_mix: requests of the serving program."""
    return [serve.Request(0, "small", 0.4, 1.0), serve.Request(1, "small", 0.6, -2.0),
            serve.Request(2, "medium", 0.5, 2.0), serve.Request(3, "small", 0.3, 4.0, rans=True),
            serve.Request(4, "medium", 0.3, 1.0, rans=True), serve.Request(5, "small", 0.5, 0.0, nharms=2)]


@functools.lru_cache(maxsize=8)
def _grid(key):
    """The repository's Case objects of a case: grids and metrics, which do
    not depend on the state and which a program keeps."""
    c = dict(key)
    k, nl = c["kind"], c.get("nlevel", 1)
    if k in ("channel", "uneven"):
        kw = dict(EULER, machfs=0.7, **_irs(c))
        if c["drive"] == "dual":
            kw.update(machfs=0.5, rkimp=1, cfl_irs=3.5, ncycle=c["cycles"])
        return [cases.channel_case(_dims(c), nlevel=nl, **kw)]
    if k == "naca":
        return [cases.naca_case(c["ni"], c["nj"], c["nk"], nlevel=nl, **EULER, **_irs(c))]
    if k == "hb":
        return [cases.naca_case(c["ni"], c["nj"], c["nk"], nlevel=nl, irsop=1, cfl=2.0, cfl_irs=3.5, machfs=0.5,
                                alpha_deg=0.0, nharms=c["nharms"], harbal=1, omega=0.1,
                                pitch=dict(dtheta0=math.radians(5.0), xh=0.25, yh=0.0), **EULER)]
    if k == "sst":
        kw = dict(irsop=c["irsop"], cfl=1.0, cfl_irs=2.0, nl_crs=2, ncycle=100000)
        return [cases.naca_case(c["ni"], c["nj"], c["nk"], nlevel=nl, wall=1500, ds_wall=2e-5, **kw,
                                **kw_turbulence(0.4, 1.0e6, model="sst", tu=1e-4, mutfar=1e-2,
                                                stemp=110.4 / 288.15, ifixq=1))]
    if k == "wing":
        return [cases.wing_case(c["ni"], c["nj"], c["nk"], nblocks=c["nblocks"], nlevel=nl, irsop=1, cfl=2.0,
                                cfl_irs=4.0, nl_crs=2, ncycle=100000, ds_wall=5e-6,
                                **kw_turbulence(0.3, 3.0e6, **KOMEGA))]
    if k == "batch":
        return [serve.batch_case(serve.Request(0, c["grid"], 0.5, 1.0, max_cycles=100000), c["slots"])]
    if k == "mix":
        return [r.make_case() for r in _mix()]
    raise ValueError(k)


def _cases_of(c):
    return _grid(tuple(sorted((k, v) for k, v in c.items() if k not in ("name", "autotune", "precision"))))


class _Resident:
    """One solve a program keeps, its initial state and its read-back buffer
    in pinned host memory."""

    def __init__(self, c, case, seed, amp):
        self.case = case
        q0 = case.perturbed(amp=amp, seed=seed)
        self.solve = s = Solve(case, device=0, q=q0)
        self.q0 = torch.from_numpy(q0).pin_memory().numpy()
        self.q = torch.empty(q0.size, dtype=torch.float64, pin_memory=True).numpy()
        if c.get("precision"):
            s.set_precision(c["precision"])

    def load(self):
        self.solve.upload("q", self.q0)

    def read(self):
        s = self.solve
        s._check(s.lib.cosahip_download(s.h, 1, _lib.FIELD_IDS["q"], _lib.dptr(self.q), self.q.size), "download")
        return self.q


def prepare(case, seed):
    c = case
    # a smaller perturbation where a boundary layer is resolved
    amp = 0.01 if c["kind"] in ("channel", "uneven", "naca", "hb") else 0.002
    st = dict(c=c, r=[_Resident(c, g, 1000 * seed + m, amp) for m, g in enumerate(_cases_of(c))])
    s = st["r"][0].solve
    if c["kind"] == "batch":
        rng = np.random.default_rng(seed)
        for b in range(c["slots"]):
            s.set_block_freestream(b + 1, float(rng.uniform(0.3, 0.6)), float(rng.uniform(-2.0, 4.0)))
        s.set_block_rms(True)
    if c["drive"] == "dual":
        s.set_dual_time(0.5)
        return st
    for r in st["r"]:
        r.solve.cycle_async(1)   # the first cycle of a solve, which differs from the later ones (k-omega)
    if c.get("autotune"):
        s.autotune(1)
    return st


def run(state):
    c, rs = state["c"], state["r"]
    n = c["cycles"]
    for r in rs:
        r.load()
        r.solve.history.clear()
    s = rs[0].solve
    if c["drive"] == "dual":
        s.dual_step(1, n)
    elif c["drive"] == "steps":
        for m in range(n):
            s.cycle(m + 2)
    elif len(rs) == 1:
        for m in range(n):
            s.cycle_async(m + 2)
    else:
        # the serving loop: every resident solve keeps one cycle in flight
        left = {i: n for i in range(len(rs))}
        for r in rs:
            r.solve.cycle_enqueue(2)
        while left:
            for i in list(left):
                if not rs[i].solve.cycle_ready():
                    continue
                rs[i].solve.cycle_wait()
                left[i] -= 1
                if left[i]:
                    rs[i].solve.cycle_enqueue(2 + n - left[i])
                else:
                    del left[i]
    out = dict(q=[r.read() for r in rs], history=[np.array(r.solve.history) for r in rs])
    if c["kind"] == "batch":
        out["block_rms"] = s.block_rms()
        out["forces"] = s.force_blocks()
    return out


# ---------------------------------------------------------------------------
# what a pass needs, and how far it may be off

def _cells(c):
    """Interior cell-snapshots of level 1."""
    if c["kind"] in ("channel", "uneven"):
        return sum((a - 1) * (b - 1) * (d - 1) for a, b, d in _dims(c))
    if c["kind"] == "batch":
        ni, nj = serve.GRIDS[c["grid"]]
        return (ni - 1) * (nj - 1) * (serve.NK - 1) * c["slots"]
    if c["kind"] == "mix":
        return sum((serve.GRIDS[r.grid][0] - 1) * (serve.GRIDS[r.grid][1] - 1) * (serve.NK - 1) *
                   (2 * r.nharms + 1) for r in _mix())
    return ((c["ni"] - 1) * (c["nj"] - 1) * (c["nk"] - 1) * c.get("nblocks", 1)) * (2 * c.get("nharms", 0) + 1)


def work(case):
    """Bytes: the state in and out, face metrics (with metric derivatives and
    wall distance where viscous) and volume, once per pass.  Operations: the
    fluxes, smoothing and update of every RK stage of every cycle and level."""
    turb = case["kind"] in ("wing", "sst")
    cells = _cells(case)
    # stages of a V-cycle in level-1 cells (4 per smoothing, level 2 smoothed twice of three levels)
    stages = 4.0 * (1 + {1: 0.0, 2: 1 / 8, 3: 2 / 8 + 1 / 64}[case.get("nlevel", 2)])
    return {"bytes": cells * 8 * (2 * 7 + 12 + 27 + 2 if turb else 2 * 5 + 12 + 1),
            "flops": cells * stages * case["cycles"] * (2000 if turb else 1000)}


def tolerance(case):
    """About four times what one unit in the last place of the input, or the
    contracted instead of the exact FP64 residual, changes in a pass (at most
    4e-14, single values 2e-13); with the FP32 residual four times its
    distance from the FP64 pass (1.6e-7 and 5e-7, RANS 4.6e-7 and 9.3e-6)."""
    if case.get("precision", 0) == 1:
        return {"rel": 2e-6, "max": 4e-5} if case["kind"] == "wing" else {"rel": 6e-7, "max": 2e-6}
    return {"rel": 2e-13, "max": 2e-12}


# ---------------------------------------------------------------------------
# the same pass in 64-bit numpy: steady Euler channels on one level

def exact(case, seed):
    c = case
    if c["kind"] != "channel" or c["nlevel"] != 1 or c["drive"] == "dual":
        return None   # multigrid, moving-grid and turbulent passes take minutes in numpy
    g = _cases_of(c)[0]
    if g.ncell() * c["cycles"] > 3_000_000:
        return None
    q, hist = _Channels(g, g.perturbed(amp=0.01, seed=1000 * seed)).cycles(c["cycles"])
    return dict(q=[q], history=[hist])


class _Channels:
    """Steady Euler on one level, every block on its own: arrays
    [variable, k, j, i] with two halo layers, so cell i sits at index i + 1."""

    def __init__(self, g, q):
        self.cf, self.q, self.blk = g.config, q.copy(), []
        L = g.levels[0]
        o3, o2 = L.offsets(3), L.offsets(2)
        for b in range(L.nblocks):
            nk, nj, ni = int(L.kmax[b]), int(L.jmax[b]), int(L.imax[b])
            n3, n2 = (nk + 3) * (nj + 3) * (ni + 3), (nk + 2) * (nj + 2) * (ni + 2)
            qb = self.q[o3[b] * 5:o3[b] * 5 + 5 * n3].reshape(5, nk + 3, nj + 3, ni + 3)
            met = [np.moveaxis(g.geom[0][s][o2[b] * 4:(o2[b] + n2) * 4].reshape(nk + 2, nj + 2, ni + 2, 4), -1, 0)
                   for s in ("si", "sj", "sk")]
            self.blk.append((qb, met))

    @staticmethod
    def _at(qb, ax, m):
        """Cells m of axis ax (1 k, 2 j, 3 i), interior of the other axes."""
        sl = [slice(None)] + [slice(2, -2)] * 3
        sl[ax] = m + 1
        return tuple(sl)

    def _far(self, qb, ax, halo, cell, s, sgn):
        p, gam = self.cf, self.cf["gamma"]
        u = qb[self._at(qb, ax, cell)]
        sx, sy, sz = (s[m] * sgn for m in range(3))
        qf = [p["rhoinf"], p["machfs"] * math.cos(p["alpha"]) * math.cos(p["beta"]),
              p["machfs"] * math.sin(p["alpha"]) * math.cos(p["beta"]), p["machfs"] * math.sin(p["beta"]), p["pinf"]]
        qext, qinf = u[1] * sx + u[2] * sy + u[3] * sz, qf[1] * sx + qf[2] * sy + qf[3] * sz
        rext = qext + 2 * np.sqrt(gam * u[4] / u[0]) / (gam - 1)
        rinf = qinf - 2 * p["ainf"] / (gam - 1)
        qn, a = (rext + rinf) / 2, (gam - 1) * (rext - rinf) / 4
        sup, inflow = np.abs(qn / a) >= 1, qn <= 0
        ent = np.where(inflow, p["pinf"] / p["rhoinf"] ** gam, u[4] / u[0] ** gam)
        ref = np.where(inflow, np.array(qf).reshape(5, 1, 1), u)
        rho = (a * a / (gam * ent)) ** (1 / (gam - 1))
        dq = qn - np.where(inflow, qinf, qext)
        sub = np.stack([rho, ref[1] + dq * sx, ref[2] + dq * sy, ref[3] + dq * sz, rho * a * a / gam])
        v = np.where(sup, ref, sub)
        for h in halo:
            qb[self._at(qb, ax, h)] = v

    def _bc(self, qb, met):
        n = qb.shape[3] - 3   # i: farfield
        for halo, c1, f, sgn in (((0, -1), 1, 1, -1.0), ((n, n + 1), n - 1, n, 1.0)):
            self._far(qb, 3, halo, c1, met[0][:, 1:-2, 1:-2, f], sgn)
        n = qb.shape[2] - 3   # j: slip walls
        for halo, c1, c2, f in (((0, -1), 1, 2, 1), ((n, n + 1), n - 1, n - 2, n)):
            s = met[1][:, 1:-2, f, 1:-2]
            w = (3 * qb[self._at(qb, 2, c1)] - qb[self._at(qb, 2, c2)]) / 2
            un = w[1] * s[0] + w[2] * s[1] + w[3] * s[2]
            for m in range(3):
                w[m + 1] -= un * s[m]
            for h in halo:
                qb[self._at(qb, 2, h)] = w
        n = qb.shape[1] - 3   # k: symmetry
        for h, m in ((0, 1), (-1, 2), (n, n - 1), (n + 1, n - 2)):
            v = qb[self._at(qb, 1, m)].copy()
            v[3] *= -1
            qb[self._at(qb, 1, h)] = v

    def _flux(self, qb, s, ax):
        """Face flux difference along axis ax (j faces are slip walls)."""
        gam, eps = self.cf["gamma"], self.cf["epslimf"] ** 2
        sl = [slice(None)] + [slice(2, -2)] * 3
        sl[ax] = slice(None)
        q = np.moveaxis(qb[tuple(sl)], ax, -1)           # cells -1 .. L + 1 along the last axis
        sm = [slice(None)] + [slice(1, -2)] * 3
        sm[ax] = slice(1, -1)
        kx, ky, kz, ds = np.moveaxis(s[tuple(sm)], ax, -1)
        d = np.diff(q, axis=-1)                            # d[m] = q(m) - q(m - 1), m = 0 .. L + 1
        if ax == 2:
            d[..., 1] *= 2
            d[..., -2] *= 2
        d1, d2 = d[..., 1:], d[..., :-1]
        h = (d1 * (d2 * d2 + eps) + d2 * (d1 * d1 + eps)) / (d1 * d1 + d2 * d2 + 2 * eps) / 2   # cells 0 .. L
        qr, ql = q[..., 2:-1] - h[..., 1:], q[..., 1:-2] + h[..., :-1]
        if ax == 2:
            qr[..., 0] = ql[..., 0] = q[..., 1]
            qr[..., -1] = ql[..., -1] = q[..., -2]

        def side(w):
            un = w[1] * kx + w[2] * ky + w[3] * kz
            h0 = gam / (gam - 1) * w[4] / w[0] + (w[1] ** 2 + w[2] ** 2 + w[3] ** 2) / 2
            m = w[0] * un
            return un, h0, np.stack([m, m * w[1] + w[4] * kx, m * w[2] + w[4] * ky, m * w[3] + w[4] * kz, m * h0])

        unr, h0r, fr = side(qr)
        unl, h0l, fl = side(ql)
        sl_, sr_ = np.sqrt(ql[0]), np.sqrt(qr[0])
        rho, den = sl_ * sr_, sl_ + sr_
        u, v, w, h0 = ((sl_ * x + sr_ * y) / den for x, y in ((ql[1], qr[1]), (ql[2], qr[2]), (ql[3], qr[3]), (h0l, h0r)))
        un, q2 = u * kx + v * ky + w * kz, u * u + v * v + w * w
        a2 = (gam - 1) * (h0 - q2 / 2)
        a = np.sqrt(a2)
        dr, du, dv, dw, dp = qr - ql
        dun = unr - unl
        a1, ash = np.abs(un) * (dr - dp / a2), np.abs(un) * rho
        a3 = np.abs(un + a) * (dp / a2 + rho * dun / a) / 2
        a4 = np.abs(un - a) * (dp / a2 - rho * dun / a) / 2
        df = np.stack([a1 + a3 + a4,
                       a1 * u + ash * (du - dun * kx) + a3 * (u + a * kx) + a4 * (u - a * kx),
                       a1 * v + ash * (dv - dun * ky) + a3 * (v + a * ky) + a4 * (v - a * ky),
                       a1 * w + ash * (dw - dun * kz) + a3 * (w + a * kz) + a4 * (w - a * kz),
                       a1 * q2 / 2 + ash * (u * du + v * dv + w * dw - un * dun) + a3 * (h0 + a * un) + a4 * (h0 - a * un)])
        return np.moveaxis(np.diff((fr + fl - df) / 2 * ds, axis=-1), -1, ax)

    def _step(self, qb, met):
        """Local time step and the smoothing coefficients of the three directions."""
        p = self.cf
        r, u, v, w, pr = qb[:, 2:-2, 2:-2, 2:-2]
        a, lam = np.sqrt(p["gamma"] * pr / r), []
        for s, ax in zip(met, (3, 2, 1)):
            f = [s[:, 1:-2, 1:-2, 1:-2], None]
            sl = [slice(None)] + [slice(1, -2)] * 3
            sl[ax] = slice(2, -1)
            f[1] = s[tuple(sl)]
            x = [0.5 * (f[0][m] * f[0][3] + f[1][m] * f[1][3]) for m in range(3)]
            lam.append(np.abs(u * x[0] + v * x[1] + w * x[2]) + a * (f[0][3] + f[1][3]) / 2)
        tot = lam[0] + lam[1] + lam[2]
        beta = [np.full_like(tot, 0.25 * (p["rat"] ** 2 - 1))] * 3
        for d in range(3) if p["irsop"] != 1 else ():
            l1, l2 = lam[(d + 1) % 3], lam[(d + 2) % 3]
            if p["irsop"] == 2:
                t = p["rat"] * lam[d] * (1 + (l1 / lam[d]) ** 0.4 + (l2 / lam[d]) ** 0.4) / tot
            else:
                t = p["rat"] / (1 + p["psirs"] * (l1 / lam[d] + l2 / lam[d]))
            beta[d] = np.maximum(0.0, (t * t - 1) / 4)
        return p["cfl"] / tot, beta

    @staticmethod
    def _smooth(x, eps, ax):
        """Tridiagonal solve along axis ax, in place."""
        x, e = np.moveaxis(x, ax, 0), np.moveaxis(eps, ax - 1, 0)
        n = x.shape[0]
        r = np.zeros_like(e)
        for m in range(n):
            den = 1 + 2 * e[m] + (r[m - 1] * e[m] if m else 0.0)
            r[m] = (-e[m] if m < n - 1 else 0.0) / den
            x[m] = (x[m] + (x[m - 1] * e[m] if m else 0.0)) / den
        for m in range(n - 2, -1, -1):
            x[m] -= x[m + 1] * r[m]

    def cycles(self, n):
        gam, hist = self.cf["gamma"], []
        for _ in range(n):
            sums, ncell = np.zeros(5), 0
            for qb, met in self.blk:
                inner = (slice(None), slice(2, -2), slice(2, -2), slice(2, -2))
                old = qb[inner].copy()
                for st in range(self.cf["nstage"]):
                    w = qb[inner]
                    w[1:4] /= w[0]
                    w[4] = (gam - 1) * (w[4] - w[0] * (w[1] ** 2 + w[2] ** 2 + w[3] ** 2) / 2)
                    self._bc(qb, met)
                    if st == 0:
                        dt, beta = self._step(qb, met)
                    res = sum(self._flux(qb, s, ax) for s, ax in zip(met, (3, 2, 1)))
                    if st == 0:
                        sums += (res ** 2).sum(axis=(1, 2, 3))
                        ncell += dt.size
                    # back to conservative variables, face halos included
                    for ax in (3, 2, 1):
                        for h in (-1, 0, qb.shape[ax] - 3, qb.shape[ax] - 2):
                            sl = self._at(qb, ax, h)
                            qb[sl] = self._cons(qb[sl], gam)
                    res = res * dt
                    for d, ax in enumerate((3, 2, 1)):
                        self._smooth(res, beta[d], ax)
                    qb[inner] = old - self.cf["alphas"][st] * res
            rms = np.zeros(8)
            rms[:5] = np.sqrt(sums / ncell)
            rms[5] = math.sqrt(sums.sum() / ncell / 5)
            hist.append(rms)
        return self.q, np.array(hist)

    @staticmethod
    def _cons(w, gam):
        w = w.copy()
        w[4] = w[4] / (gam - 1) + w[0] * (w[1] ** 2 + w[2] ** 2 + w[3] ** 2) / 2
        w[1:4] *= w[0]
        return w
