"""Timed cases of the hydro path: what a user's program has this framework do, through its public
entry points (`Sim`, `AmrSim`, `Ensemble`).

A pass advances a resident run by some steps and reads its state back, as a driver does between
two frames or outputs (README's quick start). `prepare` is what such a program has done before:
the initial conditions uploaded and, where the case says so, the tile tuned.

The kinds, and the grids they come from:

- ``uniform``: one grid. The turbulence box, the Sedov blast and the 2D Kelvin-Helmholtz layer at
  the sizes `bench.py` reports, the four-quadrant Riemann problem, a grid with walls and ragged
  sizes, and the FP64 twin.
- ``ensemble``: independent 2D Riemann problems of seeded sizes, stepped together.
- ``blast``: 3D blocks refined around a hot sphere (the fused march, or the passes with per-block
  timesteps).
- ``shear``: the shear layer on a 2D quadtree (static, or re-meshed every few steps).

`exact` restates the scheme in 64 bits with plain torch. It leaves out per-block timesteps and
re-meshed runs (whose mesh follows thresholds on the state) and the runs that are too long for it.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from shaderous_amd import amr_tree, problems
from shaderous_amd.amr import AmrSim
from shaderous_amd.ensemble import Ensemble
from shaderous_amd.sim import Sim, SimConfig, config_for

BS = 16


# ---------------- the cases ----------------
def listed():
    return [
        # the smallest call a caller makes: a small grid, a few steps between two looks at it
        # (an interactive driver); outflow on all four sides, as created (no tuning)
        _uniform("quadrants-64", "quadrants", (64, 64, 1), steps=16, scheme="mc", tune=False),
        # the 2D shear layer at the size a CPU can still check: one launch per ~10 us step
        _uniform("kh-256", "kh", (256, 256, 1), steps=200, scheme="mc", tune=True),
        # the large published 2D grid with the default scheme of the reference
        _uniform("kh-2048-koren", "kh", (2048, 2048, 1), steps=200, scheme="koren", tune=True),
        # the published 3D blast with the default scheme
        _uniform("sedov-128-koren", "sedov", (128, 128, 128), steps=150, scheme="koren", tune=True),
        # the throughput benchmark's grid
        _uniform("turbulence-256", "turbulence", (256, 256, 256), steps=300, scheme="mc", tune=True),
        # a box with walls and odd sizes along every axis, as created (no tuning)
        _uniform("walls-150x101x67", "walls", (150, 101, 67), steps=100, scheme="mc", tune=False),
        # the all-FP64 twin, for precision studies
        _uniform("turbulence-96-f64", "turbulence", (96, 96, 96), steps=40, scheme="mc", tune=True, precision=64),
        # uneven 2D grids, each with its own dt, one launch per step
        {"name": "ensemble-24", "kind": "ensemble", "count": 24, "largest": 512, "steps": 150, "scheme": "mc",
         "tune": True},
        # the 3D blast on blocks, two refinements, the fused march
        {"name": "blast-fused", "kind": "blast", "root": 8, "levels": 2, "steps": 80, "scheme": "mc",
         "path": "fused", "bins": 0},
        # the same physics with per-block timesteps (eight cycles of eight substeps)
        {"name": "blast-bins", "kind": "blast", "root": 4, "levels": 2, "steps": 64, "scheme": "mc",
         "path": "passes", "bins": 3},
        # the published adaptive 2D run's mesh (256^2 root cells, finest 4096^2), default scheme
        {"name": "shear-4096-koren", "kind": "shear", "root": 16, "levels": 4, "steps": 100, "scheme": "koren",
         "regrid": 0},
        # a run that re-meshes as it goes, every eight steps
        {"name": "shear-regrid", "kind": "shear", "root": 8, "levels": 2, "steps": 24, "scheme": "mc", "regrid": 8},
    ]


def _uniform(name, problem, n, steps, scheme, tune, precision=32):
    c = {"name": name, "kind": "uniform", "problem": problem, "nx": n[0], "ny": n[1], "nz": n[2], "steps": steps,
         "scheme": scheme, "tune": tune, "precision": precision}
    if name is None:
        del c["name"]
    return c


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above: 2D grids of 48^2 to 1500^2, 3D ones of 24^3 to 180^3
    (120^3 in FP64), ensembles of 4 to 28 grids, block trees of 64 to a few thousand blocks."""
    kind = rng.choice(["2d", "2d", "3d", "3d", "walls", "f64", "ensemble", "blast", "blast", "shear", "shear"])
    scheme = rng.choice(["mc", "koren"])
    tune = rng.random() < 0.6
    if kind == "2d":
        n = _log_int(rng, 48, 1500)
        if rng.random() < 0.5:
            return _uniform(None, "kh", (n, n, 1), _log_int(rng, 16, 120), scheme, tune)
        return _uniform(None, "quadrants", (n, _log_int(rng, max(48, n // 2), n), 1), _log_int(rng, 16, 120), scheme,
                        tune)
    if kind == "3d":
        n = _log_int(rng, 24, 180)
        return _uniform(None, rng.choice(["sedov", "turbulence"]), (n, n, n), _log_int(rng, 20, 100), scheme, tune)
    if kind == "walls":
        return _uniform(None, "walls", tuple(_log_int(rng, 20, 160) for _ in range(3)), _log_int(rng, 20, 100), scheme,
                        tune)
    if kind == "f64":
        n = _log_int(rng, 24, 120)
        flat = rng.random() < 0.4
        return _uniform(None, "kh" if flat else "turbulence", (n, n, 1 if flat else n), _log_int(rng, 10, 40), scheme,
                        True, 64)
    if kind == "ensemble":
        return {"kind": "ensemble", "count": rng.randint(4, 28), "largest": _log_int(rng, 96, 512),
                "steps": _log_int(rng, 40, 120), "scheme": scheme, "tune": tune}
    if kind == "blast":
        bins = rng.choice([0, 0, 0, 2, 3])
        return {"kind": "blast", "root": rng.randint(3, 6), "levels": rng.randint(1, 2),
                "steps": 8 << bins if bins else _log_int(rng, 10, 60), "scheme": "mc" if bins else scheme,
                "path": "passes" if bins else "fused", "bins": bins}
    regrid = rng.choice([0, 0, 8])
    return {"kind": "shear", "root": rng.randint(4, 14), "levels": rng.randint(1, 2 if regrid else 3),
            "steps": 16 if regrid else _log_int(rng, 16, 100), "scheme": scheme, "regrid": regrid}


# ---------------- inputs ----------------
def _scheme(case):
    return {"limiter": case["scheme"], "isentropic": case["scheme"] == "koren"}


def _turbulence(n, seed):
    """problems.turbulence's field (solenoidal, k^-2 on 1 <= |k| <= 8, rms Mach 1) made on the GPU."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    k1 = torch.fft.fftfreq(n, d=1.0 / n, device="cuda", dtype=torch.float64)
    kx = torch.fft.rfftfreq(n, d=1.0 / n, device="cuda", dtype=torch.float64)
    k = torch.stack(torch.meshgrid(k1, k1, kx, indexing="ij"))           # (kz, ky, kx)
    kk = (k * k).sum(0)
    amp = torch.where((kk >= 1) & (kk <= 64), 1.0 / kk.clamp(min=1.0), 0.0)
    vk = torch.view_as_complex(torch.randn((3, *kk.shape, 2), generator=gen, device="cuda", dtype=torch.float64)) * amp
    vk = vk - k * (k * vk).sum(0) / kk.clamp(min=1.0)
    v = torch.fft.irfftn(vk, s=(n, n, n), dim=(1, 2, 3))
    v = v * (math.sqrt(5.0 / 3.0) / (v * v).sum(0).mean().sqrt())
    one = torch.ones(n, n, n, device="cuda", dtype=torch.float64)
    return {"rho": one, "vx": v[2], "vy": v[1], "vz": v[0], "p": one, "s": 0 * one}


def _walls(n, seed):
    """Gas at rest with a few smooth seeded bumps in density and pressure between reflecting walls
    along x, outflow along y and z."""
    rng = np.random.default_rng(seed)
    ax = [(torch.arange(m, device="cuda", dtype=torch.float64) + 0.5) / max(n) for m in n]
    z, y, x = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    rho, p = 1.0 + 0 * x, 1.0 + 0 * x
    for _ in range(6):
        c = rng.uniform(0.1, 0.9, 3) * np.asarray(n) / max(n)
        g = torch.exp(-((x - c[0]) ** 2 + (y - c[1]) ** 2 + (z - c[2]) ** 2) / (2 * rng.uniform(0.03, 0.12) ** 2))
        rho, p = rho + rng.uniform(0.2, 2.0) * g, p + rng.uniform(0.5, 8.0) * g
    return {"rho": rho, "vx": 0.1 * torch.sin(9 * x + y), "vy": 0 * x, "vz": 0 * x, "p": p, "s": rho - 1.0}


def _state(prims, gamma, dtype):
    """The state layout from primitives on the GPU: (cells, 4) u1 and u2 as host arrays."""
    rho, vx, vy, vz, p, s = (prims[k].reshape(-1) for k in ("rho", "vx", "vy", "vz", "p", "s"))
    ei = p / (gamma - 1.0)
    u1 = torch.stack([rho, rho * vx, rho * vy, rho * vz], 1)
    u2 = torch.stack([ei + 0.5 * rho * (vx * vx + vy * vy + vz * vz), ei, rho * s, 0 * rho], 1)
    return u1.to(dtype).cpu().numpy(), u2.to(dtype).cpu().numpy()


def _uniform_input(case, seed):
    """(SimConfig, u1, u2) of a uniform case."""
    n, kind = (case["nx"], case["ny"], case["nz"]), case["problem"]
    over = {"precision": case["precision"], **_scheme(case)}
    dtype = np.float64 if case["precision"] == 64 else np.float32
    if kind in ("kh", "quadrants", "sedov"):
        if kind == "kh":
            pb = problems.kelvin_helmholtz(n[0], seed=seed)
        elif kind == "sedov":
            pb = problems.sedov(n[0], seed=seed, t_end=math.inf)
        else:
            pb = problems.riemann_quadrants(n[0], seed)
            pb.n = n                              # fewer rows: the lower part of the square, kept centred
            rows = (pb.prims["rho"].shape[1] - n[1]) // 2
            pb.prims = {k: v[:, rows:rows + n[1], :] for k, v in pb.prims.items()}
        return (config_for(pb, **over), *pb.state(dtype))
    cfg = SimConfig(n=n, ndim=3, dx=1.0 / max(n), gamma=5.0 / 3.0, cfl=0.4, **over)
    if kind == "walls":
        cfg.bc_lo, cfg.bc_hi = (2, 1, 1), (2, 1, 1)
        prims = _walls(n, seed)
    else:
        prims = _turbulence(n[0], seed)
    return (cfg, *_state(prims, cfg.gamma, torch.float64 if dtype == np.float64 else torch.float32))


def _ensemble_sizes(case):
    """Grid sizes up to `largest`, a power of two apart, as many of each as a fixed draw gives."""
    most = case["largest"]
    return problems.ensemble_sizes(case["count"], seed=42, choices=tuple(max(32, most >> k) for k in (3, 2, 1, 0)))


def _ensemble_input(case, seed):
    cfg = SimConfig(n=(64, 64, 1), ndim=2, dx=1.0 / 64, gamma=1.4, bc_lo=(1, 1, 0), bc_hi=(1, 1, 0), cfl=0.4,
                    **_scheme(case))
    return cfg, [problems.riemann_quadrants(n, 1000 * seed + i).state()
                 for i, n in enumerate(_ensemble_sizes(case))]


@functools.lru_cache(maxsize=4)
def _tree(kind, root, levels):
    if kind == "blast":
        return problems.amr_blast(seed=7, root=root, max_level=levels)[:3]
    return problems.kh_adaptive(root=root, max_level=levels)


def _block_input(case, seed):
    """(SimConfig, blocks, root, u1, u2) of a block case: the workload's state with seeded noise."""
    kind, root = case["kind"], case["root"]
    blocks, dx0, prim_fn = _tree(kind, root, case["levels"])
    ndim = 3 if kind == "blast" else 2
    gamma = 1.4 if kind == "blast" else 5.0 / 3.0
    rng = np.random.default_rng(seed)

    def noisy(x, y, z):
        pr = dict(prim_fn(x, y, z))
        key = "rho" if kind == "blast" else "vy"
        pr[key] = pr[key] + rng.uniform(-1e-3, 1e-3, x.shape)
        return pr
    u1, u2 = amr_tree.blocks_state(blocks, dx0, noisy, gamma, ndim=ndim)
    n = BS * root
    cfg = SimConfig(n=(n, n, n if ndim == 3 else 1), ndim=ndim, dx=dx0, gamma=gamma, cfl=0.4, **_scheme(case))
    return cfg, blocks, (root, root, root if ndim == 3 else 1), u1, u2


# ---------------- a pass ----------------
def prepare(case, seed):
    if case["kind"] == "uniform":
        cfg, u1, u2 = _uniform_input(case, seed)
        sim = Sim(cfg)
        sim.set_state(u1, u2)
    elif case["kind"] == "ensemble":
        cfg, states = _ensemble_input(case, seed)
        sim = Ensemble(cfg, [(n, n) for n in _ensemble_sizes(case)])
        for i, s in enumerate(states):
            sim.set_state(i, *s)
    else:
        cfg, blocks, root, u1, u2 = _block_input(case, seed)
        if case["kind"] == "blast":
            sim = AmrSim(cfg, blocks, root, path=case["path"], time_bins=case["bins"])
        else:
            sim = AmrSim(cfg, blocks, root, path="passes", regrid_every=case["regrid"], max_level=case["levels"])
        sim.set_state(u1, u2)
    if case.get("tune"):
        sim.autotune()
    return {"sim": sim, "steps": case["steps"]}


def run(state):
    sim = state["sim"]
    sim.step(state["steps"])
    if isinstance(sim, Ensemble):
        return [sim.read_state(i) for i in range(sim.count)]
    u1, u2 = sim.read_state()
    out = {"u1": u1, "u2": u2}
    if isinstance(sim, AmrSim):
        out["blocks"] = sim.blocks
    ck = sim.clock()
    out["time"] = float(ck[0] + ck[1])
    return out


def _cells(case):
    if case["kind"] == "uniform":
        return case["nx"] * case["ny"] * case["nz"]
    if case["kind"] == "ensemble":
        return sum(n * n for n in _ensemble_sizes(case))
    blocks = _tree(case["kind"], case["root"], case["levels"])[0]
    return int(amr_tree.leaf_mask(blocks).sum()) * BS ** (3 if case["kind"] == "blast" else 2)


def work(case):
    """Each step reads and writes the 8 values of every cell once; the operations of one update
    (slopes, half step, a face solve per axis, the update) counted from the scheme."""
    per_cell = 64 * (2 if case.get("precision") == 64 else 1)
    flat = case["kind"] in ("ensemble", "shear") or case.get("nz") == 1
    flops = (420 if flat else 640) * (2 if case["scheme"] == "koren" else 1)
    updates = _cells(case) * case["steps"]
    return {"bytes": per_cell * updates, "flops": flops * updates}


# ---------------- the same in 64 bits ----------------
# A batch of blocks, each with its own dt: q holds (rho, vx, vy, vz, p, s) as [6, blocks, z, y, x],
# two ghost layers along every axis a block has (no z axis on flat grids).
class _Scheme:
    def __init__(self, cfg):
        self.lim, self.isen = cfg.limiter, cfg.isentropic
        self.gamma, self.gm1 = cfg.gamma, cfg.gamma - 1.0
        self.rho_floor, self.p_floor, self.eta, self.thresh = cfg.rho_floor, cfg.p_floor, cfg.eta_dual, cfg.shock_thresh
        self.ndim = cfg.ndim

    def prims(self, u):
        rho = u[0].clamp(min=self.rho_floor)
        return torch.stack([rho, u[1] / rho, u[2] / rho, u[3] / rho, (self.gm1 * u[5]).clamp(min=self.p_floor),
                            u[6] / rho])

    def sound(self, q):
        return torch.where(q[0] > 0, (self.gamma * q[4] / torch.where(q[0] > 0, q[0], 1.0)).sqrt(), 0.0)

    def rate(self, q):
        return q[1].abs() + q[2].abs() + q[3].abs() + self.ndim * self.sound(q)

    def edge(self, far, near, scale):
        """Twice the limited increment toward the face; scale: one per channel (Koren's)."""
        if self.lim != "koren":
            return _minmod(2 * far, 2 * near, 0.5 * (far + near))
        fr = (far + 2 * near) / 3
        s = 0.01 * scale
        k = 1 / s.abs().clamp(min=1e-37)
        plain = ((s * s >= 1e-30) & (s * s < 1e30)) | (s == 0)
        eta = torch.where(plain, (far * far + near * near) / (s * s).clamp(min=1e-30), (far * k) ** 2 + (near * k) ** 2)
        w = (1.5 - eta).clamp(0, 1)
        lim = _minmod(2 * far, 2 * near, fr)
        return torch.where(w == 1, fr, lim * (1 - w) + fr * w)

    def edges(self, lo, c, hi):
        """(up, down) increments of the six channels."""
        cs = self.sound(c)
        scale = torch.stack([c[0], cs, cs, cs, c[4], 0 * cs])
        below, above = c - lo, hi - c
        up = self.edge(below, above, scale)
        dn = self.edge(above, below, scale) if self.lim == "koren" else up
        if not self.isen:
            return up, dn
        ok = (lo[0] > 0) & (lo[4] > 0) & (c[0] > 0) & (c[4] > 0) & (hi[0] > 0) & (hi[4] > 0)
        gi = 1 / self.gamma
        tl = lo[0] * (c[4] / lo[4]) ** gi - c[0]
        tr = hi[0] * (c[4] / hi[4]) ** gi - c[0]

        def switch(v, width):
            return (2 - v / width).clamp(0, 1)
        ks = switch(torch.maximum((lo[4] - c[4]).abs(), (hi[4] - c[4]).abs()), 0.2 * c[4])
        ka = switch(torch.maximum(tl.abs(), tr.abs()), 0.01 * c[0])
        shear = torch.maximum((above[1:4] ** 2).sum(0).sqrt(), (below[1:4] ** 2).sum(0).sqrt())
        room = 0.01 * c[0] * ks * ka * switch(shear, 0.1 * cs.clamp(min=1e-30))
        bound = torch.maximum(0.25 * torch.minimum(below[0].abs(), above[0].abs()), room)
        out = []
        for x, sgn, far, near, wn in ((up, 1.0, -tl, tr, hi[0]), (dn, -1.0, tr, -tl, lo[0])):
            d = self.edge(far, near, c[0])
            pf = c[4] + 0.5 * sgn * x[4]
            rf = (c[0] + 0.5 * sgn * d) * (pf.clamp(min=1e-30) / c[4]) ** gi
            rf = torch.minimum(torch.maximum(rf, torch.minimum(c[0], wn)), torch.maximum(c[0], wn))
            off = torch.maximum(torch.minimum(2 * sgn * (rf - c[0]) - x[0], bound), -bound)
            x = x.clone()
            x[0] = torch.where(ok, x[0] + off, x[0])
            out.append(x)
        return out

    def half_steps(self, q, axes, dtdx, masks=None):
        """The half step of every cell and first-layer ghost, its flags, and the edge increments
        by axis. masks: per axis, zero where its slope is dropped."""
        c = _inner(q, axes, 1)
        inc, slope, big, fall = {}, {}, 0 * c[0], 0 * c[0]
        conv, jump = 0 * c[0], 0 * c[0]
        for a in axes:
            lo, hi = _shift(q, axes, a, -1), _shift(q, axes, a, 1)
            up, dn = self.edges(lo, c, hi)
            inc[a] = (up, dn)
            slope[a] = 0.5 * (up + dn) * (masks[a] if masks else 1.0)
            big = torch.maximum(big, torch.maximum(up[4].abs(), dn[4].abs()))
            drop = torch.minimum(0.5 * up[0], -0.5 * dn[0]) if self.lim == "koren" else -0.5 * up[0].abs()
            fall = torch.minimum(fall, drop)
            conv = conv + hi[1 + a] - lo[1 + a]
            jump = torch.maximum(jump, (hi[4] - lo[4]).abs() / torch.minimum(hi[4], lo[4]))
        h = 0.5 * dtdx
        div = sum(slope[a][1 + a] for a in axes)
        adv = sum(c[1 + a] * slope[a] for a in axes)
        o = c - h * adv
        o[0] -= h * c[0] * div
        o[4] -= h * c[0] * self.sound(c) ** 2 * div
        for a in axes:
            o[1 + a] -= h * slope[a][4] / c[0]
        first = ~((o[0] + fall > 0) & (o[4] - 0.5 * big > 0))
        o = torch.where(first, c, o)
        return o, ((conv < 0) & (jump > self.thresh)).to(q.dtype), first.to(q.dtype), inc

    def face(self, axis, L, R, hl, hr, w):
        """HLLC fluxes (m, mx, my, mz, e, ei, s) and the face velocity between two sides."""
        n, t1, t2 = 1 + axis, 1 + (axis + 1) % 3, 1 + (axis + 2) % 3
        lo_rho, lo_p = 0.5 * torch.minimum(hl[0], hr[0]), 0.5 * torch.minimum(hl[4], hr[4])
        sides = []
        for s in (L, R):
            rho = torch.maximum(s[0], lo_rho.clamp(min=self.rho_floor))
            p = torch.maximum(s[4], lo_p.clamp(min=self.p_floor))
            v, ei = s[n], p / self.gm1
            E = ei + 0.5 * rho * (s[1] ** 2 + s[2] ** 2 + s[3] ** 2)
            U = torch.stack([rho, rho * v, rho * s[t1], rho * s[t2], E])
            F = torch.stack([rho * v, rho * v * v + p, rho * v * s[t1], rho * v * s[t2], (E + p) * v])
            sides.append((rho, p, v, ei, U, F, (self.gamma * p / rho).sqrt(), s[t1], s[t2], s[5]))
        (rl, pl, vl, el, Ul, Fl, cl, a1, a2, xl), (rr, pr, vr, er, Ur, Fr, cr, b1, b2, xr) = sides
        sl, sr = torch.minimum(vl - cl, vr - cr), torch.maximum(vl + cl, vr + cr)
        ql, qr = rl * (sl - vl), rr * (sr - vr)
        star = (ql < 0) & (qr > 0)
        hll = (sr * Fl - sl * Fr + sl * sr * (Ur - Ul)) / (sr - sl)
        sm = (pr - pl + vl * ql - vr * qr) / torch.where(ql - qr != 0, ql - qr, 1.0)
        left = sm >= 0

        def pick(x, y):
            return torch.where(left, x, y)
        S, rho, un, u1, u2, p, q = pick(sl, sr), pick(rl, rr), pick(vl, vr), pick(a1, b1), pick(a2, b2), pick(pl, pr), pick(ql, qr)
        F, E = pick(Fl, Fr), pick(Ul[4], Ur[4])
        k = (sm - un) / (S - sm)
        dr = rho * k
        c = F + S * torch.stack([dr, sm * dr + rho * (sm - un), dr * u1, dr * u2,
                                 E * k + (rho + dr) * (sm - un) * (sm + p / q)])
        c = torch.where(w != 0, c * (1 - w) + hll * w, c)
        f = torch.where(star, c, hll)
        vn = torch.where(star, sm, 0.5 * (vl + vr))
        f, vn = torch.where(sr <= 0, Fr, f), torch.where(sr <= 0, vr, vn)
        f, vn = torch.where(sl >= 0, Fl, f), torch.where(sl >= 0, vl, vn)
        upw = f[0] >= 0
        out = [None] * 8
        out[0], out[n], out[t1], out[t2], out[4] = f[0], f[1], f[2], f[3], f[4]
        out[5] = f[0] * torch.where(upw, el / rl, er / rr)
        out[6] = f[0] * torch.where(upw, xl, xr)
        out[7] = vn
        return torch.stack(out)

    def fluxes(self, axes, h, shock, first, inc):
        """Per axis the fluxes through every face of the blocks' cells (n + 1 along the axis)."""
        out = {}
        for a in axes:
            up, dn = inc[a]
            hs = 0.5 * (1 - first)

            def side(x, j):
                return _faces(x, axes, a, j)
            L, R = side(h + hs * up, 0), side(h - hs * dn, 1)
            w = torch.maximum(side(shock[None], 0), side(shock[None], 1))[0]
            out[a] = self.face(a, L, R, side(h, 0), side(h, 1), w)
        return out

    def advance(self, u, f, axes, p_half, dtdx):
        net = 0
        for a in axes:
            d = f[a].ndim - 1 - a
            n = f[a].shape[d] - 1
            net = net + f[a].narrow(d, 0, n) - f[a].narrow(d, 1, n)
        o = u + dtdx * net[:7]
        o[5] += dtdx * p_half.clamp(min=self.p_floor) * net[7]
        o[0] = o[0].clamp(min=self.rho_floor)
        ke = 0.5 * (o[1] ** 2 + o[2] ** 2 + o[3] ** 2) / o[0]
        eth, emin = o[4] - ke, self.p_floor / self.gm1
        total = (eth > self.eta * o[4]) & (eth >= emin) & (eth >= 0)
        ei = torch.where(total, eth, o[5].clamp(min=emin))
        o[4], o[5] = torch.where(total, o[4], ke + ei), ei
        return o


def _minmod(*v):
    v = torch.stack(v)
    return torch.where((v > 0).all(0), v.min(0).values, torch.where((v < 0).all(0), v.max(0).values, 0.0))


def _inner(x, axes, by):
    for a in axes:
        x = x.narrow(x.ndim - 1 - a, by, x.shape[x.ndim - 1 - a] - 2 * by)
    return x


def _shift(x, axes, axis, by):
    """The cells and first-layer ghosts, moved by one along an axis."""
    for a in axes:
        d = x.ndim - 1 - a
        x = x.narrow(d, 1 + (by if a == axis else 0), x.shape[d] - 2)
    return x


def _faces(x, axes, axis, j):
    """From cells with one ghost layer: the cells left (j 0) or right (j 1) of the axis's faces."""
    for a in axes:
        d = x.ndim - 1 - a
        x = x.narrow(d, j, x.shape[d] - 1) if a == axis else x.narrow(d, 1, x.shape[d] - 2)
    return x


def _cons(u1, u2, shape):
    """The 7 conserved values as [7, blocks, z, y, x] in 64 bits."""
    a, b = (torch.from_numpy(np.asarray(u)).to("cuda", torch.float64) for u in (u1, u2))
    return torch.cat([a, b[:, :3]], 1).t().reshape(7, *shape).contiguous()


def _pair(u):
    u = u.reshape(7, -1)
    return u[:4].t().contiguous().cpu().numpy(), torch.cat([u[4:], 0 * u[:1]]).t().contiguous().cpu().numpy()


def _ghosted(x, axes, bc, depth):
    """Cells with `depth` ghost layers by the boundary maps (0 periodic, 1 outflow, 2 reflecting);
    component 1 + axis of a reflected ghost turns its sign."""
    for a in axes:
        d, n = x.ndim - 1 - a, x.shape[x.ndim - 1 - a]
        i = torch.arange(-depth, n + depth, device=x.device)
        out = (i < 0) | (i >= n)
        at = {0: i % n, 1: i.clamp(0, n - 1), 2: torch.where(i < 0, -1 - i, torch.where(i >= n, 2 * n - 1 - i, i))}[bc[a]]
        x = x.index_select(d, at).clone()
        if bc[a] == 2:
            x[1 + a] *= torch.where(out, -1.0, 1.0).view([-1 if e == d - 1 else 1 for e in range(x.ndim - 1)])
    return x


def _run_grids(cfg, u, dx, steps):
    """Grids of one size, [7, grids, z, y, x], each advanced `steps` steps with its own dt."""
    S = _Scheme(cfg)
    axes = (0, 1) if u.shape[2] == 1 else (0, 1, 2)
    t = torch.zeros(u.shape[1], device=u.device, dtype=u.dtype)
    for _ in range(steps):
        w = S.prims(u)
        dt = cfg.cfl * dx / S.rate(w).flatten(1).max(1).values
        k = (dt / dx).view(-1, 1, 1, 1)
        h, shock, first, inc = S.half_steps(_ghosted(w, axes, cfg.bc_lo, 2), axes, k)
        # a ghost's half step is that of the cell it stands for
        g = _ghosted(_inner(torch.cat([h, shock[None], first[None]]), axes, 1), axes, cfg.bc_lo, 1)
        f = S.fluxes(axes, g[:6], g[6], g[7], inc)
        u = S.advance(u, f, axes, _inner(h[4], axes, 1), k)
        t = t + dt
    return u, t


class _Blocks:
    """A static tree's links, as index lists by face (0 -x, 1 +x, 2 -y, ...; all axes periodic)."""

    def __init__(self, blocks, root, axes):
        self.axes, at = axes, {tuple(b): i for i, b in enumerate(blocks.tolist())}
        kids = [[(x, y, z) for x in (0, 1)] for z in ((0, 1) if 2 in axes else (0,)) for y in (0, 1)]
        self.octs = [o for row in kids for o in row]
        child = {i: [at.get((b[0] + 1, *(2 * b[1 + a] + o[a] for a in range(3)))) for o in self.octs]
                 for b, i in at.items()}
        self.parents = [i for i, c in child.items() if c[0] is not None]
        inside = set(self.parents)
        self.leaves = [i for i in range(len(blocks)) if i not in inside]
        self.pos = {s: k for k, s in enumerate(self.leaves)}
        self.child = child
        self.same = {k: [] for k in range(2 * len(axes))}      # (slot, neighbour of its level)
        self.coarse = {k: [] for k in range(2 * len(axes))}    # (leaf, coarser leaf)
        for b, i in at.items():
            for a in axes:
                for up in (0, 1):
                    c = list(b)
                    c[1 + a] = (c[1 + a] + (1 if up else -1)) % (root[a] << b[0])
                    j = at.get(tuple(c))
                    if j is not None:
                        self.same[2 * a + up].append((i, j))
                    elif i in self.pos:
                        self.coarse[2 * a + up].append((i, at[(b[0] - 1, *(v >> 1 for v in c[1:]))]))
        self.blocks, self.root = torch.as_tensor(blocks, device="cuda").long(), root

    def pairs(self, which, k):
        v = torch.tensor(which[k], device="cuda").reshape(-1, 2)
        return v[:, 0], v[:, 1]


def _slab(x, axes, k, lo, n, pad):
    """Layers [lo, lo + n) along face k's axis of blocks padded by `pad`, the cells of the others."""
    for a in axes:
        d = x.ndim - 1 - a
        x = x.narrow(d, lo + pad, n) if a == k // 2 else x.narrow(d, pad, BS)
    return x


def _run_blocks(cfg, blocks, root, u, steps):
    """Leaves of a static tree, [7, blocks, z, y, x], with one dt."""
    S, axes = _Scheme(cfg), ((0, 1) if cfg.ndim == 2 else (0, 1, 2))
    T = _Blocks(blocks, root, axes)
    dev, nl = u.device, len(T.leaves)
    leaves = torch.tensor(T.leaves, device=dev)
    pos = torch.full((len(blocks),), -1, device=dev)
    pos[leaves] = torch.arange(nl, device=dev)
    dx = cfg.dx / 2.0 ** T.blocks[leaves, 0].double()
    links = {k: T.pairs(T.same, k) for k in T.same}
    coarse = {k: T.pairs(T.coarse, k) for k in T.coarse}
    ok_face = torch.zeros(len(blocks), 6, dtype=torch.bool, device=dev)
    for k, (i, _) in links.items():
        ok_face[i, k] = True
    size = [BS + 4 if a in axes else 1 for a in (2, 1, 0)]
    # texels outside along more than one axis are never filled; at a ghost's rim the slopes along
    # the face are dropped
    out = [((torch.arange(n, device=dev) < 2) | (torch.arange(n, device=dev) >= n - 2)) & (n > 1) for n in size]
    count = out[0][:, None, None].int() + out[1][None, :, None].int() + out[2][None, None, :].int()
    filled = (count <= 1).to(u.dtype)
    masks = {}
    for a in axes:
        i = torch.arange(-1, BS + 1, device=dev)
        rim = ((i == 0) | (i == BS - 1)).view([-1 if d == 2 - a else 1 for d in range(3)])
        ghost = torch.zeros((), dtype=torch.bool, device=dev)
        for b in axes:
            if b != a:
                ghost = ghost | ((i < 0) | (i >= BS)).view([-1 if d == 2 - b else 1 for d in range(3)])
        masks[a] = (~(rim & ghost)).to(u.dtype)
    kids = {}
    for o, oc in enumerate(T.octs):
        pc = [(p, T.child[p][o]) for p in T.parents if T.child[p][o] in T.pos]
        kids[oc] = torch.tensor(pc, device=dev).reshape(-1, 2)
    t = torch.zeros((), device=dev, dtype=u.dtype)
    for _ in range(steps):
        # parents' cells: the mean of their leaf children's
        for oc, pc in kids.items():
            m = u[:, pc[:, 1]]
            m = m.reshape(7, len(pc), -1, 2 if 2 in axes else 1, BS // 2, 2, BS // 2, 2).mean((3, 5, 7))
            at = tuple(slice(BS // 2 * oc[a], BS // 2 * (oc[a] + 1)) if a in axes else slice(0, 1) for a in (2, 1, 0))
            u[(slice(None), pc[:, 0], *at)] = m
        x = torch.zeros(7, len(blocks), *size, device=dev, dtype=u.dtype)
        _inner(x, axes, 2)[:] = u
        for k, (i, j) in links.items():
            up = k & 1
            _slab(x, axes, k, BS if up else -2, 2, 2)[:, i] = _slab(u, axes, k, 0 if up else BS - 2, 2, 0)[:, j]
        g = x[:, leaves]
        for k, (i, j) in coarse.items():
            if len(i):
                _slab(g, axes, k, BS if k & 1 else -2, 2, 2)[:, pos[i]] = _from_coarse(S, T, x, ok_face, i, j, k)
        w = S.prims(g) * filled
        inner = _inner(w, axes, 2)
        dt = cfg.cfl / (S.rate(inner).flatten(1).max(1).values / dx).max()
        dtdx = (dt / dx).view(-1, 1, 1, 1)
        h, shock, first, inc = S.half_steps(w, axes, dtdx, masks)
        hs = torch.cat([h, shock[None], first[None]])
        src = hs.clone()
        for k, (i, j) in links.items():        # same-level leaves: the half steps of their own cells
            sel = (pos[i] >= 0) & (pos[j] >= 0)
            up = k & 1
            _slab(hs, axes, k, BS if up else -1, 1, 1)[:, pos[i[sel]]] = _slab(src, axes, k, 0 if up else BS - 1, 1, 1)[:, pos[j[sel]]]
        f = S.fluxes(axes, hs[:6], hs[6], hs[7], inc)
        for k, (i, j) in links.items():        # refined neighbours: the mean of their fluxes
            sel = (pos[i] >= 0) & (pos[j] < 0)
            if bool(sel.any()):
                _match(T, f, k, i[sel], j[sel], pos)
        u = u.clone()
        u[:, leaves] = S.advance(u[:, leaves], f, axes, _inner(h[4], axes, 1), dtdx)
        t = t + dt
    parents = torch.tensor(T.parents, device=dev, dtype=torch.long)
    return u, t, parents


def _from_coarse(S, T, x, ok_face, i, j, k):
    """The two ghost layers of leaves i on face k, interpolated from the coarser leaves j."""
    axes, lev = T.axes, T.blocks[j, 0]
    cell, par = {}, {}
    for a in axes:
        n = torch.arange(2, device=x.device) + (BS if k & 1 else -2) if a == k // 2 else torch.arange(BS, device=x.device)
        gf = T.blocks[i, 1 + a][:, None] * BS + n
        gc = torch.div(gf, 2, rounding_mode="floor") % ((T.root[a] * BS) << lev)[:, None]
        shape = [len(i)] + [len(n) if d == 2 - a else 1 for d in range(3)]
        cell[a], par[a] = (gc - T.blocks[j, 1 + a][:, None] * BS).view(shape), (gf % 2).view(shape)
    s = j.view(-1, 1, 1, 1)

    def at(a, by):
        ix = [cell[b] + 2 + (by if b == a else 0) if b in axes else torch.zeros_like(s) for b in (2, 1, 0)]
        return x[:, s, ix[0], ix[1], ix[2]]
    c = at(None, 0)
    slopes = {}
    for a in axes:
        m, p = at(a, -1), at(a, 1)
        good = (ok_face[:, 2 * a][s] | (cell[a] > 0)) & (ok_face[:, 2 * a + 1][s] | (cell[a] < BS - 1))
        d = _minmod(2 * (c - m), 2 * (p - c), 0.5 * (p - m))
        v = [y[1:4] / y[0].clamp(min=S.rho_floor) for y in (m, c, p)]
        dv = _minmod(2 * (v[1] - v[0]), 2 * (v[2] - v[1]), 0.5 * (v[2] - v[0]))
        d[1:4] = v[1] * d[0] + c[0] * dv
        slopes[a] = torch.where(good, d, 0.0)
    spread = sum(slopes[a].abs() for a in axes)
    fit = torch.ones_like(c[0])
    for q in (0, 4, 5):
        fit = torch.minimum(fit, 0.5 * c[q].clamp(min=0) / (0.25 * spread[q]).clamp(min=1e-37))
    return c + sum(fit * (par[a] - 0.5) * 0.5 * slopes[a] for a in axes)


def _match(T, f, k, i, j, pos):
    """The fluxes of leaves i through face k, whose neighbours j are refined: the fine means."""
    a, up = k // 2, k & 1
    across = [b for b in T.axes if b != a]
    d = f[a].ndim - 1 - a
    for o, oc in enumerate(T.octs):
        if oc[a] == up:                       # the children that do not touch the face
            continue
        ch = torch.tensor([T.child[int(p)][o] for p in j.tolist()], device=pos.device)
        fine = f[a].select(d, 0 if up else BS)[:, pos[ch]]
        rest = [b for b in (2, 1, 0) if b != a]
        shape = [8, len(ch)]
        for b in rest:
            shape += [BS // 2, 2] if b in T.axes else [1, 1]
        fine = fine.reshape(shape).mean((3, 5))
        at = tuple(slice(BS // 2 * oc[b], BS // 2 * (oc[b] + 1)) if b in across else slice(None) for b in rest)
        f[a].select(d, BS if up else 0)[(slice(None), pos[i], *at)] = fine


def exact(case, seed):
    """run's answer in 64 bits, or None where this would take too long or has no such value."""
    if _cells(case) * case["steps"] > 9e8 or case.get("bins") or case.get("regrid"):
        return None
    if case["kind"] == "uniform":
        cfg, u1, u2 = _uniform_input(case, seed)
        u, t = _run_grids(cfg, _cons(u1, u2, (1, *cfg.n[::-1])), cfg.dx, case["steps"])
        return {"u1": _pair(u)[0], "u2": _pair(u)[1], "time": float(t[0])}
    if case["kind"] == "ensemble":
        cfg, states = _ensemble_input(case, seed)
        sizes, out = _ensemble_sizes(case), [None] * case["count"]
        for n in sorted(set(sizes)):
            sel = [i for i, m in enumerate(sizes) if m == n]
            u = torch.cat([_cons(*states[i], (1, 1, n, n)) for i in sel], 1)
            u, _ = _run_grids(cfg, u, 1.0 / n, case["steps"])
            for j, i in enumerate(sel):
                out[i] = _pair(u[:, j])
        return out
    cfg, blocks, root, u1, u2 = _block_input(case, seed)
    shape = (len(blocks), BS if cfg.ndim == 3 else 1, BS, BS)
    u, t, parents = _run_blocks(cfg, blocks, root, _cons(u1, u2, shape), case["steps"])
    u[:, parents] = _cons(u1, u2, shape)[:, parents]      # parents' cells are never written
    return {"u1": _pair(u)[0], "u2": _pair(u)[1], "time": float(t), "blocks": None}
