"""The framework's work as timed cases: SuLi's pressure step through the
public entry points of ``suli_amd.solver``.

Each case is one call (or one time step's calls) as a SuLi program makes it,
at sizes of the repository's own workloads (the 64x64x32 Poisson problem, the
256x128x96 sloshing tank, the 384x192x128 stretched masked cylinder, uneven
batches of 32..128 cells a side, SuLi-IT's 256x128x48 state), and at generic
odd sizes between them.

Solves run to a 1e-12 relative residual, where the pressure is settled to
about 1e-9: there it no longer shows in which order the iteration's sums were
taken.  (The reference's own absolute rule, r.r <= 1e-4/(nx ny nz), is about
1e-10 relative on these velocity fields.)  Every solve starts cold, from
prd1 = 0, as the first of a run does.

A program keeps one solver for its whole run and hands it new fields, so the
states of one kind share a solver (one per set of options) here too.
"""
from __future__ import annotations

import ctypes as C
import dataclasses
import math

import numpy as np
import torch

from suli_amd import cases
from suli_amd.solver import PressureSolver

TOL = 1e-12
GZ = 9.80665
PI = math.pi


def listed():
    return [
        # one small two-phase tank: the smallest grids of a batch or a test
        # run, where launches and latency count
        dict(name="tank_40x32x24_mixed", kind="solve", field="tank", precision="mixed", nx=40, ny=32, nz=24),
        # the single-phase Poisson problem with a p = 0 lid, FP64, the
        # Fortran shim's default precision
        dict(name="poisson_lid_64x64x32_fp64", kind="solve", field="poisson_lid", precision="fp64", nx=64, ny=64,
             nz=32),
        # the headline: the two-phase sloshing tank, mixed precision and FP64,
        # tile shapes from the autotuner as the benchmark runs them
        dict(name="tank_256x128x96_mixed", kind="solve", field="tank", precision="mixed", nx=256, ny=128, nz=96,
             autotune=True),
        dict(name="tank_256x128x96_fp64", kind="solve", field="tank", precision="fp64", nx=256, ny=128, nz=96,
             autotune=True),
        # the largest: stretched dz, a masked-out cylinder
        dict(name="cylinder_384x192x128_mixed", kind="solve", field="cylinder", precision="mixed", nx=384, ny=192,
             nz=128),
        # one IPA time step on an odd, x-periodic grid: exp_press, then the
        # solve with the constant density
        dict(name="ipa_191x95x97_mixed", kind="ipa", precision="mixed", nx=191, ny=95, nz=97, periodic_x=True),
        # twelve independent uneven tanks solved together
        dict(name="batch_12_mixed", kind="batch", precision="mixed", count=12, lo=32, hi=128),
        # SuLi-IT's non-hydrostatic solve
        dict(name="suli_it_256x128x48_mixed", kind="it", precision="mixed", nx=256, ny=128, nz=48),
        # one RK sub-stage as the Fortran shim runs it: host arrays through
        # graddin and posdin
        dict(name="dropin_128x96x64_fp64", kind="dropin", precision="fp64", nx=128, ny=96, nz=64),
        # the once-per-stage kernels on resident fields: the velocity
        # correction; the hydrostatic step; the density from the level set
        # with its surface-tension gradients
        dict(name="posdin_256x128x96", kind="posdin", nx=256, ny=128, nz=96),
        dict(name="hydro_256x128x96", kind="hydro", nx=256, ny=128, nz=96),
        dict(name="level_set_256x128x96", kind="levelset", nx=256, ny=128, nz=96),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One case of the ranges above: any kind, each side of the grid spread
    over its logarithm (odd sizes among them), never more cells than the
    largest listed case of its kind."""
    kind = rng.choice(["solve"] * 5 + ["ipa", "batch", "it", "dropin", "posdin", "hydro", "levelset"])
    if kind == "batch":
        return dict(kind=kind, precision=rng.choice(["mixed", "fp64"]), count=rng.randint(3, 12), lo=32,
                    hi=rng.choice([64, 96, 128]))
    most = {"solve": 256 * 128 * 96, "it": 256 * 128 * 48, "dropin": 128 * 96 * 64, "ipa": 191 * 95 * 97}.get(
        kind, 256 * 128 * 96)
    while True:
        nx, ny, nz = _logint(rng, 24, 384), _logint(rng, 16, 192), _logint(rng, 16, 128)
        if nx * ny * nz <= most:
            break
    c = dict(kind=kind, nx=nx, ny=ny, nz=nz)
    if kind in ("solve", "ipa", "it", "dropin"):
        c["precision"] = rng.choice(["mixed", "mixed", "fp64"])
    if kind == "solve":
        c["field"] = rng.choice(["tank", "tank", "poisson_lid", "cylinder", "stretched"])
    if kind in ("ipa", "posdin") or c.get("field") in ("tank", "stretched"):
        c["periodic_x"] = rng.random() < 0.3
    return c


# ---- solvers ---------------------------------------------------------------
_solvers: dict = {}


def _solver(precision="fp64", autotune=False) -> PressureSolver:
    key = (precision, autotune)
    if key not in _solvers:
        _solvers[key] = PressureSolver(precision=precision, stop_rule="relative", tol=TOL, verbose=False,
                                       autotune=autotune)
    return _solvers[key]


# ---- inputs ----------------------------------------------------------------
def _make(case, seed) -> cases.Case:
    """The synthetic fields of a one-grid case (host arrays)."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    px = bool(case.get("periodic_x"))
    field = case.get("field", "tank")
    if field == "poisson_lid":
        return cases.config1(seed=seed, nx=nx, ny=ny, nz=nz, top_dirichlet=True)
    if field == "cylinder":
        c = cases.config3(seed=seed, nx=nx, ny=ny, nz=nz)
        cases.make_stretched_compatible(c)
        return c
    if field == "stretched":
        c = cases.random_case(nx, ny, nz, seed, periodic_x=px, stretched=True)
        cases.make_stretched_compatible(c)
        return c
    if px:
        return cases.random_case(nx, ny, nz, seed, periodic_x=True)
    return cases.config2(seed=seed, nx=nx, ny=ny, nz=nz)


def _up(a):
    """A device copy of a Fortran-ordered array (dims reversed), or None."""
    return None if a is None else torch.from_numpy(np.ascontiguousarray(np.asarray(a).T)).cuda()


class Resident:
    """Fields resident on the device, as the _dev entry points take them."""

    NAMES = ("u", "v", "w", "rho", "prd1", "obs_lsx", "obs_lsy", "obs_lsz", "dz", "dzz", "solid", "hs")

    def __init__(self, grid, fields):
        self.t = {n: _up(getattr(fields, n, None)) for n in self.NAMES}
        self.t["dz"], self.t["dzz"] = _up(grid.dzv), _up(grid.dzzv)
        self.ptrs = {n: _ptr(t) for n, t in self.t.items()}


def _ptr(t):
    return None if t is None else C.c_void_p(t.data_ptr())


def _rough_pressure(shape, seed):
    """A smooth pressure with noise on the halo box (device)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    z = torch.linspace(1.0, 0.0, shape[0], dtype=torch.float64, device="cuda")[:, None, None]
    return 50.0 * z + torch.rand(shape, dtype=torch.float64, device="cuda", generator=g)


def prepare(case, seed):
    kind = case["kind"]
    s = dict(kind=kind)
    if kind == "batch":
        s["solver"] = _solver(case["precision"])
        s["items"] = [(c.grid, Resident(c.grid, c.fields)) for c in _batch(case, seed)]
    elif kind == "it":
        s["solver"] = _solver(case["precision"])
        s["grid"], f = cases.it_case(case["nx"], case["ny"], case["nz"], seed)
        s["t"] = {a.name: _up(getattr(f, a.name)) for a in dataclasses.fields(f)}
        s["ptrs"] = {n: _ptr(t) for n, t in s["t"].items()}
    elif kind == "dropin":
        s["solver"] = _solver(case["precision"])
        c = _make(case, seed)
        s["grid"], s["fields"] = c.grid, c.fields
        # the velocities posdin corrects, beside those graddin reads (a time
        # loop forms new ones for every sub-stage)
        s["after"] = dataclasses.replace(c.fields, u=c.fields.u.copy(order="F"), v=c.fields.v.copy(order="F"),
                                         w=c.fields.w.copy(order="F"))
    else:
        s["solver"] = _solver(case.get("precision", "fp64"), bool(case.get("autotune")))
        c = _make(case, seed)
        g, f = c.grid, c.fields
        if kind == "ipa":
            g.t_press, g.rho_f1 = 2, 1000.0
        if kind in ("hydro", "levelset"):
            height = (0.4 + 0.2 * np.random.default_rng(seed).random()) * g.nz * g.dz
            ls = cases.sloshing_level_set(g, height, 0.04 * g.nz * g.dz)
            s["eps"] = 1.5 * max(g.dx, g.dy, g.dz)
            f.hs = np.asfortranarray(cases.heaviside_rho(ls, s["eps"], 0.0, 1.0))
            f.rho = np.asfortranarray(1.2 * (1.0 - f.hs) + 1000.0 * f.hs)
            s["ls"] = _up(ls)
        s["grid"], s["df"] = g, Resident(g, f)
        t = s["df"].t
        if kind == "posdin":
            t["prd1"].copy_(_rough_pressure(t["prd1"].shape, seed))
        elif kind == "ipa":
            s["prd0"] = _rough_pressure(t["prd1"].shape, seed)
            s["prdn"] = _rough_pressure(t["prd1"].shape, seed + 7)
            s["p"] = [torch.empty(sh, dtype=torch.float64, device="cuda") for sh in
                      ((g.nz, g.ny, g.nx + 1), (g.nz, g.ny + 1, g.nx), (g.nz + 1, g.ny, g.nx))]
        elif kind == "levelset":
            s["out"] = {n: torch.empty_like(s["ls"]) for n in ("hs", "rho", "mu", "hsx", "hsy", "hsz")}
    torch.cuda.synchronize()
    return s


def _batch(case, seed):
    out = []
    for i, (nx, ny, nz) in enumerate(cases.log_uniform_sizes(case["count"], case["count"], case["lo"], case["hi"])):
        r = np.random.default_rng(1000 * seed + i)
        out.append(cases.random_case(nx, ny, nz, 1000 * seed + i, ratio=float(r.choice([1.0, 10.0, 1000.0])),
                                     surface=float(r.uniform(0.3, 0.7))))
    return out


# ---- one pass --------------------------------------------------------------
def run(s):
    kind, solver = s["kind"], s["solver"]
    if kind == "solve":
        t = s["df"].t["prd1"]
        solver.dev_zero(s["df"].ptrs["prd1"], t.numel() * 8)
        st = solver.graddin_dev(s["grid"], s["df"])
        return dict(prd1=t, status=int(st.status))
    if kind == "ipa":
        t, p = s["df"].t["prd1"], s["p"]
        solver.exp_press_dev(s["grid"], s["df"].ptrs["rho"], _ptr(s["prdn"]), _ptr(s["prd0"]), *map(_ptr, p))
        solver.dev_zero(s["df"].ptrs["prd1"], t.numel() * 8)
        st = solver.graddin_dev(s["grid"], s["df"])
        return dict(prd0=s["prd0"], px=p[0], py=p[1], pz=p[2], prd1=t, status=int(st.status))
    if kind == "batch":
        for _, df in s["items"]:
            solver.dev_zero(df.ptrs["prd1"], df.t["prd1"].numel() * 8)
        sts = solver.graddin_batch_dev(s["items"])
        return dict(prd1=[df.t["prd1"] for _, df in s["items"]], status=max(int(st.status) for st in sts))
    if kind == "it":
        solver.dev_zero(s["ptrs"]["prd1"], s["t"]["prd1"].numel() * 8)
        st = solver.it_graddin_dev(s["grid"], s["ptrs"])
        return dict(prd1=s["t"]["prd1"], status=int(st.status))
    if kind == "dropin":
        s["fields"].prd1[...] = 0.0
        st = solver.graddin(s["grid"], s["fields"])
        prd = solver.posdin(s["grid"], s["after"])
        a = s["after"]
        return dict(prd=prd, u=a.u, v=a.v, w=a.w, status=int(st.status))
    if kind == "posdin":
        solver.posdin_dev(s["grid"], s["df"])
        return dict((n, s["df"].t[n]) for n in ("u", "v", "w"))
    if kind == "hydro":
        solver.pressh_dev(s["grid"], s["df"], GZ)
        solver.posdin_hydro_dev(s["grid"], s["df"])
        return dict((n, s["df"].t[n]) for n in ("prd1", "u", "v", "w"))
    if kind == "levelset":
        o = s["out"]
        solver.heaviside_tens_dev(s["grid"], _ptr(s["ls"]), s["eps"], 1000.0, 1.8e-5, 1e-3, _ptr(o["rho"]),
                                  _ptr(o["hsx"]), _ptr(o["hsy"]), _ptr(o["hsz"]), _ptr(o["hs"]), _ptr(o["mu"]))
        return o
    raise ValueError(kind)


# ---- the least a pass can move --------------------------------------------
# words (8 bytes) per cell, inputs read once and outputs written once: a solve
# reads u, v, w, rho and the initial prd1 and writes prd1; SuLi-IT's reads the
# three thicknesses instead of rho; posdin reads u, v, w, rho, prd1 and writes
# u, v, w; ...
WORDS = {"solve": 6, "ipa": 6 + 7, "batch": 6, "it": 8, "dropin": 6 + 8 + 1, "posdin": 8, "hydro": 2 + 8,
         "levelset": 7}
# operations per cell: one operator application and divergence; the
# gradients; the column integral and continuity; three WENO5 lines both ways
FLOPS = {"solve": 30, "ipa": 50, "batch": 30, "it": 35, "dropin": 50, "posdin": 21, "hydro": 40, "levelset": 600}


def work(case):
    if case["kind"] == "batch":
        n = sum(a * b * c for a, b, c in cases.log_uniform_sizes(case["count"], case["count"], case["lo"], case["hi"]))
    else:
        n = case["nx"] * case["ny"] * case["nz"]
    return {"bytes": 8.0 * WORDS[case["kind"]] * n, "flops": float(FLOPS[case["kind"]]) * n}


# ---- 64-bit values in plain torch -----------------------------------------
def _interp(g, rho):
    """Face values of a cell field, (nz, ny, nx) order."""
    fx = torch.empty((g.nz, g.ny, g.nx + 1), dtype=torch.float64, device=rho.device)
    fy = torch.empty((g.nz, g.ny + 1, g.nx), dtype=torch.float64, device=rho.device)
    fz = torch.empty((g.nz + 1, g.ny, g.nx), dtype=torch.float64, device=rho.device)
    fx[:, :, 1:-1] = (rho[:, :, 1:] + rho[:, :, :-1]) * 0.5
    if g.ccx0 == 0:
        fx[:, :, 0] = fx[:, :, -1] = (rho[:, :, 0] + rho[:, :, -1]) * 0.5
    else:
        fx[:, :, 0], fx[:, :, -1] = fx[:, :, 1], fx[:, :, -2]
    fy[:, 1:-1] = (rho[:, 1:] + rho[:, :-1]) * 0.5
    fy[:, 0], fy[:, -1] = fy[:, 1], fy[:, -2]
    if g.stretched:
        d = _up(g.dzv)[1:-1, None, None]
        fz[1:-1] = (rho[1:] * d[1:] + rho[:-1] * d[:-1]) / (d[1:] + d[:-1])
    else:
        fz[1:-1] = (rho[1:] + rho[:-1]) * 0.5
    fz[0], fz[-1] = fz[1], fz[-2]
    return fx, fy, fz


def _halo(p, px, top):
    """The halo box: mirrored (x periodic on px); the top ghosts times top."""
    out = torch.nn.functional.pad(p[None, None], (1, 1, 1, 1, 1, 1), mode="replicate")[0, 0].clone()
    if px:
        out[:, :, 0], out[:, :, -1] = out[:, :, -2], out[:, :, 1]
    out[-1] *= top
    return out


def _cg(apply, d, q, keep, null):
    """Jacobi-preconditioned CG to the accuracy of 64 bits: solved, then the
    residual solved for once more.  keep: 1 in cells that are solved for."""
    def once(b, tol):
        x, r = torch.zeros_like(b), b.clone()
        z = r / d
        p, rz = z.clone(), (r * z).sum()
        first = float((r * r / d).sum())
        for it in range(8000):
            ap = apply(p)
            a = rz / (p * ap).sum()
            x += a * p
            r -= a * ap
            z = r / d
            rn = (r * z).sum()
            p.mul_(rn / rz).add_(z)
            rz = rn
            if it % 25 == 24 and float(rz) <= tol * tol * first:
                break
        return x

    def consistent(b):
        b = b * keep
        return b - (b.sum() / (d * keep).sum()) * d * keep if null else b

    b = consistent(q)
    x = once(b, 1e-14)
    return x + once(consistent(b - apply(x)), 1e-4)


def _pressure(g, f):
    """prd1 (whole halo box) of graddin from prd1 = 0: the zero-flux (x
    periodic, lid at p = 0) projection system, in the gauge sum(d p) = 0."""
    u, v, w, rho = _up(f.u), _up(f.v), _up(f.w), _up(f.rho)
    nx, ny, nz = g.nx, g.ny, g.nz
    solid = _up(f.solid)
    if g.t_press == 2:
        fx, fy, fz = (torch.full(s, g.rho_f1, dtype=torch.float64, device="cuda") for s in
                      ((nz, ny, nx + 1), (nz, ny + 1, nx), (nz + 1, ny, nx)))
    else:
        fx, fy, fz = _interp(g, rho)
    sx, sy = g.dt / (g.dx * g.dx) / fx, g.dt / (g.dy * g.dy) / fy
    uf, vf, wf = u[1:-1, 1:-1, 1:-1].clone(), v[1:-1, 1:-1, 1:-1].clone(), w[1:-1, 1:-1, 1:-1].clone()
    if g.stretched:
        dzf = _up(g.dzv)[1:, None, None]
        sz, dzz = g.dt / (dzf * dzf * fz), _up(g.dzzv)[1:-1, None, None]
    else:
        sz, dzz = g.dt / (g.dz * g.dz) / fz, g.dz
    keep = torch.ones((nz, ny, nx), dtype=torch.float64, device="cuda")
    if solid is not None:
        h = _halo(solid.double(), False, 1.0) > 0
        keep = 1.0 - solid.double()
        cx = h[1:-1, 1:-1, 1:] | h[1:-1, 1:-1, :-1]
        cy = h[1:-1, 1:, 1:-1] | h[1:-1, :-1, 1:-1]
        cz = h[1:, 1:-1, 1:-1] | h[:-1, 1:-1, 1:-1]
        for a, c in ((sx, cx), (sy, cy), (sz, cz), (uf, cx), (vf, cy), (wf, cz)):
            a[c] = 0.0
    d = sx[:, :, 1:] + sx[:, :, :-1] + sy[:, 1:] + sy[:, :-1] + sz[1:] + sz[:-1]
    d = torch.where(keep > 0, d, torch.ones_like(d))
    q = (uf[:, :, :-1] - uf[:, :, 1:]) / g.dx + (vf[:, :-1] - vf[:, 1:]) / g.dy + (wf[:-1] - wf[1:]) / dzz
    px, lid = g.ccx0 == 0, g.top_bc == 1
    ix, iy, iz = sx[:, :, 1:-1], sy[:, 1:-1], sz[1:-1]

    def apply(p):
        out = torch.zeros_like(p)
        t = ix * (p[:, :, 1:] - p[:, :, :-1])
        out[:, :, 1:] += t
        out[:, :, :-1] -= t
        t = iy * (p[:, 1:] - p[:, :-1])
        out[:, 1:] += t
        out[:, :-1] -= t
        t = iz * (p[1:] - p[:-1])
        out[1:] += t
        out[:-1] -= t
        if px:
            t = sx[:, :, 0] * (p[:, :, 0] - p[:, :, -1])
            out[:, :, 0] += t
            out[:, :, -1] -= t
        if lid:
            out[-1] += 2.0 * sz[-1] * p[-1]
        return out

    p = _cg(apply, d, q, keep, not lid)
    if not lid:
        p = (p - (d * p * keep).sum() / (d * keep).sum()) * keep
    return _halo(p, px, -1.0 if lid else 1.0)


def _correct(g, u, v, w, rho, prd1, vertical=True):
    """posdin's velocity correction in place."""
    fx, fy, fz = _interp(g, rho)
    p = prd1
    u[1:-1, 1:-1, 1:-1] -= g.dt / g.dx * (p[1:-1, 1:-1, 1:] - p[1:-1, 1:-1, :-1]) / fx
    v[1:-1, 1:-1, 1:-1] -= g.dt / g.dy * (p[1:-1, 1:, 1:-1] - p[1:-1, :-1, 1:-1]) / fy
    if vertical:
        w[1:-1, 1:-1, 1:-1] -= g.dt / g.dz * (p[1:, 1:-1, 1:-1] - p[:-1, 1:-1, 1:-1]) / fz


def _hydro(g, t):
    """pressh, then posdin's hydrostatic branch."""
    rho, p = t["rho"], t["prd1"]
    c = p[1:-1, 1:-1, 1:-1]
    c[-1] = g.dz * GZ * rho[-1]
    c[-2] = g.dz * GZ * (rho[-2] + rho[-1]) * 0.5 + c[-1]
    for k in range(g.nz - 3, -1, -1):
        c[k] = GZ * g.dz * (rho[k] + 4.0 * rho[k + 1] + rho[k + 2]) / 3.0 + c[k + 2]
    u, v, w = t["u"], t["v"], t["w"]
    _correct(g, u, v, w, rho, p, vertical=False)
    w[1] = 0.0
    for k in range(1, g.nz + 1):
        w[k + 1, 1:-1, 1:-1] = (w[k, 1:-1, 1:-1] - (u[k, 1:-1, 2:-1] - u[k, 1:-1, 1:-2]) * g.dz / g.dx
                                - (v[k, 2:-1, 1:-1] - v[k, 1:-2, 1:-1]) * g.dz / g.dy)
    for a, h in zip((u, v, w), _interp(g, t["hs"])):
        a[1:-1, 1:-1, 1:-1][h < 1e-4] = 0.0
    return dict((n, t[n]) for n in ("prd1", "u", "v", "w"))


def _weno(ls, h):
    """Along the last axis: of the two one-sided WENO5 derivatives the one of
    larger magnitude; line ends extrapolated with zero derivative."""
    p = [ls[..., m] for m in range(ls.shape[-1])]
    for _ in range(3):
        p.insert(0, (18.0 * p[0] - 9.0 * p[1] + 2.0 * p[2]) / 11.0)
        p.append((18.0 * p[-1] - 9.0 * p[-2] + 2.0 * p[-3]) / 11.0)
    ph = torch.stack(p, -1)
    n = ls.shape[-1]
    dd = (ph[..., 1:] - ph[..., :-1]) / h          # dd[m]: between cells m-3 and m-2 (0-based)

    def one(a, b, c, d, e):
        s0 = 13.0 / 12.0 * (a - 2 * b + c) ** 2 + 0.25 * (a - 4 * b + 3 * c) ** 2
        s1 = 13.0 / 12.0 * (b - 2 * c + d) ** 2 + 0.25 * (b - d) ** 2
        s2 = 13.0 / 12.0 * (c - 2 * d + e) ** 2 + 0.25 * (3 * c - 4 * d + e) ** 2
        w0, w1, w2 = 0.1 / (1e-8 + s0) ** 2, 0.6 / (1e-8 + s1) ** 2, 0.3 / (1e-8 + s2) ** 2
        return (w0 * (2 * a - 7 * b + 11 * c) + w1 * (-b + 5 * c + 2 * d) + w2 * (2 * c + 5 * d - e)) / (
            6.0 * (w0 + w1 + w2))

    # the five differences from the far end of the biased stencil on
    plus = one(*(dd[..., 5 - m:5 - m + n] for m in range(5)))
    minus = one(*(dd[..., m:m + n] for m in range(5)))
    return torch.where(plus.abs() > minus.abs(), plus, minus)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("batch", "it"):
        return None
    c = _make(case, seed)
    g, f = c.grid, c.fields
    if kind == "solve":
        return dict(prd1=_pressure(g, f), status=None)
    if kind == "ipa":
        g.t_press, g.rho_f1 = 2, 1000.0
        p1, p0 = (_rough_pressure((g.nz + 2, g.ny + 2, g.nx + 2), seed + k) for k in (7, 0))
        p0 = p1 + p0
        a = p1 + p0
        fx, fy, fz = _interp(g, _up(f.rho))
        return dict(prd0=p0, px=-(a[1:-1, 1:-1, 1:] - a[1:-1, 1:-1, :-1]) / g.dx / fx,
                    py=-(a[1:-1, 1:, 1:-1] - a[1:-1, :-1, 1:-1]) / g.dy / fy,
                    pz=-(a[1:, 1:-1, 1:-1] - a[:-1, 1:-1, 1:-1]) / g.dz / fz, prd1=_pressure(g, f), status=None)
    if kind in ("hydro", "levelset"):
        s = prepare(case, seed)
        if kind == "hydro":
            return _hydro(g, s["df"].t)
        ls, eps = s["ls"], s["eps"]
        hs = torch.where(ls < -eps, 0.0, torch.where(
            ls > eps, 1.0, 0.5 * (1.0 + ls / eps + torch.sin(PI * ls / eps) / PI)))
        cs = torch.where(ls.abs() <= eps, 0.5 * (1.0 + torch.cos(PI * ls / eps)) / eps, 0.0)
        return dict(hs=hs, rho=g.rho_f1 * (1.0 - hs) + 1000.0 * hs, mu=1.8e-5 * (1.0 - hs) + 1e-3 * hs,
                    hsx=cs * _weno(ls, g.dx), hsy=cs * _weno(ls.transpose(1, 2), g.dy).transpose(1, 2),
                    hsz=cs * _weno(ls.transpose(0, 2), g.dz).transpose(0, 2))
    u, v, w, rho = _up(f.u), _up(f.v), _up(f.w), _up(f.rho)
    if kind == "posdin":
        _correct(g, u, v, w, rho, _rough_pressure((g.nz + 2, g.ny + 2, g.nx + 2), seed))
        return dict(u=u, v=v, w=w)
    p = _pressure(g, f)
    _correct(g, u, v, w, rho, p)
    fort = lambda t: np.asfortranarray(t.cpu().numpy().T)
    return dict(prd=fort(p), u=fort(u), v=fort(v), w=fort(w), status=None)
