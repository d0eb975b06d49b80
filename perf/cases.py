"""Performance cases of the solvers: what a user of this framework has them do, through the public entry points.

A case is a plain dict. `path` says which entry points a pass goes through:
  forward   `Solver.step` over one output interval, then the products a run writes: station records, the PGV
            map and the surface displacement (`products` = "maps"), with velocity slices on three planes too
            ("slices"), or those and the whole wavefield ("field");
  record    `Solver.forward_record` and `Solver.adjoint` on a solver that is kept, as the iterations of an
            inversion for one medium's sources do: seismograms and gradients;
  gradient  `seismograms(...)` of the autograd wrapper and its backward pass: one misfit gradient of a waveform
            inversion, where every new medium makes a new solver.
`scheme` is "cgfdm" or "aweno", `precision` 4 (FP32 wavefield) or 8 (FP64), `coef` the storage of the
coefficients (0 native, 1 fp16, 2 bf16). `grid` is "flat", "hills" (terrain-following, regular in x and y) or
"skewed" (terrain-following and curved in x and y too). The solver is advanced from a smooth random velocity
field, so that every cell, layer and boundary carries signal from the first step.

`exact` evaluates the same schemes in 64 bits with plain torch; gradients come from its automatic
differentiation.
"""
import math
import os
import sys

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cgfdm3d-eqr-sc_amd"))
from cgfdm_amd import autograd, model, solver  # noqa: E402

H = 3  # ghost layers on every side
DH = 100.0


def _case(name, path, scheme, nx, ny, nz, steps, *, npml=0, free_surface=True, precision=4, coef=0, grid="hills",
          stations=25, sources=1, nt=256, products="maps", checkpoint_every=0):
    return {"name": name, "path": path, "scheme": scheme, "nx": nx, "ny": ny, "nz": nz, "steps": steps, "npml": npml,
            "free_surface": free_surface, "precision": precision, "coef": coef, "grid": grid, "stations": stations,
            "sources": sources, "nt": nt, "products": products, "checkpoint_every": checkpoint_every}


def listed():
    return [
        # the smallest runs: quick checks and parameter studies, bounded by launches
        _case("cgfdm_tiny", "forward", "cgfdm", 24, 20, 16, 12, npml=4, stations=4, nt=2048),
        _case("aweno_tiny", "forward", "aweno", 48, 44, 20, 12, stations=4, nt=2048),
        # the plain half-space: flat grid, homogeneous layers, 25 receivers
        _case("cgfdm_half_space", "forward", "cgfdm", 128, 128, 64, 50, npml=12, grid="flat", nt=1000),
        # a run without a free surface (absorbing top) on a grid curved in all directions, odd extents
        _case("cgfdm_no_surface", "forward", "cgfdm", 333, 150, 117, 20, npml=10, free_surface=False, grid="skewed",
              stations=400, sources=128),
        # 16-bit coefficient storage on the medium-size terrain grid, finite fault
        _case("cgfdm_fp16", "forward", "cgfdm", 256, 256, 128, 20, npml=20, coef=1, stations=64, sources=128),
        # FP64 runs, the references of the FP32 ones
        _case("cgfdm_fp64", "forward", "cgfdm", 200, 180, 100, 20, npml=12, precision=8, stations=64),
        _case("aweno_fp64", "forward", "aweno", 150, 140, 90, 8, precision=8, stations=64),
        # one output interval of a run that writes snapshots: slices on three planes and the whole wavefield
        _case("cgfdm_snapshot", "forward", "cgfdm", 150, 130, 70, 100, npml=12, products="field"),
        # the largest: the production terrain grid with its 20-layer absorbing frame and 400 stations
        _case("cgfdm_terrain", "forward", "cgfdm", 512, 512, 256, 10, npml=20, stations=400),
        # the sharp-basin scheme on a large terrain grid
        _case("aweno_basin", "forward", "aweno", 320, 300, 200, 10, stations=400),
        # waveform gradients: a kept solver with two checkpoint segments, and one evaluation through autograd
        _case("adjoint", "record", "cgfdm", 256, 256, 128, 16, npml=20, stations=64, sources=128, nt=2048,
              checkpoint_every=8),
        _case("gradient_small", "gradient", "cgfdm", 64, 60, 40, 24, npml=8, stations=16, sources=8,
              checkpoint_every=10),
    ]


def draw(rng):
    """One more case of the same ranges: kinds, extents over their logarithm (odd ones among them), options."""
    kind = rng.choice(["cgfdm", "cgfdm", "cgfdm", "aweno", "aweno", "record", "gradient"])
    most = {"cgfdm": 16e6, "aweno": 8e6, "record": 3e6, "gradient": 4e5}[kind]
    cells = math.exp(rng.uniform(math.log(8e3), math.log(most)))
    # depth is the short axis of most domains
    fx, fy, fz = (math.exp(rng.uniform(-0.35, 0.35)) for _ in range(3))
    fz *= 0.6
    s = (cells / (fx * fy * fz)) ** (1.0 / 3.0)
    nx, ny, nz = max(24, int(s * fx)), max(20, int(s * fy)), max(20, int(s * fz))
    fs = rng.random() < 0.75
    npml = 0 if kind == "aweno" else rng.choice([0, min(20, max(3, min(nx, ny, nz) // 6)), min(12, max(3, min(nx, ny, nz) // 6))])
    prec = rng.choice([4, 4, 4, 8])
    coef = rng.choice([0, 0, 1, 2]) if kind == "cgfdm" and prec == 4 else 0
    steps = rng.randint(6, 20)
    c = _case("", "forward" if kind in ("cgfdm", "aweno") else kind, "aweno" if kind == "aweno" else "cgfdm", nx, ny, nz,
              steps, npml=npml, free_surface=fs, precision=prec, coef=coef,
              grid=rng.choice(["flat", "hills", "hills", "skewed"]), stations=rng.choice([4, 25, 64]),
              sources=rng.choice([1, 8, 128]), nt=rng.choice([512, 1024]), products=rng.choice(["maps", "maps", "maps", "slices"]),
              checkpoint_every=rng.randint(4, steps + 2) if kind in ("record", "gradient") else 0)
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------
def _device():
    return torch.device("cuda:0" if torch.cuda.is_available() else "cpu")


def _smooth(gen, shape, cells, dev):
    """Random field with features of about `cells` cells, unit size."""
    coarse = torch.randn([max(3, n // cells + 2) for n in shape], generator=gen).to(dev)
    return torch.nn.functional.interpolate(coarse[None, None], size=shape, mode="trilinear", align_corners=True)[0, 0]


def _inputs(case, seed):
    """Grid, medium, time step, source table, stations and initial velocity of a case (float32 tensors)."""
    dev = _device()
    gen = torch.Generator().manual_seed(int(seed) * 7919 + 17)
    rnd = np.random.default_rng(int(seed) * 104729 + 5)
    nx, ny, nz, npml = case["nx"], case["ny"], case["nz"], case["npml"]
    NX, NY, NZ = nx + 2 * H, ny + 2 * H, nz + 2 * H
    f64 = dict(dtype=torch.float64, device=dev)
    X = ((torch.arange(NX, **f64) - H) * DH)[None, None, :]
    Y = ((torch.arange(NY, **f64) - H) * DH)[None, :, None]
    K = (torch.arange(NZ, **f64) - H)[:, None, None]
    depth = nz * DH
    terrain = torch.zeros(1, NY, NX, **f64)
    if case["grid"] != "flat":
        for _ in range(8):
            s = rnd.uniform(0.08, 0.3) * min(nx, ny) * DH
            h = rnd.uniform(0.02, 0.06) * min(depth, 4 * s)
            cx, cy = rnd.uniform(0, nx * DH), rnd.uniform(0, ny * DH)
            terrain = terrain + h * torch.exp(-0.5 * ((X - cx) ** 2 + (Y - cy) ** 2) / s ** 2)
    coord = torch.empty(3, NZ, NY, NX, dtype=torch.float32, device=dev)
    z = -depth + (terrain + depth) / (nz - 1) * K
    coord[0], coord[1], coord[2] = X.expand(NZ, NY, NX), Y.expand(NZ, NY, NX), z
    if case["grid"] == "skewed":
        a = 0.1 / (2 * math.pi)
        coord[0] += a * ny * DH * torch.sin(2 * math.pi * Y / (ny * DH)) + 0.05 * z
        coord[1] += a * nx * DH * torch.sin(2 * math.pi * X / (nx * DH))
    below = terrain - z
    med = torch.empty_like(coord)
    if case["scheme"] == "aweno":
        # sharp low-velocity basin under the surface
        r = ((X / (nx * DH) - 0.5) / 0.25) ** 2 + ((Y / (ny * DH) - 0.5) / 0.2) ** 2 + (below.clamp(min=0) / (0.3 * depth)) ** 2
        for q, (a, b) in enumerate([(400.0, 3464.0), (1200.0, 6000.0), (1900.0, 2700.0)]):
            med[q] = torch.where(r <= 1, a, b)
    else:
        # four layers with a 5 % random perturbation of the speeds (none on the flat grid)
        vp = torch.full_like(z, 3000.0)
        rho = torch.full_like(z, 2300.0)
        for top, v, d in ((0.08, 4500.0, 2500.0), (0.3, 6000.0, 2700.0), (0.7, 7000.0, 3000.0)):
            vp[below > top * depth] = v
            rho[below > top * depth] = d
        if case["grid"] != "flat":
            vp *= 1 + 0.05 * _smooth(gen, (NZ, NY, NX), 8, dev).clamp(-3, 3).double()
        med[0], med[1], med[2] = vp / 1.73, vp, rho
        del vp, rho
    del below, z
    dt = 0.22 * DH / float(med[1].max())
    # moment-rate table of the source points, merged where points share a cell
    nt_src = 256
    t = np.arange(nt_src) * dt
    cells, rate = [], []
    for _ in range(case["sources"]):
        ijk = [int(H + npml + rnd.integers(0, max(1, n - 2 * npml))) for n in (nx, ny, nz)]
        ijk = [min(v, H + n - 1) for v, n in zip(ijk, (nx, ny, nz))]
        cells.append(ijk[0] + NX * (ijk[1] + NY * ijk[2]))
        # double couple of random orientation times area and a triangular slip rate
        u, v = np.linalg.qr(rnd.standard_normal((3, 2)))[0].T
        m = np.outer(u, v) + np.outer(v, u)
        m = np.array([m[0, 0], m[1, 1], m[2, 2], m[0, 1], m[0, 2], m[1, 2]])
        rise = rnd.uniform(0.2, 0.6) * t[-1]
        t0 = rnd.uniform(-0.3, 0.3) * rise
        slip = np.maximum(0.0, 1.0 - np.abs((t - t0) / (0.5 * rise) - 1.0)) * 2.0 * rnd.uniform(0.5, 2.0) / rise
        rate.append(m[None, :] * 1e4 * slip[:, None])
    # receivers on the surface and, every other one, at depth
    st = [[int(H + rnd.integers(0, n)) for n in (nx, ny, nz)] for _ in range(case["stations"])]
    for q in st[::2]:
        q[2] = H + nz - 1
    # smooth random velocity, zero in the ghost cells (momentum for the conservative scheme)
    scale = 0.1 * (2700.0 if case["scheme"] == "aweno" else 1.0)
    vel = []
    for _ in range(3):
        v = torch.zeros(NZ, NY, NX, dtype=torch.float32, device=dev)
        v[H:-H, H:-H, H:-H] = scale * _smooth(gen, (nz, ny, nx), 7, dev)
        vel.append(v)
    return {"coord": coord, "medium": med, "dt": dt, "cells": np.array(cells, np.int64),
            "rate": np.ascontiguousarray(np.array(rate), np.float32), "stations": np.array(st, np.int32), "vel": vel,
            "obs_seed": int(rnd.integers(1 << 30))}


def _model(case, inp):
    return model.Model(case["nx"], case["ny"], case["nz"], DH, inp["dt"], case["nt"], case["npml"],
                       inp["coord"].cpu().numpy(), inp["medium"].cpu().numpy(), case["free_surface"],
                       src_cells=inp["cells"], src_rate=inp["rate"], src_dt=inp["dt"], stations=inp["stations"])


def _observed(case, inp):
    """Recorded seismograms that the gradients' residuals are taken against."""
    r = np.random.default_rng(inp["obs_seed"])
    n = case["steps"]
    ph, am = r.uniform(0, 2 * math.pi, (case["stations"], 1, 3)), r.uniform(0.02, 0.1, (case["stations"], 1, 3))
    return am * np.sin(ph + 2 * math.pi * np.arange(n)[None, :, None] / n)


def prepare(case, seed):
    inp = _inputs(case, seed)
    m = _model(case, inp)
    state = {"case": case, "model": m}
    if case["path"] == "gradient":
        dev = _device()
        state["medium"] = [inp["medium"][c].clone() for c in range(3)]
        state["rate"] = torch.from_numpy(inp["rate"]).to(dev)
        state["observed"] = torch.from_numpy(_observed(case, inp)).to(dev)
        return state
    scheme = solver.SCHEME_AWENO if case["scheme"] == "aweno" else solver.SCHEME_CGFDM
    s = solver.Solver(m, precision=case["precision"], coef_storage=case["coef"], scheme=scheme)
    for c in range(3):
        s.set_field(c, inp["vel"][c].cpu().numpy())
    state["solver"] = s
    if case["path"] == "record":
        state["observed"] = _observed(case, inp)
    return state


def _planes(case):
    return ((0, H + case["nx"] // 2), (1, H + case["ny"] // 2), (2, H + case["nz"] // 2))


def _real(a, case):
    """Fields of an FP32 run are held in 32 bits (the getters widen them)."""
    return a if case["precision"] == 8 else torch.from_numpy(a).to(torch.float32)


def run(state):
    case = state["case"]
    if case["path"] == "gradient":
        vs, vp, rho, rate = (t.detach().requires_grad_(True) for t in (*state["medium"], state["rate"]))
        rec = autograd.seismograms(vs, vp, rho, rate, state["model"], case["steps"], precision=case["precision"],
                                   checkpoint_every=case["checkpoint_every"])
        (0.5 * (rec - state["observed"]).square().sum()).backward()
        return {"seismograms": rec.detach().to(torch.float32), "vs": vs.grad, "vp": vp.grad, "rho": rho.grad,
                "rate": rate.grad}
    s = state["solver"]
    if case["path"] == "record":
        rec = s.forward_record(case["steps"], case["checkpoint_every"])
        g = s.adjoint(rec - state["observed"])
        return {"seismograms": _real(rec, case), **{k: _real(g[k], case) for k in ("gmu", "glam", "gb", "grate")}}
    s.step(case["steps"])
    out = {"stations": s.stations(), "pgv": s.pgv(), "displacement": s.surface_displacement()}
    if case["products"] != "maps":
        for axis, index in _planes(case):
            for c in range(3):
                out["v%d_axis%d" % (c, axis)] = s.slice(c, axis, index)
    if case["products"] == "field":
        out["field"] = [_real(s.field(c), case) for c in range(9)]
    return out


def work(case):
    """Bytes and operations a pass cannot do without: per stage the state read and written once, the
    coefficients read once; the products written once."""
    n = case["nx"] * case["ny"] * case["nz"]
    b = case["precision"]
    cb = 2 if case["coef"] else b
    slabs = 0
    p = case["npml"]
    if p:
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        slabs = 2 * p * ny * nz + 2 * nx * p * nz + (1 if case["free_surface"] else 2) * nx * ny * p
    if case["scheme"] == "aweno":
        # three stages: stage state in and out, step-start state in the last two, 13 coefficients
        per_step = n * (8 * 9 * b + 3 * 13 * cb)
        flops = n * 3 * (27 * 80 + 27 * 20 + 150)
    else:
        # four stages: in and out, and 5 further passes of the RK combination (base in stages 1..3, two of the
        # other stage states in the last); 12 coefficients; the same for the absorbing faces' auxiliaries
        per_step = (n + slabs) * 13 * 9 * b + n * 4 * 12 * cb
        flops = n * 4 * 350 + slabs * 4 * 60
    steps = case["steps"]
    nbytes, nflops = per_step * steps, flops * steps
    if case["path"] != "forward":
        # backward: each stage reads the stage state, the adjoint and the coefficients and writes the adjoint
        # and the three gradients
        nbytes += steps * 4 * (n * (9 * b + 2 * 9 * b + 12 * cb + 2 * 3 * 8) + slabs * 2 * 9 * b)
        nflops += steps * 4 * (n * 900 + slabs * 120)
        nbytes += 3 * 8 * n
    elif case["products"] == "field":
        nbytes += 9 * 8 * n
    nbytes += case["nx"] * case["ny"] * (2 * 4 + 3 * 4) + case["stations"] * steps * 36
    return {"bytes": float(nbytes), "flops": float(nflops)}


# ---------------------------------------------------------------------------
# the same schemes in 64 bits, plain torch
# ---------------------------------------------------------------------------
_AF = (-0.30874, -0.6326, 1.2330, -0.3334, 0.04168)  # MacCormack weights at -1, 0, 1, 2, 3
_CF = (-1.16666667, 1.33333333, -0.16666667)
_RK_A = (0.5, 0.5, 1.0)
_RK_B = (0.16666667, 0.33333333, 0.33333333, 0.16666667)
_PATTERN = ((-1, -1, -1), (1, 1, -1), (1, 1, 1), (-1, -1, 1), (-1, 1, -1), (1, -1, -1), (1, -1, 1), (-1, 1, 1))


def _at(f, axis, off, lo=H, hi=H):
    """The cells [lo, n - hi) of every axis of a padded array, shifted by `off` along axis (0 = x)."""
    sl = []
    for a in (2, 1, 0):
        o = off if a == axis else 0
        n = f.shape[f.dim() - 1 - a]
        sl.append(slice(lo + o, n - hi + o))
    return f[(Ellipsis, *sl)]


def _mac(f, axis, fb):
    return fb / DH * sum(w * _at(f, axis, fb * (m - 1)) for m, w in enumerate(_AF))


def _pad(f):
    return torch.nn.functional.pad(f, (H,) * 6)


def _assemble(D, m, mu, lam, b):
    m1, m2, m3 = m
    div = m1 * D[0] + m2 * D[1] + m3 * D[2]
    return [(m1 * D[3] + m2 * D[6] + m3 * D[7]) * b, (m1 * D[6] + m2 * D[4] + m3 * D[8]) * b,
            (m1 * D[7] + m2 * D[8] + m3 * D[5]) * b, *_stress(D, m, mu, lam, div)]


def _stress(V, m, mu, lam, div=None):
    m1, m2, m3 = m
    div = m1 * V[0] + m2 * V[1] + m3 * V[2] if div is None else div
    return [lam * div + 2 * mu * m1 * V[0], lam * div + 2 * mu * m2 * V[1], lam * div + 2 * mu * m3 * V[2],
            mu * (m2 * V[0] + m1 * V[1]), mu * (m3 * V[0] + m1 * V[2]), mu * (m3 * V[1] + m2 * V[2])]


def _matrix(zt, a, lam, mu, ll, ml):
    """3 x 3 matrices of the traction condition: chi on the diagonal, `ll`/`ml` off it."""
    chi = 2 * lam + mu
    dot = sum(zt[q] * a[q] for q in range(3))
    return [[(chi - mu) * zt[r] * a[c] + mu * dot if r == c else ll * zt[r] * a[c] + ml * zt[c] * a[r] for c in range(3)]
            for r in range(3)]


def _solve3(A, B):
    """A^-1 B for 3 x 3 nests of tensors."""
    cof = [[A[(r + 1) % 3][(c + 1) % 3] * A[(r + 2) % 3][(c + 2) % 3] - A[(r + 1) % 3][(c + 2) % 3] * A[(r + 2) % 3][(c + 1) % 3]
            for c in range(3)] for r in range(3)]
    det = sum(A[0][c] * cof[0][c] for c in range(3))
    return [[sum(cof[q][r] * B[q][c] for q in range(3)) / det for c in range(3)] for r in range(3)]


class _Cgfdm64:
    """MacCormack differences, classical RK4, CFS-PML, traction-image free surface. `med` = (vs, vp, rho) or
    `params` = (mu, lambda, 1/rho), padded."""

    def __init__(self, case, inp, med=None, params=None, rate=None):
        self.case, self.dt = case, inp["dt"]
        self.fs, self.npml = case["free_surface"], case["npml"]
        n = [case["nx"], case["ny"], case["nz"]]
        dev = inp["coord"].device
        c = inp["coord"].double()
        d = [[0.5 * (_mac(c[q], ax, 1) + _mac(c[q], ax, -1)) for q in range(3)] for ax in range(3)]
        cross = lambda u, v: [u[1] * v[2] - u[2] * v[1], u[2] * v[0] - u[0] * v[2], u[0] * v[1] - u[1] * v[0]]  # noqa: E731
        cof = [cross(d[1], d[2]), cross(d[2], d[0]), cross(d[0], d[1])]
        self.J = sum(d[0][q] * cof[0][q] for q in range(3))
        self.m = [[v / self.J for v in row] for row in cof]
        del c, d, cof
        if params is None:
            vs, vp, rho = (t.double() for t in (med if med is not None else inp["medium"]))
            params = rho * vs * vs, rho * (vp * vp - 2 * vs * vs), 1 / rho
        self.mu, self.lam, self.b = (_at(t, 0, 0) for t in params)
        # moment-rate table, scaled by mu / (J DH^3) of the cell
        NX, NY = n[0] + 2 * H, n[1] + 2 * H
        cell = torch.from_numpy(inp["cells"]).to(dev)
        self.src = (cell // (NX * NY), cell // NX % NY, cell % NX)
        inner = tuple(q - H for q in self.src)
        rate = torch.from_numpy(inp["rate"]).to(dev).double() if rate is None else rate
        self.rate = rate * (self.mu[inner] / (self.J[inner] * DH ** 3))[:, None, None]
        st = torch.from_numpy(inp["stations"]).to(dev).long()
        self.st = (st[:, 2], st[:, 1], st[:, 0])
        if self.fs:
            top = lambda t: t[-1]  # noqa: E731
            zt, mu, lam = [top(t) for t in self.m[2]], top(self.mu), top(self.lam)
            DZ = _matrix(zt, zt, lam, mu, lam, mu)
            self.R = [[[-v for v in row] for row in _solve3(DZ, _matrix(zt, [top(t) for t in self.m[ax]], lam, mu, lam, mu))]
                      for ax in range(2)]
        # PML profiles and faces: (axis, slices of the interior)
        L, p = DH * (self.npml - 1), self.npml
        self.prof, self.faces = [], []
        d0 = 0.0
        if p > 1:
            rc = 10.0 ** (-(math.log10(p) - 1.0) / math.log10(2.0) - 3.0)
            d0 = -3.0 * 6000.0 / (2.0 * L) * math.log(rc)
        for ax in range(3):
            q = torch.arange(n[ax], dtype=torch.float64, device=dev)
            lo, hi = (p - 1 - q) * DH, (q - (n[ax] - p)) * DH
            use_hi = not (ax == 2 and self.fs)
            l = torch.where(hi >= 0, hi, lo) if use_hi and p else lo
            inside = (l >= 0) & (p > 0)
            x = (l / L if L > 0 else torch.zeros_like(l)).clamp(min=0)
            beta = torch.where(inside, 1 + 2.0 * x * x, 1.0)
            alpha = torch.where(inside, 3.141592657 * 0.5 * (1 - x), 0.0)
            dd = torch.where(inside, d0 * x * x, 0.0) / beta
            sh = [1, 1, 1]
            sh[2 - ax] = -1
            self.prof.append([t.reshape(sh) for t in (alpha, 1 / beta, dd)])
            for side in range(2 if use_hi else 1):
                if p:
                    sl = [slice(None)] * 3
                    sl[2 - ax] = slice(0, p) if side == 0 else slice(n[ax] - p, n[ax])
                    self.faces.append((ax, tuple(sl)))

    def start(self, inp):
        W = torch.zeros(9, *inp["vel"][0].shape, dtype=torch.float64, device=inp["coord"].device)
        for c in range(3):
            W[c] = inp["vel"][c]
        A = [torch.zeros(9, *self.J[sl].shape, dtype=torch.float64, device=W.device) for _, sl in self.faces]
        return W, A

    def rates(self, W, A, fb):
        """Right-hand sides of the state and of the PML auxiliaries."""
        mu, lam, b = self.mu, self.lam, self.b
        Q, V = [], []
        for ax in range(3):
            D = [_mac(W[v], ax, fb[ax]) for v in range(9)]
            Q.append(torch.stack(_assemble(D, self.m[ax], mu, lam, b)))
            V.append([t[-3:] for t in D[:3]] if self.fs else None)
            del D
        h = sum(self.prof[ax][1] * Q[ax] for ax in range(3))
        extra = {}
        if self.fs:
            h = torch.cat([h[:, :-3], self.surface(W, V, fb, extra)], 1)
        hA = []
        for (ax, sl), a in zip(self.faces, A):
            al, be, d = (t.expand_as(self.J)[sl] for t in self.prof[ax])
            g = d * Q[ax][(slice(None), *sl)] - (al + d) * a
            if self.fs and ax < 2:
                g = torch.cat([g[:, :-1], g[:, -1:] + extra[ax][(slice(None), *sl)]], 1)
            hA.append(g)
        for (ax, sl), a in zip(self.faces, A):
            h[(slice(None), *sl)] -= self.prof[ax][1].expand_as(self.J)[sl] * a
        return h, hA

    def surface(self, W, V, fb, extra):
        """Rows of the top three layers: image of the traction for the velocity, one-sided or traction-free
        vertical derivative for the stress."""
        top = lambda t: t[-3:]  # noqa: E731
        mu, lam, b, J = top(self.mu), top(self.lam), top(self.b), top(self.J)
        layers = slice(W.shape[1] - H - 6, W.shape[1] - H)  # six layers under the surface, itself included
        low = slice(self.J.shape[0] - 6, None)
        hv = 0
        for ax in range(3):
            m = [t[low] * self.J[low] for t in self.m[ax]]
            T = W[:, layers, H:-H, H:-H]
            g = torch.stack([m[0] * T[3] + m[1] * T[6] + m[2] * T[7], m[0] * T[6] + m[1] * T[4] + m[2] * T[8],
                             m[0] * T[7] + m[1] * T[8] + m[2] * T[5]])
            if ax < 2:
                g = torch.nn.functional.pad(g, (H, H, H, H, 0, H))
            else:  # odd image about the surface
                img = -g.flip(1)[:, 1:4]
                g = torch.nn.functional.pad(torch.cat([g[:, :5], torch.zeros_like(g[:, :1]), img], 1), (H, H, H, H))
            hv = hv + _mac(g, ax, fb[ax]) * (self.prof[ax][1] if ax < 2 else 1.0)
        hv = hv * b / J
        bx, by = self.prof[0][1], self.prof[1][1]
        Vx, Vy = [t * bx for t in V[0]], [t * by for t in V[1]]
        kt = W.shape[1] - H - 1
        f, s = W[:3, :, H:-H, H:-H], fb[2]
        Vz = []
        for r in range(3):
            surf = sum(self.R[0][r][c] * Vx[c][-1] + self.R[1][r][c] * Vy[c][-1] for c in range(3))
            one = s / DH * (f[r, kt - 1 + s] - f[r, kt - 1])
            two = s / DH * (_CF[0] * f[r, kt - 2] + _CF[1] * f[r, kt - 2 + s] + _CF[2] * f[r, kt - 2 + 2 * s])
            Vz.append(torch.stack([two, one, surf]))
        m = [[top(t) for t in self.m[ax]] for ax in range(3)]
        hs = sum(torch.stack(_stress(v, m[ax], mu, lam)) for ax, v in enumerate((Vx, Vy, Vz)))
        for ax in range(2):
            d = self.prof[ax][2]
            Z = [sum(self.R[ax][r][c] * (V[ax][c] * d)[-1:] for c in range(3)) for r in range(3)]
            s6 = torch.stack(_stress(Z, [t[-1:] for t in m[2]], mu[-1:], lam[-1:]))
            extra[ax] = torch.cat([torch.zeros_like(s6[:3]), s6])
        return torch.cat([hv, hs])

    def step(self, W, A, it):
        f32 = np.float32
        now = f32(it) * f32(self.dt)
        src = int(now / f32(self.dt))
        if src + 1 < self.rate.shape[1]:
            tw = float((now - f32(src) * f32(self.dt)) / f32(self.dt))
            s = (self.rate[:, src + 1] - self.rate[:, src]) * tw + self.rate[:, src]
            inc = torch.zeros_like(W)
            q = torch.arange(3, 9, device=W.device)[:, None]
            inc = inc.index_put((q, *(t[None, :] for t in self.src)), s.t() * self.dt, accumulate=True)
            W = W - inc
            del inc
        fb = list(_PATTERN[it % 8])
        X, Y, T, S = W, A, W, A
        for stage in range(4):
            h, hA = self.rates(X, Y, fb)
            h = _pad(h) * self.dt
            T = T + _RK_B[stage] * h
            S = [t + _RK_B[stage] * g * self.dt for t, g in zip(S, hA)]
            if stage < 3:
                X = W + _RK_A[stage] * h
                Y = [t + _RK_A[stage] * g * self.dt for t, g in zip(A, hA)]
            fb = [-v for v in fb]
            del h, hA
        return T, S

    def physical(self, W):
        return W

    def velocity(self, W):
        """Surface velocity."""
        return W[:3, -H - 1, H:-H, H:-H]


class _Aweno64:
    """WENO5 alternative-flux differences, TVD-RK3, characteristic free surface, exponential sponge."""

    def __init__(self, case, inp):
        self.case, self.dt, self.fs = case, inp["dt"], case["free_surface"]
        dev = inp["coord"].device
        c = inp["coord"].double()
        NZ, NY, NX = c.shape[1:]
        one = lambda t: torch.nn.functional.pad(t, (1,) * 6)  # noqa: E731
        cov = [[one((_at(c[q], ax, 1, 1, 1) - _at(c[q], ax, -1, 1, 1)) * (0.5 / DH)) for q in range(3)] for ax in range(3)]
        cross = lambda u, v: [u[1] * v[2] - u[2] * v[1], u[2] * v[0] - u[0] * v[2], u[0] * v[1] - u[1] * v[0]]  # noqa: E731
        self.n = [[torch.nn.functional.pad(_at(t, 0, 0, 2, 2), (2,) * 6) for t in cross(cov[(a + 1) % 3], cov[(a + 2) % 3])] for a in range(3)]
        self.J = sum(cov[0][q] * cross(cov[1], cov[2])[q] for q in range(3))
        self.tangents = [[t[-H - 1] for t in cov[0]], [t[-H - 1] for t in cov[1]]]
        vs, vp, rho = inp["medium"].double()
        self.mu, self.lam, self.b = rho * vs * vs, rho * (vp * vp - 2 * vs * vs), 1 / rho
        self.alpha = float(inp["medium"][1].max())
        cell = torch.from_numpy(inp["cells"]).to(dev)
        self.src = (cell // (NX * NY), cell // NX % NY, cell % NX)
        mu, lam = self.mu[self.src][:, None], self.lam[self.src][:, None]
        s = torch.from_numpy(inp["rate"]).to(dev).double() * (self.mu[self.src] / (self.J[self.src] * DH ** 3))[:, None, None]
        den = 2 * mu * mu + 3 * lam * mu
        tr = s[..., 0] + s[..., 1] + s[..., 2]
        e = [(s[..., q] * (lam + mu) - 0.5 * lam * (tr - s[..., q])) / den for q in range(3)]
        self.rate = torch.stack(e + [s[..., q] / mu for q in (5, 4, 3)], -1)  # strain rates per point and time
        st = torch.from_numpy(inp["stations"]).to(dev).long()
        self.st = (st[:, 2], st[:, 1], st[:, 0])
        # sponge: factors of the sides a cell lies in
        L, g = 20, 1.0
        for ax, n in enumerate((case["nx"], case["ny"], case["nz"])):
            q = torch.arange(n, dtype=torch.float64, device=dev)
            lo = torch.where(q <= L, torch.exp(-(0.015 * (L - q)) ** 2), 1.0)
            hi = torch.where(q >= n - L, torch.exp(-(0.015 * (L - (n - q))) ** 2), 1.0)
            sh = [1, 1, 1]
            sh[2 - ax] = -1
            g = g * (lo if ax == 2 and self.fs else lo * hi).reshape(sh)
        self.sponge = g

    def start(self, inp):
        W = torch.zeros(9, *inp["vel"][0].shape, dtype=torch.float64, device=inp["coord"].device)
        for c in range(3):
            W[c] = inp["vel"][c]
        return W, []

    @staticmethod
    def weno(u1, u2, u3, u4, u5):
        k = 3 * 0.3333333333
        b1 = k * (13 / 12 * (u3 - 2 * u4 + u5) ** 2 + 0.25 * (3 * u3 - 4 * u4 + u5) ** 2)
        b2 = k * (13 / 12 * (u2 - 2 * u3 + u4) ** 2 + 0.25 * (u2 - u4) ** 2)
        b3 = k * (13 / 12 * (u1 - 2 * u2 + u3) ** 2 + 0.25 * (u1 - 4 * u2 + 3 * u3) ** 2)
        w1, w2, w3 = 0.3125 / (b1 + 1e-6) ** 2, 0.625 / (b2 + 1e-6) ** 2, 0.0625 / (b3 + 1e-6) ** 2
        p = w1 * (0.375 * u3 + 0.75 * u4 - 0.125 * u5) + w2 * (-0.125 * u2 + 0.75 * u3 + 0.375 * u4) + \
            w3 * (0.375 * u1 - 1.25 * u2 + 1.875 * u3)
        return p / (w1 + w2 + w3)

    @staticmethod
    def flux(u, n, mu, lam, b):
        n1, n2, n3 = n
        lm = lam + 2 * mu
        return torch.stack([
            -(n1 * (lam * (u[4] + u[5]) + lm * u[3]) + mu * (n2 * u[8] + n3 * u[7])),
            -(n2 * (lam * (u[3] + u[5]) + lm * u[4]) + mu * (n1 * u[8] + n3 * u[6])),
            -(n3 * (lam * (u[3] + u[4]) + lm * u[5]) + mu * (n1 * u[7] + n2 * u[6])),
            -n1 * u[0] * b, -n2 * u[1] * b, -n3 * u[2] * b,
            -(n2 * u[2] + n3 * u[1]) * b, -(n1 * u[2] + n3 * u[0]) * b, -(n1 * u[1] + n2 * u[0]) * b])

    def rates(self, W):
        h = 0
        for ax in range(3):
            # faces q + 1/2 of cells q in [2, n - 3) along ax, interior across it
            dim = 3 - ax
            n = W.shape[dim]
            idx = [slice(None)] + [slice(H, s - H) for s in W.shape[1:]]

            def cells(t, off, first, last, idx=idx, dim=dim):
                sl = list(idx)
                sl[dim] = slice(first + off, last + off)
                return t[tuple(sl[4 - t.dim():])]

            w = [cells(W, o, 2, n - H) for o in range(-2, 4)]
            um = torch.stack([self.weno(*(w[q][v] for q in range(5))) for v in range(9)])
            up = torch.stack([self.weno(*(w[q][v] for q in (5, 4, 3, 2, 1))) for v in range(9)])
            del w
            at = lambda t: cells(t, 0, 2, n - H)  # noqa: E731
            F = 0.5 * (self.flux(um + up, [at(t) for t in self.n[ax]], at(self.mu), at(self.lam), at(self.b)) -
                       self.alpha * (up - um))
            del um, up
            # zero flux outside the faces above: pad to faces 0 .. n - 1
            pad = [0] * 6
            pad[2 * ax], pad[2 * ax + 1] = 2, H
            F = torch.nn.functional.pad(F, pad)
            f = lambda o: F.narrow(dim, H + o, n - 2 * H)  # noqa: E731

            def value(o):
                u1, u2, u3, u4, u5 = (f(o + q) for q in range(-2, 3))
                return u3 - (-u1 + 16 * u2 - 30 * u3 + 16 * u4 - u5) / 288 + 7 / 5760 * (u1 - 4 * u2 + 6 * u3 - 4 * u4 + u5)

            du = value(0) - value(-1)
            # top three layers: corrections on the physical fluxes of the neighbouring cells
            z = slice(W.shape[1] - H - 3, W.shape[1] - H)
            tops = []
            for o in range(-3, 4):
                sl = [slice(None), z, slice(H, W.shape[2] - H), slice(H, W.shape[3] - H)]
                sl[dim] = slice(sl[dim].start + o, sl[dim].stop + o)
                c3 = tuple(sl[1:])
                tops.append(self.flux(W[tuple(sl)], [t[c3] for t in self.n[ax]], self.mu[c3], self.lam[c3], self.b[c3]))

            def corr(u):
                return -(-5 * u[0] + 39 * u[1] - 34 * u[2] - 34 * u[3] + 39 * u[4] - 5 * u[5]) / 1152 + \
                    7 / 11520 * (u[0] - 3 * u[1] + 2 * u[2] + 2 * u[3] - 3 * u[4] + u[5])

            dt = (f(0) - f(-1))[:, -3:] + corr(tops[1:]) - corr(tops[:6])
            h = h - torch.cat([du[:, :-3], dt], 1)
            del F, du, dt, tops
        return h / (DH * _at(self.J, 0, 0))

    def step(self, W, A, it):
        f32 = np.float32
        now = f32(it) * f32(self.dt)
        src = int(now / f32(self.dt))
        W = W.clone()
        if src + 1 < self.rate.shape[1]:
            tw = float((now - f32(src) * f32(self.dt)) / f32(self.dt))
            s = (self.rate[:, src + 1] - self.rate[:, src]) * tw + self.rate[:, src]
            for q in range(6):
                W[3 + q].index_put_(self.src, -s[:, q] * self.dt, accumulate=True)
        U = W + _pad(self.rates(W) * self.dt)
        U = 0.75 * W + 0.25 * (U + _pad(self.rates(U) * self.dt))
        U = W / 3 + 2 / 3 * (U + _pad(self.rates(U) * self.dt))
        if self.fs:
            self.characteristic(U)
        U[:, H:-H, H:-H, H:-H] *= self.sponge
        return U, A

    def tension(self, w, mu, lam):
        lm = lam + 2 * mu
        d = [lam * (w[4] + w[5]) + lm * w[3], lam * (w[3] + w[5]) + lm * w[4], lam * (w[3] + w[4]) + lm * w[5]]
        return d + [mu * w[8], mu * w[7], mu * w[6]]  # xx yy zz xy xz yz

    def characteristic(self, W):
        k = W.shape[1] - H - 1
        inner = lambda t: t[H:-H, H:-H]  # noqa: E731
        mu, lam, b = inner(self.mu[k]), inner(self.lam[k]), inner(self.b[k])
        J = inner(self.J[k])
        rows = [[inner(t[k]) / J for t in self.n[2]], [inner(t) for t in self.tangents[0]], [inner(t) for t in self.tangents[1]]]
        B = torch.stack([torch.stack(r) / torch.sqrt(sum(t * t for t in r)) for r in rows])  # rows n, s, t
        C = torch.stack([torch.linalg.cross(B[(r + 1) % 3], B[(r + 2) % 3], dim=0) for r in range(3)])
        det = (B[0] * C[0]).sum(0)
        C = C / det
        w = W[:, k, H:-H, H:-H].clone()
        xx, yy, zz, xy, xz, yz = self.tension(w, mu, lam)
        S = torch.stack([torch.stack([xx, xy, xz]), torch.stack([xy, yy, yz]), torch.stack([xz, yz, zz])])
        mul = lambda M, T: torch.stack([torch.stack([sum(M[r, q] * T[q, c] for q in range(3)) for c in range(3)]) for r in range(3)])  # noqa: E731
        tr = lambda M: M.transpose(0, 1)  # noqa: E731
        S = mul(mul(C, S), tr(C))
        v = torch.stack([sum(C[r, q] * w[q] * b for q in range(3)) for r in range(3)])
        vs, vp, l2m = torch.sqrt(mu * b), torch.sqrt((lam + 2 * mu) * b), lam + 2 * mu
        v = torch.stack([v[0] - S[0, 0] * b / vp, v[1] - S[0, 1] * b / vs, v[2] - S[0, 2] * b / vs])
        zero = torch.zeros_like(mu)
        S = torch.stack([torch.stack([zero, zero, zero]), torch.stack([zero, S[1, 1] - S[0, 0] * lam / l2m, S[1, 2]]),
                         torch.stack([zero, S[2, 1], S[2, 2] - S[0, 0] * lam / l2m])])
        S = mul(mul(tr(B), S), B)
        v = torch.stack([sum(B[q, r] * v[q] for q in range(3)) for r in range(3)])
        tr3 = S[0, 0] + S[1, 1] + S[2, 2]
        e = [(S[r, r] - lam * tr3 / (3 * lam + 2 * mu)) / (2 * mu) for r in range(3)]
        new = torch.stack([*(v / b), *e, S[1, 2] / mu, S[0, 2] / mu, S[0, 1] / mu])
        f = W[:, :, H:-H, H:-H]
        f[:, k] = new
        for g in range(1, H + 1):
            f[:, k + g] = 4 * f[:, k + g - 1] - 6 * f[:, k + g - 2] + 4 * f[:, k + g - 3] - f[:, k + g - 4]

    def physical(self, W):
        return torch.stack([W[0] * self.b, W[1] * self.b, W[2] * self.b, *self.tension(W, self.mu, self.lam)])

    def velocity(self, W):
        return W[:3, -H - 1, H:-H, H:-H] * self.b[-H - 1, H:-H, H:-H]


def _exact_forward(case, inp):
    s = _Aweno64(case, inp) if case["scheme"] == "aweno" else _Cgfdm64(case, inp)
    W, A = s.start(inp)
    dev, n = W.device, (case["ny"], case["nx"])
    rec = torch.zeros(case["stations"], case["nt"], 9, dtype=torch.float64, device=dev)
    pgv = torch.zeros(*n, 2, dtype=torch.float64, device=dev)
    dis = torch.zeros(3, *n, dtype=torch.float64, device=dev)
    for it in range(case["steps"]):
        W, A = s.step(W, A, it)
        at = (slice(None), *s.st)
        if case["scheme"] == "aweno":
            mu, lam, b = s.mu[s.st], s.lam[s.st], s.b[s.st]
            w = W[at]
            rec[:, it] = torch.stack([*(w[:3] * b), *s.tension(w, mu, lam)], -1)
        else:
            rec[:, it] = W[at].t()
        if case["free_surface"]:
            v = s.velocity(W)
            dis += v * s.dt
            h = v[0] ** 2 + v[1] ** 2
            pgv = torch.maximum(pgv, torch.stack([h.sqrt(), (h + v[2] ** 2).sqrt()], -1))
    out = {"stations": rec, "pgv": pgv, "displacement": dis}
    if case["products"] != "maps":
        P = s.physical(W)
        for axis, index in _planes(case):
            for c in range(3):
                out["v%d_axis%d" % (c, axis)] = P[c].select(2 - axis, index)[H:-H, H:-H]
    if case["products"] == "field":
        out["field"] = [W[c] for c in range(9)]
    return out


def _exact_gradient(case, inp):
    dev = inp["coord"].device
    leaf = lambda t: t.double().requires_grad_(True)  # noqa: E731
    rate = leaf(torch.from_numpy(inp["rate"]).to(dev))
    med = inp["medium"].double()
    if case["path"] == "gradient":
        vel = [torch.zeros_like(v) for v in inp["vel"]]
        params = [leaf(t) for t in med]
        s = _Cgfdm64(case, {**inp, "vel": vel}, med=params, rate=rate)
    else:
        vel = inp["vel"]
        params = [leaf(t) for t in (med[2] * med[0] ** 2, med[2] * (med[1] ** 2 - 2 * med[0] ** 2), 1 / med[2])]
        s = _Cgfdm64(case, inp, params=params, rate=rate)
    W, A = s.start({**inp, "vel": vel})
    rec = []
    for it in range(case["steps"]):
        flat = checkpoint(lambda w, *a, it=it: (lambda r: (r[0], *r[1]))(s.step(w, list(a), it)), W, *A, use_reentrant=False)
        W, A = flat[0], list(flat[1:])
        rec.append(W[(slice(0, 3), *s.st)].t())
    rec = torch.stack(rec, 1)
    obs = torch.from_numpy(_observed(case, inp)).to(dev)
    (0.5 * (rec - obs).square().sum()).backward()
    names = ("vs", "vp", "rho") if case["path"] == "gradient" else ("gmu", "glam", "gb")
    g = {k: p.grad for k, p in zip(names, params)}
    return {"seismograms": rec.detach(), **g, "rate" if case["path"] == "gradient" else "grate": rate.grad}


def exact(case, seed):
    inp = _inputs(case, seed)
    return _exact_forward(case, inp) if case["path"] == "forward" else _exact_gradient(case, inp)
