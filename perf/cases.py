"""Performance cases of the MI355X fractional-step solver.

Each case is a piece of work that a program using this framework has it do,
through the public entry points of ``amressif_amd.api`` and
``amressif_amd.adjoint``: load a state, advance it, read it back; take the
gradient of a rollout; advance a two-level run; or drive one predictor and
projection through the module functions, as a code does that keeps its own
time loop.  ``exact`` restates the same work in plain FP64 torch: the converged
predictor, a Poisson solve by the operator's eigenvectors, and autograd for the
gradients.

Kinds
  cavity    2D lid-driven cavity (walls), FP64 or mixed precision
  channel2  2D, periodic in x, a moving and a resting wall in y
  cavity3   3D lid-driven cavity
  channel3  3D, periodic in x and z, a moving and a resting wall in y
  adjoint   checkpointed rollout of the 2D cavity, forward and backward
  twolevel  coarse cavity + ratio-2 patch over its top quarter, mixed
  modules   one RK4 pseudo-iteration and one projection by module functions
"""
from __future__ import annotations

import math

import numpy as np
import torch

from amressif_amd import adjoint, api
from amressif_amd import workloads as W

F64 = torch.float64


def _case(name, kind, n, steps, ren, precision="fp64", solver="mg"):
    return dict(name=name, kind=kind, n=n, steps=steps, ren=ren, precision=precision, solver=solver)


def listed():
    return [
        # the smallest run in use: the 128^2, Re = 100 validation cavity, where launches and latency count
        _case("cavity_fp64_128", "cavity", 128, 10, 100.0),
        # the FP64 production run of the 1024^2, Re = 1000 workload
        _case("cavity_fp64_1024", "cavity", 1024, 3, 1000.0),
        # the FP64 side of the 2048^2 workload
        _case("cavity_fp64_2048", "cavity", 2048, 2, 5000.0),
        # the headline workload: 2048^2, Re = 5000, mixed precision
        _case("cavity_mixed_2048", "cavity", 2048, 8, 5000.0, "mixed"),
        # a user's round number that is no power of two: partial tiles, an odd coarsest level of 125^2
        _case("cavity_mixed_1000", "cavity", 1000, 8, 1000.0, "mixed"),
        # a periodic channel: the 2D side of the general path
        _case("channel2_fp64_384", "channel2", 384, 3, 400.0),
        # a small 3D run, as a user sets one up before the large one
        _case("cavity3_fp64_64", "cavity3", 64, 3, 200.0),
        # 3D with periodic directions at a size that is no multiple of the tiles
        _case("channel3_fp64_144", "channel3", 144, 2, 400.0),
        # the 3D cavity of the benchmark, the largest call
        _case("cavity3_fp64_256", "cavity3", 256, 1, 1000.0),
        # control and data assimilation: forward and backward of a 512^2 rollout with checkpoints
        _case("adjoint_fp64_512", "adjoint", 512, 12, 1000.0),
        # the two-level workload: 512^2 and a 1024 x 256 patch, Re = 2000
        _case("twolevel_mixed_512", "twolevel", 512, 8, 2000.0, "mixed"),
        # a code with its own time loop: the module functions, one call each
        _case("modules_fp64_640", "modules", 640, 1, 1000.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cavity", "cavity", "cavity", "channel2", "cavity3", "channel3", "adjoint", "twolevel", "modules"])
    ren = float(rng.choice([100, 200, 400, 1000, 2000, 5000]))
    precision = solver = None
    if kind == "cavity":
        # mostly multiples of 8, one in four any even size
        n = 2 * _log_int(rng, 20, 1000) if rng.random() < 0.25 else 8 * _log_int(rng, 5, 256)
        steps = rng.randint(2, 8)
        precision = rng.choice(["fp64", "mixed"])
        solver = "gmres" if rng.random() < 0.15 else "mg"
    elif kind == "channel2":
        n, steps = _log_int(rng, 3, 62) * 16, rng.randint(2, 4)
    elif kind in ("cavity3", "channel3"):
        # the general path's hierarchy wants m 2^k cells per side with m^3 <= 1024
        n = rng.choice([24, 28, 36, 40, 48, 56, 64, 72, 80, 96, 112, 128, 144, 160, 192, 224])
        steps = rng.randint(1, 3) if n <= 144 else 1
    elif kind == "adjoint":
        n, steps = 8 * _log_int(rng, 8, 64), rng.randint(4, 12)
    elif kind == "twolevel":
        n, steps, precision = 16 * _log_int(rng, 6, 32), rng.randint(4, 8), rng.choice(["fp64", "mixed"])
    else:
        n, steps = 8 * _log_int(rng, 5, 160), 1
    return dict(kind=kind, n=n, steps=steps, ren=ren, precision=precision or "fp64", solver=solver or "mg")


# ------------------------------------------------------------------ geometry
def _dim(case):
    return 3 if case["kind"] in ("cavity3", "channel3") else 2


def _periodic(case):
    return {"channel2": (True, False), "channel3": (True, False, True)}.get(case["kind"], (False,) * _dim(case))


def _inputs(case):
    n, dim, per = case["n"], _dim(case), _periodic(case)
    lo = [111 if p else 135 for p in per] + [135] * (3 - dim)
    hi = list(lo)
    hi[1] = 165  # the lid
    return api.cavity_inputs(n, case["ren"], api.AMRESSIF_MIXED if case["precision"] == "mixed" else api.AMRESSIF_FP64,
                             phy_bc_lo=lo, phy_bc_hi=hi, spacedim=dim,
                             poisson_solver=1 if case["solver"] == "gmres" else 0)


def _rng(seed):
    return np.random.Generator(np.random.PCG64(int(seed) & 0x7FFFFFFFFFFFFFFF))


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=F64, device="cuda")


def _profile(g, x, per, kmax):
    """kmax smooth random functions of the node coordinates x: vanishing twice at walls, or periodic"""
    k = np.arange(1, kmax + 1)
    if per:
        return np.sin(2 * np.pi * np.outer(k, x) + g.uniform(0, 2 * np.pi, (kmax, 1)))
    return np.sin(np.pi * np.outer(k, x)) * np.sin(np.pi * x) ** 2


def _faces(case, seed):
    """Discretely divergence-free faces: the curl of smooth random potentials on the edges, no flow
    through the walls, of order 1."""
    n, dim, per = case["n"], _dim(case), _periodic(case)
    g, h, kmax = _rng(seed), 1.0 / n, 6
    node = np.arange(n + 1) * h
    cell = (np.arange(n) + 0.5) * h
    ext = lambda d: tuple(n + (a == d) for a in reversed(range(dim)))  # noqa: E731
    out = [torch.zeros(ext(d), dtype=F64, device="cuda") for d in range(dim)]
    for c in ((2,) if dim == 2 else (0, 1, 2)):
        a, b = (c + 1) % 3, (c + 2) % 3
        fa, fb = _profile(g, node, per[a], kmax), _profile(g, node, per[b], kmax)
        if not per[a]:
            fa[:, [0, -1]] = 0.0
        if not per[b]:
            fb[:, [0, -1]] = 0.0
        # shape (b, a): potential along c at the nodes of the (a, b) plane
        psi = _t(fb.T) @ _t(g.normal(0.0, 0.1, (kmax, kmax))) @ _t(fa)
        if per[a]:
            psi[:, -1] = psi[:, 0]
        if per[b]:
            psi[-1, :] = psi[0, :]
        ua, ub = (psi[1:, :] - psi[:-1, :]) / h, -(psi[:, 1:] - psi[:, :-1]) / h  # on the a- and the b-faces
        if dim == 2:
            out[a] += ua
            out[b] += ub
            continue
        mod = _t(0.5 + 0.5 * np.cos(2 * np.pi * (cell + g.uniform())))
        for d, part in ((a, ua), (b, ub)):  # axes (b, a), then c, put into (z, y, x) order
            full = part[..., None] * mod
            axes = [b, a, c]
            out[d] += full.permute(*[axes.index(k) for k in (2, 1, 0)])
    return [o.contiguous() for o in out]


def _lid(n, seed):
    """a per-column lid profile around 1, smoothed"""
    return _t(W.lid_profile(n, seed=int(seed)))


# ------------------------------------------------------------------ prepare / run
def prepare(case, seed):
    kind, n, dim = case["kind"], case["n"], _dim(case)
    s = {"case": case}
    if kind == "twolevel":
        s["amr"] = api.TwoLevel(_inputs(case), 3 * n // 4, W.seeded_two_level(n, 3 * n // 4, seed=int(seed)))
        return s
    f = _faces(case, seed)
    if kind == "adjoint":
        s["rollout"] = adjoint.CheckpointedRollout(_inputs(case), case["steps"], every=max(1, case["steps"] // 3))
        s["lid"], s["u0"], s["v0"] = _lid(n, seed + 1), f[0], f[1]
        # the sensitivity of a cost to the final velocity: a smooth field on the faces
        s["gu"], s["gv"] = _faces(case, seed + 2)
        return s
    s["ctx"] = api.Context(_inputs(case))
    s["faces"] = f
    if kind == "modules":
        g = _rng(seed + 3)
        # the step before: the same field a little earlier; a smooth pressure with its Neumann ghosts
        s["prev"] = [0.999 * a for a in f]
        s["prevprev"] = [0.9975 * a for a in f]
        x = (np.arange(n) + 0.5) / n
        c = np.cos(np.pi * np.outer(np.arange(5), x))
        p = c.T @ g.normal(0.0, 0.2, (5, 5)) @ c
        s["userCtx"] = torch.zeros((2, n + 2, n + 2), dtype=F64, device="cuda")
        s["userCtx"][0] = _t(np.pad(p - p.mean(), 1, mode="edge"))
        s["star"] = [torch.empty_like(a) for a in f]
        s["work"] = torch.empty_like(s["userCtx"])
        return s
    s["prev"] = [a.clone() for a in f]
    s["userCtx"] = torch.zeros((2,) + (n + 2,) * dim, dtype=F64, device="cuda")
    s["out"] = [torch.zeros_like(a) for a in f]
    s["outprev"] = [torch.zeros_like(a) for a in f]
    s["outctx"] = torch.zeros_like(s["userCtx"])
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "twolevel":
        s["amr"].advance(case["steps"])
        return s["amr"].fetch()
    if kind == "adjoint":
        r = s["rollout"]
        u, v = r.forward(s["lid"], s["u0"], s["v0"])
        glid, gu0, gv0 = r.backward(s["gu"], s["gv"])
        return {"u": u, "v": v, "glid": glid, "gu0": gu0, "gv0": gv0}
    c = s["ctx"]
    if kind == "modules":
        (u, v), (up, vp), (upp, vpp), (us, vs), w = s["faces"], s["prev"], s["prevprev"], s["star"], s["work"]
        w.copy_(s["userCtx"])
        us.copy_(u)
        vs.copy_(v)
        for sub in range(4):
            c.runge_kutta4_pseudo_time_stepping(sub, us, vs, u, v, up, vp, upp, vpp, w)
        norm = c.Error_Computation(u, v, us, vs)
        rhs, div, total = c.poisson_righthand_side_calc(us, vs)
        sol, _, _ = c.poisson_advance(rhs)
        w[1].copy_(sol)
        un, vn, _ = c.update_solution(us, vs, w)
        cart = c.cont2cart(un, vn)
        return {"us": us, "vs": vs, "norm": norm, "rhs": rhs, "div": div, "u": un, "v": vn, "userCtx": w, "velCart": cart}
    c.load_faces(s["faces"], s["prev"], s["userCtx"])
    c.advance(case["steps"])
    c.store_faces(s["out"], s["outprev"], s["outctx"])
    return {"faces": s["out"], "prev": s["outprev"], "ctx": s["outctx"]}


# ------------------------------------------------------------------ work and tolerance
def work(case):
    """A step reads u^n, u^{n-1} and p, and writes u^{n+1}, p and phi, once each; it evaluates the momentum
    residual at least once (about 90 operations per cell, component and direction) and relaxes the
    Poisson problem at least once (about 30 per cell)."""
    n, dim, steps = case["n"], _dim(case), case["steps"]
    cells = n ** dim * (1.5 if case["kind"] == "twolevel" else 1.0) + (n * n / 4 if case["kind"] == "twolevel" else 0)
    per_step = 8.0 * cells * (3 * dim + 3)
    flops = cells * (90.0 * dim * dim + 30.0)
    if case["kind"] == "adjoint":
        # forward, the same again from the checkpoints, and the adjoint sweep of the same state
        return {"bytes": 3.0 * steps * per_step, "flops": 3.0 * steps * flops}
    return {"bytes": steps * per_step, "flops": steps * flops}


def tolerance(case):
    """Iterative results: the predictor stops at an update of 1e-10 and the Poisson solve at a residual of
    1e-10 relative.  Two correct runs differ by what their last iterations leave.  The velocities agree to
    about 1e-9 and the pressure to 1e-7 (the Poisson residual times its operator's condition); where the
    predictor is the FP64 dual-time loop the pressure also takes (1.5/dt) times the predictor's rest, which
    grows as n^2: 6.9e-5 was seen at 2048^2 and 1.9e-6 at 256^3 against exact().  About four times these."""
    n, kind = case["n"], case["kind"]
    if case["precision"] == "mixed" or kind in ("modules", "adjoint"):
        return {"rel": 4e-7}
    return {"rel": 4e-7 + (8e-6 if _dim(case) == 3 else 4.4e-6) * (n / 256.0) ** 2}


# ------------------------------------------------------------------ FP64 restatement
class _Plain:
    """The step in plain torch: faces f[d] with axis dim-1-d along d."""

    def __init__(self, case, lid=None):
        self.n, self.dim, self.per = case["n"], _dim(case), _periodic(case)
        self.h, self.dt = 1.0 / self.n, api.dt_of(_inputs(case))
        self.c15, self.iren = 1.5 / self.dt, 1.0 / case["ren"]
        self.lid = lid if lid is not None else 1.0
        self.basis = [self._basis(p) for p in self.per]

    def _basis(self, per):
        """orthonormal eigenvectors (columns) and eigenvalues of the 1D second difference"""
        n = self.n
        i = torch.arange(n, dtype=F64, device="cuda")
        k = torch.arange(n, dtype=F64, device="cuda")
        if per:
            m = torch.floor((k + 1) / 2)
            arg = 2 * math.pi * torch.remainder(i[:, None] * m[None, :], n) / n
            q = torch.where((k % 2 == 1)[None, :], torch.cos(arg), torch.sin(arg))
            q[:, 0] = 1.0
            lam = -(2 - 2 * torch.cos(2 * math.pi * m / n))
        else:
            q = torch.cos(math.pi * torch.remainder((i[:, None] + 0.5) * k[None, :], 2 * n) / n)
            lam = -(2 - 2 * torch.cos(math.pi * k / n))
        return q / q.norm(dim=0, keepdim=True), lam / self.h ** 2

    def ax(self, d):
        return self.dim - 1 - d

    def cut(self, t, d, lo, hi):
        return t.narrow(self.ax(d), lo, t.shape[self.ax(d)] - lo - hi)

    def pad(self, x, c, d):
        """component c with two ghosts along d: periodic images, or the wall rules (the lid on the upper y side)"""
        a, n = self.ax(d), self.n
        if self.per[d]:
            return torch.cat([x.narrow(a, n - 2, 2), x, x.narrow(a, 0, 2)], a)
        lo, hi = -x.narrow(a, 0, 2).flip(a), -x.narrow(a, n - 2, 2).flip(a)
        if d == 1 and c == 0:
            hi = hi + 2.0 * self.lid
        return torch.cat([lo, x, hi], a)

    def rhs(self, f):
        """the face average of -div(QUICK) + viscous; 0 on wall faces"""
        n, out = self.n, []
        for c in range(self.dim):
            x = 0.5 * (self.cut(f[c], c, 0, 1) + self.cut(f[c], c, 1, 0))
            t = torch.zeros_like(x)
            for d in range(self.dim):
                g = self.pad(x, c, d)
                a2, a1, b0, b1 = (g.narrow(self.ax(d), k, n + 1) for k in range(4))
                con = 0.5 * f[d]
                ud, up = con + con.abs(), con - con.abs()
                q = up * (0.125 * (-b1 - 2 * b0 + 3 * a1) + b0) + ud * (0.125 * (-a2 - 2 * a1 + 3 * b0) + a1)
                t = t - (self.cut(q, d, 1, 0) - self.cut(q, d, 0, 1)) / self.h
                t = t + (self.cut(g, d, 3, 1) - 2 * x + self.cut(g, d, 1, 3)) * (self.iren / self.h ** 2)
            a = self.ax(c)
            mid = 0.5 * (self.cut(t, c, 0, 1) + self.cut(t, c, 1, 0))
            end = 0.5 * (t.narrow(a, n - 1, 1) + t.narrow(a, 0, 1)) if self.per[c] else torch.zeros_like(t.narrow(a, 0, 1))
            out.append(torch.cat([end, mid, end], a))
        return out

    def grad(self, p):
        out = []
        for d in range(self.dim):
            a = self.ax(d)
            mid = (self.cut(p, d, 1, 0) - self.cut(p, d, 0, 1)) / self.h
            end = (p.narrow(a, 0, 1) - p.narrow(a, self.n - 1, 1)) / self.h if self.per[d] else torch.zeros_like(p.narrow(a, 0, 1))
            out.append(torch.cat([end, mid, end], a))
        return out

    def div(self, f):
        return sum((self.cut(f[d], d, 1, 0) - self.cut(f[d], d, 0, 1)) / self.h for d in range(self.dim))

    def solve(self, b):
        """mean-zero solution of the Neumann / periodic Poisson problem"""
        x, lam = b, 0.0
        for d in range(self.dim):
            q, l1 = self.basis[d]
            x = torch.movedim(torch.movedim(x, self.ax(d), -1) @ q, -1, self.ax(d))
            shape = [1] * self.dim
            shape[self.ax(d)] = self.n
            lam = lam + l1.reshape(shape)
        zero = lam.abs() < 1e-9 / self.h ** 2 / self.n ** 2
        x = torch.where(zero, torch.zeros_like(x), x / torch.where(zero, torch.ones_like(lam), lam))
        for d in range(self.dim):
            x = torch.movedim(torch.movedim(x, self.ax(d), -1) @ self.basis[d][0].T, -1, self.ax(d))
        return x - x.mean()

    def step(self, f, prev, p, iters):
        gp = self.grad(p)
        c = [self.c15 * u + (0.5 / self.dt) * (u - um) - g for u, um, g in zip(f, prev, gp)]
        s = f
        for _ in range(iters):  # contracts by about dt |R'| / 1.5 per sweep
            s = [(r + k) / self.c15 for r, k in zip(self.rhs(s), c)]
        phi = self.solve(self.c15 * self.div(s))
        new = [u - g * (self.dt / 1.5) for u, g in zip(s, self.grad(phi))]
        return new, f, p + phi, phi

    def ghosted(self, p):
        for d in range(self.dim):
            a, n = self.ax(d), self.n
            lo, hi = (n - 1, 0) if self.per[d] else (0, n - 1)
            p = torch.cat([p.narrow(a, lo, 1), p, p.narrow(a, hi, 1)], a)
        return p


def exact(case, seed):
    kind, n, dim = case["kind"], case["n"], _dim(case)
    if kind == "twolevel":
        return None  # the composite step has no plain restatement
    f = _faces(case, seed)
    if kind == "adjoint":
        lid = _lid(n, seed + 1).requires_grad_()
        f = [a.requires_grad_() for a in f]
        m = _Plain(case, lid)
        # the wall-normal faces are fixed: no sensitivity to them
        u = [torch.cat([m.cut(a, d, 0, n).detach(), m.cut(a, d, 1, 1), m.cut(a, d, n, 0).detach()], m.ax(d))
             for d, a in enumerate(f)]
        prev, p = u, torch.zeros((n,) * dim, dtype=F64, device="cuda")
        for _ in range(case["steps"]):
            u, prev, p, _ = m.step(u, prev, p, 8)
        g = torch.autograd.grad(u, [lid] + f, _faces(case, seed + 2))
        return {"u": u[0].detach(), "v": u[1].detach(), "glid": g[0], "gu0": g[1], "gv0": g[2]}
    m = _Plain(case)
    if kind == "modules":
        s = prepare(case, seed)
        gp = m.grad(s["userCtx"][0, 1:-1, 1:-1])
        star = f
        for r in (0.25, 1.0 / 3.0, 0.5, 1.0):
            star = [u + r * 0.4 * m.dt * (q - g - m.c15 * (w - a) + (0.5 / m.dt) * (a - b)) for u, q, g, w, a, b in
                    zip(f, m.rhs(star), gp, star, s["prev"], s["prevprev"])]
        e = []
        for d in range(2):
            sq = (star[d] - f[d]).square()
            ends = sq.narrow(m.ax(d), 0, 1).sum() + sq.narrow(m.ax(d), n, 1).sum()
            e.append(math.sqrt(float(sq.sum() - 0.5 * ends)) / n)
        D = m.div(star)
        phi = m.solve(m.c15 * D)
        new = [u - g * (m.dt / 1.5) for u, g in zip(star, m.grad(phi))]
        cells = [0.5 * (m.cut(new[c], c, 0, 1) + m.cut(new[c], c, 1, 0)) for c in range(2)]
        cart = torch.stack([m.pad(m.pad(x, c, 0), c, 1) for c, x in enumerate(cells)])
        rhs, sol = (torch.zeros((n + 2, n + 2), dtype=F64, device="cuda") for _ in range(2))
        rhs[1:-1, 1:-1], sol[1:-1, 1:-1] = m.c15 * D, phi  # their ghosts stay as the caller made them
        return {"us": star[0], "vs": star[1], "norm": max(e), "rhs": rhs, "div": float(D.abs().max()), "u": new[0],
                "v": new[1], "userCtx": torch.stack([m.ghosted(s["userCtx"][0, 1:-1, 1:-1] + phi), sol]), "velCart": cart}
    u, prev, p, phi = f, f, torch.zeros((n,) * dim, dtype=F64, device="cuda"), None
    for _ in range(case["steps"]):
        u, prev, p, phi = m.step(u, prev, p, 12)
    return {"faces": u, "prev": prev, "ctx": torch.stack([m.ghosted(p), m.ghosted(phi)])}
