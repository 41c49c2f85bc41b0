"""Batched synthetic Poisson problems: many independent Coulomb-type potential
relaxations on different grids, relaxed together on one GPU.

A problem is the Coulomb potential equation of x2dhf's relaxPots
(relaxPots.F90:62-95, Delta m = 0, even symmetry) for a synthetic axial
density rho: lhs = f3, rhs = rho * g, with the Dirichlet rows mu = nmu-3..nmu
set from the density's multipole moments (coulAsympt, scfUtils.F90:275-296),
from a zero interior.  rho is a sum of K Gaussians centred on the
internuclear axis, exp(-|x - z_k e_z|^2 / (2 sigma_k^2)) with sigma_k in bohr,
normalised to one electron with the orbital-norm quadrature (wgt2 * f4); a
density of N electrons gives N times the potential of the unit one.

The problems are relaxed with x2g_relax_batch (all active problems in one
launch per sweep), FP32 correction sweeps with FP64 residuals by default,
until ||rhs - A u|| / ||rhs|| <= tol for each, or until the residual stops
decreasing; those problems leave the batch.

The FP64 floor.  A solution stored in FP64 cannot have a smaller residual
than the one its own rounding causes: with u* the exact discrete solution and
u = fl(u*), rhs - A u = A (u* - u), of size ||A (u * delta)|| with delta the
relative rounding (uniform in +-eps/2).  floors() measures exactly that on
the device for each solved problem, ||A (u * delta)|| / ||rhs||, and a
problem counts as solved when its residual is at most
max(tol, FLOOR_FACTOR * floor).  On the 256 seeded problems of the batched
benchmark the floor lies between 4e-14 and 3e-11, above 1e-12 for 174 of
them (the 17-point operator's h^-2 weights times |u| ~ the electron count,
against a density confined to a few bohr), so a tolerance of 1e-12 relative
is below what FP64 storage allows for most of them.
"""
import ctypes as C
import time

import numpy as np

from . import gpu, scf

GRIDS = [(91, 121), (169, 241), (337, 601), (505, 901)]
# a problem is solved at max(tol, FLOOR_FACTOR * its FP64 floor)
FLOOR_FACTOR = 4.0


def make_problems(count=256, seed=0, rinf=40.0):
    """Problem parameters: grid, R, Gaussians (z_k, sigma_k, weight_k), electrons."""
    rng = np.random.default_rng(seed)
    out = []
    for k in range(count):
        nni, nmu = GRIDS[rng.integers(len(GRIDS))]
        r = float(rng.uniform(1.0, 6.0))
        ng = int(rng.integers(1, 9))
        gauss = [(float(rng.uniform(-0.6 * r, 0.6 * r)), float(rng.uniform(0.1, 2.0)), float(rng.uniform(0.2, 1.0)))
                 for _ in range(ng)]
        out.append(dict(nni=nni, nmu=nmu, r=r, rinf=rinf, gauss=gauss, electrons=float(rng.uniform(1.0, 20.0))))
    return out


def density(p, vxi, veta):
    """The problem's density on its grid (nni*nmu, nu fastest), unnormalised."""
    r2 = 0.5 * p["r"]
    xi, eta = np.meshgrid(vxi, veta, indexing="ij")          # (nmu, nni)
    z = r2 * xi * eta
    rho2 = (r2 * r2) * np.maximum(xi * xi - 1.0, 0.0) * np.maximum(1.0 - eta * eta, 0.0)
    d = np.zeros_like(z)
    for zk, sk, wk in p["gauss"]:
        d += wk * np.exp(-(rho2 + (z - zk) ** 2) / (2.0 * sk * sk))
    return d.ravel()


class Batch:
    """The device side of a set of problems on one context."""

    def __init__(self, problems, ctx=None, prec=1, omega=None, mpole=4):
        self.lib = gpu.load()
        self.ctx = ctx or gpu.Context(0)
        self.own = ctx is None
        self.problems = problems
        self.prec = prec
        self.grids, self.items, self.keep = [], [], []
        for i, p in enumerate(problems):
            coef, suppl, vxi, veta = scf.grid_build(p["nni"], p["nmu"], 1.0, 1.0, p["r"], p["rinf"])
            g = gpu.Grid(self.ctx, p["nni"], p["nmu"], coef, suppl, vxi, veta)
            self.grids.append(g)
            d = density(p, vxi, veta)
            nrm = float(np.sum(suppl[13] * suppl[8] * d))
            d /= nrm
            lhs, rhs = self.ctx.upload(suppl[7]), self.ctx.upload(d * suppl[9])
            fun = self.ctx.upload(np.zeros(g.n))
            ones = self.ctx.upload(np.ones(g.n))
            dd = self.ctx.upload(d)
            mom = np.zeros(8)
            gpu.check(self.lib.x2g_moments(g.h, dd.ptr, ones.ptr, 0, mpole, mom.ctypes.data))
            gpu.check(self.lib.x2g_pot_tail(g.h, fun.ptr, 0, 0, mpole, mom.ctypes.data))
            w = omega
            if w is None:
                oo, op = C.c_double(), C.c_double()
                scf.load().x2f_omega_defaults(p["nni"], p["nmu"], 1.0, 1.0, C.byref(oo), C.byref(op))
                w = op.value
            self.keep += [lhs, rhs, fun, ones, dd]
            self.items.append(gpu.RelaxItem(fun.ptr, lhs.ptr, rhs.ptr, None, w, 1, 1, prec, i))
        self.gh = (gpu._vp * len(self.grids))(*[g.h.value for g in self.grids])

    def residuals(self, active):
        its = (gpu.RelaxItem * len(active))(*[self.items[i] for i in active])
        out = np.zeros(2 * len(active))
        gpu.check(self.lib.x2g_residual_norms(self.ctx.h, self.gh, its, len(active), out.ctypes.data))
        return np.sqrt(out[0::2] / np.maximum(out[1::2], 1e-300))

    def floors(self, idx=None, seed=0):
        """FP64 rounding floor of each problem's relative residual:
        ||A (u * delta)|| / ||rhs|| for its current solution u and a seeded
        relative perturbation delta uniform in +-eps/2 (one sample), formed
        with the device residual (rhs = 0)."""
        idx = range(len(self.items)) if idx is None else idx
        rng = np.random.default_rng(seed)
        eps = np.finfo(np.float64).eps
        out = []
        scratch = {}
        for i in idx:
            g = self.grids[i]
            if g.n not in scratch:
                scratch[g.n] = (self.ctx.alloc(g.n), self.ctx.upload(np.zeros(g.n)))
            du, zero = scratch[g.n]
            u = self.solution(i)
            du.set(u * rng.uniform(-0.5 * eps, 0.5 * eps, u.size))
            it = self.items[i]
            pert = (gpu.RelaxItem * 1)(gpu.RelaxItem(du.ptr, it.lhs_d, zero.ptr, None, it.omega, it.isym, it.bkind,
                                                     it.prec, it.grid_index))
            base = (gpu.RelaxItem * 1)(it)
            a, b = np.zeros(2), np.zeros(2)
            gpu.check(self.lib.x2g_residual_norms(self.ctx.h, self.gh, pert, 1, a.ctypes.data))
            gpu.check(self.lib.x2g_residual_norms(self.ctx.h, self.gh, base, 1, b.ctypes.data))
            out.append(float(np.sqrt(a[0] / max(b[1], 1e-300))))
        for du, zero in scratch.values():
            du.free()
            zero.free()
        return np.array(out)

    def solve(self, tol=1e-12, sweeps_per_call=10, check_every=5, max_calls=20000, stall_checks=40):
        """Relax until every problem meets tol (or stops improving for
        stall_checks residual checks, or max_calls relaxation calls); returns
        per-problem calls and final relative residuals.  A problem that left
        the batch without reaching tol is solved only if it reached its FP64
        floor (see floors and solved)."""
        n = len(self.items)
        active = list(range(n))
        calls = np.zeros(n, dtype=int)
        res = np.full(n, np.inf)
        best = np.full(n, np.inf)
        stall = np.zeros(n, dtype=int)
        k = 0
        while active and k < max_calls:
            its = (gpu.RelaxItem * len(active))(*[self.items[i] for i in active])
            for _ in range(check_every):
                gpu.check(self.lib.x2g_relax_batch(self.ctx.h, self.gh, its, len(active), 1, sweeps_per_call))
            k += check_every
            r = self.residuals(active)
            for i, v in zip(active, r):
                calls[i] += check_every
                res[i] = v
                if v < 0.9 * best[i]:
                    best[i], stall[i] = v, 0
                else:
                    stall[i] += 1
            active = [i for i in active if res[i] > tol and stall[i] < stall_checks]
        return calls, res

    def solved(self, res, tol=1e-12, floors=None):
        """Per-problem outcome: residual <= max(tol, FLOOR_FACTOR * floor)."""
        res = np.asarray(res)
        if floors is None:
            floors = self.floors([i for i in range(len(res)) if res[i] > tol])
            full = np.zeros(len(res))
            full[res > tol] = floors
            floors = full
        return res <= np.maximum(tol, FLOOR_FACTOR * np.asarray(floors)), np.asarray(floors)

    def solution(self, i):
        return self.keep[5 * i + 2].get()

    def close(self):
        for g in self.grids:
            g.destroy()
        if self.own:
            self.ctx.close()


def run(count=256, seed=0, prec=1, tol=1e-12, stall_checks=40):
    """Build, solve and time a batch; returns a summary dict."""
    probs = make_problems(count, seed)
    t0 = time.perf_counter()
    b = Batch(probs, prec=prec)
    gpu.check(b.lib.x2g_ctx_sync(b.ctx.h))
    t1 = time.perf_counter()
    gpu.check(b.lib.x2g_stats_enable(b.ctx.h, 1))
    calls, res = b.solve(tol=tol, stall_checks=stall_checks)
    gpu.check(b.lib.x2g_ctx_sync(b.ctx.h))
    t2 = time.perf_counter()
    st = (C.c_double * 6)()
    gpu.check(b.lib.x2g_stats_get(b.ctx.h, st))
    kernels = b.ctx.kernel_stats()
    gpu.check(b.lib.x2g_stats_enable(b.ctx.h, 0))
    ok, floors = b.solved(res, tol)
    b.close()
    return dict(problems=count, setup_s=t1 - t0, solve_s=t2 - t1, max_residual=float(res.max()),
                solved=int(ok.sum()), at_tol=int((res <= tol).sum()), residuals=res.tolist(),
                floors=floors.tolist(), calls=calls.tolist(), stats=list(st), kernel_stats=kernels)
