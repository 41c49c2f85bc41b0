"""Col-wise FP64 MCSOR of small grids (all sweeps in one launch, the grid in
LDS): bit for bit the result of one launch per sweep, and the oracle's where it
has the same colours (nni - 2 no multiple of 5), within the tolerance of the
FP64 sweeps everywhere, 1e-12 of the largest value.
"""
import ctypes as C

import numpy as np
import pytest

from oracle import pyoracle
from test_kernels_gpu import relerr, synthetic_problem

pytestmark = pytest.mark.gpu


def problem(nni, nmu, seed):
    P = synthetic_problem(nni, nmu, seed=seed)
    return P, (P["lhs"], P["rhs"])


# one to four groups of five a thread (and the row counts where that changes),
# every remainder of nni - 2 modulo 5, long and flat grids, the largest that
# fit and one that does not
@pytest.mark.parametrize("shape, sweeps", [
    ((19, 16), 1), ((57, 98), 2), ((57, 99), 7), ((58, 91), 2), ((61, 91), 10), ((91, 121), 10), ((92, 121), 3),
    ((95, 180), 3), ((21, 700), 2), ((500, 33), 2), ((103, 178), 2), ((103, 190), 2),
])
@pytest.mark.parametrize("isym, bkind", [(1, 0), (-1, 1)])
def test_resident_sweeps_vs_oracle(shape, sweeps, isym, bkind):
    from x2dhf_amd import gpu
    nni, nmu = shape
    print(f"shape={shape} sweeps={sweeps} isym={isym} bkind={bkind}", flush=True)
    P, _ = problem(nni, nmu, nni + nmu)
    win = pyoracle.putin(nni, nmu, isym, P["fun"])
    with gpu.Context(0) as ctx:
        g = gpu.Grid(ctx, nni, nmu, P["coef"], P["suppl"], P["vxi"], P["veta"])
        lhs, rhs = ctx.upload(P["lhs"]), ctx.upload(P["rhs"])

        def run(entry, per_sweep=False):
            w = ctx.upload(win)
            gpu.check(ctx.lib.x2g_set_sweep_plan(4 if per_sweep else 0, 0, 0))
            try:
                gpu.check(entry(g.h, isym, bkind, w.ptr, lhs.ptr, rhs.ptr, 1.8, sweeps))
            finally:
                gpu.check(ctx.lib.x2g_set_sweep_plan(0, 0, 0))
            return w.get()

        got = run(ctx.lib.x2g_mcsor)
        assert np.array_equal(got, run(ctx.lib.x2g_mcsor, per_sweep=True))
        if (nni - 2) % 5:
            want = pyoracle.mcsor(nni, nmu, isym, win.copy(), P["lhs"], P["rhs"], P["suppl"][bkind], P["suppl"][2],
                                  P["coef"][:16], P["coef"][16:21], 1.8, sweeps)
            assert relerr(got, want) < 1e-12, relerr(got, want)
        assert np.array_equal(run(ctx.lib.x2g_mcsor_noalloc), got)
        g.destroy()


def test_resident_batch_equals_single_calls():
    """A batch of unequal small grids, two macro-iterations of an odd number of
    sweeps: each function as x2g_mcsor leaves it alone."""
    from x2dhf_amd import gpu
    with gpu.Context(0) as ctx:
        grids, items, funs, want = [], [], [], []
        keep = []
        for k, (nni, nmu) in enumerate([(61, 91), (91, 121), (25, 61)]):
            P, _ = problem(nni, nmu, 40 + k)
            g = gpu.Grid(ctx, nni, nmu, P["coef"], P["suppl"], P["vxi"], P["veta"])
            grids.append(g)
            lhs, rhs = ctx.upload(P["lhs"]), ctx.upload(P["rhs"])
            keep += [lhs, rhs]
            for q in range(5):
                isym, bkind, omega = (1, -1)[q % 2], q // 2 % 2, 1.6 + 0.05 * q
                u = P["fun"] * (1.0 + 0.1 * q)
                f = ctx.upload(u)
                funs.append(f)
                items.append(gpu.RelaxItem(f.ptr, lhs.ptr, rhs.ptr, None, omega, isym, bkind, 0, k))
                for _ in range(2):
                    w = ctx.upload(pyoracle.putin(nni, nmu, isym, u))
                    gpu.check(ctx.lib.x2g_mcsor(g.h, isym, bkind, w.ptr, lhs.ptr, rhs.ptr, omega, 5))
                    u = pyoracle.putout(nni, nmu, w.get())
                    w.free()
                want.append(u)
        gh = (C.c_void_p * len(grids))(*[g.h.value for g in grids])
        gpu.check(ctx.lib.x2g_relax_batch(ctx.h, gh, (gpu.RelaxItem * len(items))(*items), len(items), 2, 5))
        for f, u in zip(funs, want):
            assert np.array_equal(f.get(), u)
        for g in grids:
            g.destroy()
