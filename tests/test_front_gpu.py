"""Ordered SOR sweeps as moving fronts against the oracle's sequential sor: every
mesh ordering forward and backward, equal bit for bit.  Shapes: the smallest
grids that run as fronts and one below, odd and even middles, columns of one
wave to eight and one more than a strand may have, few rows and many; one
sweep, and more than follow each other on the chip.
"""
import ctypes as C

import numpy as np
import pytest

from oracle import pyoracle
from test_kernels_gpu import relerr, synthetic_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape, sweeps", [
    ((23, 41), 3), ((25, 24), 4), ((24, 25), 1), ((31, 61), 300), ((57, 90), 2), ((121, 47), 5), ((248, 60), 3),
    ((249, 62), 3), ((377, 43), 2), ((504, 91), 2), ((505, 91), 2), ((61, 701), 4),
])
def test_fronts_vs_oracle(shape, sweeps):
    from x2dhf_amd import gpu
    nni, nmu = shape
    P = synthetic_problem(nni, nmu, seed=5 * nni + nmu)
    args = (P["lhs"], P["rhs"], P["suppl"][1], P["suppl"][2], P["coef"][:16], P["coef"][16:21], 1.8)
    with gpu.Context(0) as ctx:
        g = gpu.Grid(ctx, nni, nmu, P["coef"], P["suppl"], P["vxi"], P["veta"])
        lhs, rhs = ctx.upload(P["lhs"]), ctx.upload(P["rhs"])
        for name, code in pyoracle.ORDERINGS.items():
            for method in (1, 2):
                isym = 1 if (code + method) % 2 else -1
                print(f"shape={shape} sweeps={sweeps} {name} method={method} isym={isym}", flush=True)
                win = pyoracle.putin(nni, nmu, isym, P["fun"])
                want = pyoracle.relax_ordered(nni, nmu, isym, win.copy(), *args, sweeps, method, name)
                w = ctx.upload(win)
                gpu.check(ctx.lib.x2g_relax_ordered(g.h, isym, 1, w.ptr, lhs.ptr, rhs.ptr, 1.8, sweeps, method, code))
                got = w.get()
                w.free()
                assert np.array_equal(got, want), (name, method, relerr(got, want))
        g.destroy()


def test_fronts_of_a_mixed_batch():
    """Problems of several sizes and orderings in one call, more workgroups
    than compute units, with schemes that do not run as fronts among them."""
    from x2dhf_amd import gpu
    schemes = [(1, 1), (1, 0), (2, 0), (1, 4), (1, 6), (2, 1), (0, 1)]
    with gpu.Context(0) as ctx:
        grids, items, keep, want = [], [], [], []
        for k, (nni, nmu) in enumerate([(31, 41), (91, 121), (121, 61)]):
            P = synthetic_problem(nni, nmu, seed=k)
            g = gpu.Grid(ctx, nni, nmu, P["coef"], P["suppl"], P["vxi"], P["veta"])
            grids.append(g)
            lhs, rhs = ctx.upload(P["lhs"]), ctx.upload(P["rhs"])
            keep += [lhs, rhs]
            for q in range(14):
                method, ordering = schemes[q % len(schemes)]
                isym, bkind = (1, -1)[q % 2], (q // 2) % 2
                u = P["fun"] * (1.0 + 0.01 * q)
                wp = pyoracle.putin(nni, nmu, isym, u)
                pyoracle.relax_ordered(nni, nmu, isym, wp, P["lhs"], P["rhs"], P["suppl"][bkind], P["suppl"][2],
                                       P["coef"][:16], P["coef"][16:21], 1.7, 9, method, ordering)
                want.append(pyoracle.putout(nni, nmu, wp))
                f = ctx.upload(u)
                keep.append(f)
                it = gpu.RelaxItem(f.ptr, lhs.ptr, rhs.ptr, None, 1.7, isym, bkind, 0, k)
                it.method, it.ordering = method, ordering
                items.append((it, f))
        gh = (C.c_void_p * len(grids))(*[g.h.value for g in grids])
        arr = (gpu.RelaxItem * len(items))(*[it for it, _ in items])
        print(f"{len(items)} items", flush=True)
        gpu.check(ctx.lib.x2g_relax_batch(ctx.h, gh, arr, len(items), 1, 9))
        for (it, f), w in zip(items, want):
            got = f.get()
            assert np.array_equal(got, w), (it.method, it.ordering, it.grid_index, relerr(got, w))
        for g in grids:
            g.destroy()
