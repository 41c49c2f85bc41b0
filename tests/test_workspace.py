"""The workspace bound that admission budgets with (x2g_relax_workspace_bytes)
against what a call holds, for every scheme; the bound itself is host
arithmetic."""
import ctypes as C

import numpy as np
import pytest

from oracle import pyoracle
from test_kernels_gpu import synthetic_problem

SHAPES = [(7, 11), (23, 41), (24, 24), (61, 91), (91, 121), (169, 241), (331, 601), (481, 901), (505, 91)]


def test_bound_covers_every_scheme():
    """The bound without a scheme is the largest of the schemes'; the SOR orders
    that run a workgroup per sweep hold, by level, the function, lhs and rhs of
    every strand of rows: at least three arrays of nni x (nmu + nni / 2) doubles
    for the mirrored orders (a strand's levels are its rows and the columns'),
    nni x (nmu + nni) for the straight ones."""
    from x2dhf_amd import gpu
    lib = gpu.load()
    one = lib.x2g_relax_scheme_workspace_bytes
    for nni, nmu in SHAPES:
        each = {(m, o): one(nni, nmu, 0, m, o) for m in range(3) for o in range(10)}
        pad = 8 * (nni + 8) * (nmu + 8)
        assert min(each.values()) >= pad
        assert lib.x2g_relax_workspace_bytes(nni, nmu, 0) == max(each.values())
        assert one(nni, nmu, 1, 0, 0) == lib.x2g_relax_workspace_bytes(nni, nmu, 1)
        if min(nni, nmu) >= 24:
            assert each[1, 0] >= pad + 24 * nni * (nmu + nni - 16), (nni, nmu)
            if nni <= 504:
                assert each[1, 1] >= pad + 24 * nni * (nmu + nni - 16), (nni, nmu)
    assert one(91, 121, 1, 1, 0) == -1 and one(91, 121, 0, 3, 0) == -1 and one(91, 121, 0, 0, 10) == -1
    assert one(5, 121, 0, 0, 0) == -1 and one(91, 121, 2, 0, 0) == -1


def test_admission_counts_the_scheme():
    """A job's workspace: its potentials or orbitals in the scheme it asks for."""
    from x2dhf_amd import gpu, scf
    lib = gpu.load()
    one = lib.x2g_relax_scheme_workspace_bytes
    plain = scf.spec_workspace_bytes(scf.lih_spec(91, 121, 40.0))
    sor = scf.spec_workspace_bytes(scf.lih_spec(91, 121, 40.0, orb_method=1, pot_method=1, ordering=1))
    mixed = scf.spec_workspace_bytes(scf.lih_spec(91, 121, 40.0, orb_method=0, pot_method=1, ordering=0))
    # LiH: two orbitals, three potentials
    assert plain == 3 * one(91, 121, 0, 0, 0) + 2 * 65536
    assert sor == 3 * one(91, 121, 0, 1, 1) + 2 * 65536 > plain
    assert mixed == 3 * one(91, 121, 0, 1, 0) + 2 * one(91, 121, 0, 0, 0) + 2 * 65536


@pytest.mark.gpu
@pytest.mark.parametrize("nni, nmu", [(24, 24), (61, 91), (91, 121), (169, 241), (331, 601)])
def test_calls_hold_no_more_than_the_bound(nni, nmu):
    from x2dhf_amd import gpu
    P = synthetic_problem(nni, nmu, seed=1)
    for prec, method, ordering, count in [(0, m, o, 3) for m in range(3) for o in range(10)] + [(1, 0, 0, 3),
                                                                                               (1, 0, 0, 700)]:
        if count * nni * nmu > 8e6:
            count = int(8e6 / nni / nmu)
        print(f"{nni}x{nmu} prec={prec} method={method} ordering={ordering} count={count}", flush=True)
        with gpu.Context(0) as ctx:
            g = gpu.Grid(ctx, nni, nmu, P["coef"], P["suppl"], P["vxi"], P["veta"])
            lhs, rhs = ctx.upload(P["lhs"]), ctx.upload(P["rhs"])
            f = ctx.upload(np.tile(P["fun"], count))
            items = []
            for k in range(count):
                it = gpu.RelaxItem(f.ptr + 8 * k * g.n, lhs.ptr, rhs.ptr, None, 1.8, 1, 1, prec, 0)
                it.method, it.ordering = method, ordering
                items.append(it)
            gpu.check(ctx.lib.x2g_relax_batch(ctx.h, (C.c_void_p * 1)(g.h.value), (gpu.RelaxItem * count)(*items),
                                              count, 1, 2))
            held = ctx.counts()["workspace"]
            bound = ctx.lib.x2g_relax_scheme_workspace_bytes(nni, nmu, prec, method, ordering)
            assert 0 < held <= count * bound, (held, count * bound)
            g.destroy()


@pytest.mark.gpu
def test_more_sweeps_than_a_launch_of_fronts():
    """2 000 SOR sweeps: two launches of fronts, in the workspace of one."""
    from x2dhf_amd import gpu
    nni, nmu, sweeps = 61, 91, 2000
    P = synthetic_problem(nni, nmu, seed=2)
    win = pyoracle.putin(nni, nmu, 1, P["fun"])
    with gpu.Context(0) as ctx:
        g = gpu.Grid(ctx, nni, nmu, P["coef"], P["suppl"], P["vxi"], P["veta"])
        lhs, rhs = ctx.upload(P["lhs"]), ctx.upload(P["rhs"])
        for name in ("col-wise", "middle", "rrow-wis"):
            want = pyoracle.relax_ordered(nni, nmu, 1, win.copy(), P["lhs"], P["rhs"], P["suppl"][1], P["suppl"][2],
                                          P["coef"][:16], P["coef"][16:21], 1.8, sweeps, 1, name)
            w, before = ctx.upload(win), ctx.counts()["front"]
            gpu.check(ctx.lib.x2g_relax_ordered(g.h, 1, 1, w.ptr, lhs.ptr, rhs.ptr, 1.8, sweeps, 1,
                                                pyoracle.ORDERINGS[name]))
            assert ctx.counts()["front"] - before == 2
            assert np.array_equal(w.get(), want), name
            # (workspaces grow by half)
            assert ctx.counts()["workspace"] <= 1.5 * gpu.load().x2g_relax_workspace_bytes(nni, nmu, 0)
        g.destroy()
