"""Which kernel a call runs, asserted by the context's launch counts, and its
results there: the chained FP32 sweeps against one launch per sweep, over
several macro-iterations, in mixed batches and replayed from a graph; the grids
resident on a compute unit; the ordered sweeps of many sweeps that the level
tables still run.
"""
import numpy as np
import pytest

from oracle import pyoracle
from test_kernels_gpu import relerr, synthetic_problem

pytestmark = pytest.mark.gpu


class Ran:
    """The launches of each kernel inside a `with` block."""

    def __init__(self, ctx):
        self.ctx = ctx

    def __enter__(self):
        self.before = self.ctx.counts()
        return self

    def __exit__(self, *a):
        self.n = {k: v - self.before[k] for k, v in self.ctx.counts().items()}
        self.kernels = {k for k, v in self.n.items() if v and k not in ("staged", "workspace")}


class Problems:
    """Relax items on several grids: (nni, nmu, count, prec, method, ordering)
    each, of both parities and b(mu), from non-zero functions."""

    def __init__(self, ctx, shapes):
        from x2dhf_amd import gpu
        self.ctx, self.grids, self.sets, items = ctx, [], [], []
        for gi, (nni, nmu, count, prec, method, ordering) in enumerate(shapes):
            P = synthetic_problem(nni, nmu, seed=70 + gi)
            self.grids.append(gpu.Grid(ctx, nni, nmu, P["coef"], P["suppl"], P["vxi"], P["veta"]))
            l, r = ctx.upload(P["lhs"]), ctx.upload(P["rhs"])
            u = np.tile(P["fun"], (count, 1)) * (1.0 + 0.05 * (np.arange(count) % 7))[:, None]
            f = ctx.upload(u)
            self.sets.append((f, u, l, r))
            for k in range(count):
                it = gpu.RelaxItem(f.ptr + 8 * k * nni * nmu, l.ptr, r.ptr, None, (1.9, 1.7)[k % 3 == 1],
                                   (1, -1)[k % 2], int(k % 5 == 2), prec, gi)
                it.method, it.ordering = method, ordering
                items.append(it)
        self.arr, self.n = (gpu.RelaxItem * len(items))(*items), len(items)
        self.gh = (gpu._vp * len(self.grids))(*[g.h.value for g in self.grids])

    def reset(self):
        for f, u, _, _ in self.sets:
            f.set(u)

    def relax(self, maxsor1, maxsor2):
        from x2dhf_amd import gpu
        gpu.check(self.ctx.lib.x2g_relax_batch(self.ctx.h, self.gh, self.arr, self.n, maxsor1, maxsor2))

    def get(self):
        return [f.get() for f, _, _, _ in self.sets]

    def close(self):
        for g in self.grids:
            g.destroy()


def per_sweep(ctx, on):
    """A fixed cut of k_sweep: one launch per sweep."""
    from x2dhf_amd import gpu
    gpu.check(ctx.lib.x2g_set_sweep_plan(4 if on else 0, 0, 0))


# every remainder of nni - 2 modulo 5; the served grids; one and two
# macro-iterations, on functions that are not zero
@pytest.mark.parametrize("shapes, maxsor1, maxsor2", [
    ([(25, 85, 2500)], 1, 4), ([(37, 61, 2500)], 2, 7), ([(91, 121, 701)], 2, 10), ([(163, 241, 151)], 1, 10),
    ([(331, 601, 352)], 1, 4), ([(91, 121, 350), (169, 241, 101)], 2, 11), ([(67, 91, 1100)], 1, 3),
    ([(505, 901, 14), (409, 721, 20), (361, 601, 20), (217, 361, 16), (169, 241, 16)], 1, 10),
])
def test_chained_sweeps_equal_one_launch_per_sweep(shapes, maxsor1, maxsor2):
    from x2dhf_amd import gpu
    print(f"{shapes} {maxsor1} x {maxsor2}", flush=True)
    with gpu.Context(0) as ctx:
        p = Problems(ctx, [(*s, 1, 0, 0) for s in shapes])
        with Ran(ctx) as ran:
            p.relax(maxsor1, maxsor2)
        print(ran.n, flush=True)
        assert ran.kernels == {"chain"}
        got = p.get()
        p.reset()
        per_sweep(ctx, True)
        try:
            with Ran(ctx) as ran:
                p.relax(maxsor1, maxsor2)
        finally:
            per_sweep(ctx, False)
        assert ran.kernels == {"sweep32"} and ran.n["sweep32"] == maxsor1 * maxsor2
        for a, b in zip(got, p.get()):
            assert np.array_equal(a, b)
        p.close()


def test_chains_beside_other_schemes_and_replayed():
    """FP64, ordered and chained items in one call of two macro-iterations:
    each as in a call of its own, and the captured call's replays as the eager
    ones, with eager work and synchronisations between them."""
    from x2dhf_amd import gpu
    shapes = [(91, 121, 700, 1, 0, 0), (61, 91, 3, 0, 0, 0), (61, 91, 2, 0, 1, 1), (57, 91, 2, 0, 1, 2)]
    calls, res = 5, {}
    with gpu.Context(0) as ctx:
        p = Problems(ctx, shapes)
        with Ran(ctx) as ran:
            p.relax(2, 5)
        print(ran.n, flush=True)
        assert ran.kernels == {"chain", "resident", "front", "levels"}
        got = p.get()
        p.close()
    for k, s in enumerate(shapes):
        with gpu.Context(0) as ctx:
            q = Problems(ctx, [s] if k == 0 else shapes[:k + 1])
            # the last set alone, with its own inputs
            first = sum(t[2] for t in shapes[:k])
            arr = (gpu.RelaxItem * s[2])(*list(q.arr)[first if k else 0:])
            gpu.check(ctx.lib.x2g_relax_batch(ctx.h, q.gh, arr, s[2], 2, 5))
            assert np.array_equal(q.get()[-1], got[k]), s
            q.close()
    for graphs in (0, 1):
        with gpu.Context(0) as ctx:
            p = Problems(ctx, shapes)
            gpu.check(ctx.lib.x2g_set_graphs(ctx.h, graphs))
            other, out = ctx.alloc(1 << 18), []
            print(f"graphs={graphs}", flush=True)
            for call in range(calls):
                p.relax(2, 5)
                other.fill(float(call))
                ctx.sync()
                out.append(p.get())
            n = gpu._vp, gpu.C.c_longlong(), gpu.C.c_longlong()
            gpu.check(ctx.lib.x2g_graph_counts(ctx.h, gpu.C.byref(n[1]), gpu.C.byref(n[2])))
            assert (n[1].value, n[2].value >= 2) == ((1, True) if graphs else (0, False))
            res[graphs] = out
            p.close()
    for a, b in zip(res[0], res[1]):
        for x, y in zip(a, b):
            assert np.array_equal(x, y)


# one group of five a thread to four, long and flat grids within k_sweep's
# width, the widest of them; both entry points
@pytest.mark.parametrize("nni, nmu", [(19, 16), (57, 99), (91, 121), (21, 700), (300, 61), (331, 55), (336, 16)])
def test_small_grids_run_resident(nni, nmu):
    from x2dhf_amd import gpu
    print(f"{nni}x{nmu}", flush=True)
    P = synthetic_problem(nni, nmu, seed=nni)
    win = pyoracle.putin(nni, nmu, 1, P["fun"])
    want = pyoracle.mcsor(nni, nmu, 1, win.copy(), P["lhs"], P["rhs"], P["suppl"][1], P["suppl"][2], P["coef"][:16],
                          P["coef"][16:21], 1.8, 7)
    with gpu.Context(0) as ctx:
        g = gpu.Grid(ctx, nni, nmu, P["coef"], P["suppl"], P["vxi"], P["veta"])
        lhs, rhs = ctx.upload(P["lhs"]), ctx.upload(P["rhs"])
        out = {}
        for name, entry, fixed, kernel in (("mcsor", ctx.lib.x2g_mcsor, False, "resident"),
                                           ("noalloc", ctx.lib.x2g_mcsor_noalloc, False, "resident"),
                                           ("per sweep", ctx.lib.x2g_mcsor, True, "sweep64")):
            w = ctx.upload(win)
            per_sweep(ctx, fixed)
            try:
                with Ran(ctx) as ran:
                    gpu.check(entry(g.h, 1, 1, w.ptr, lhs.ptr, rhs.ptr, 1.8, 7))
            finally:
                per_sweep(ctx, False)
            assert ran.kernels == {kernel}, (name, ran.n)
            out[name] = w.get()
        assert np.array_equal(out["mcsor"], out["per sweep"]) and np.array_equal(out["noalloc"], out["mcsor"])
        if (nni - 2) % 5:
            assert relerr(out["mcsor"], want) < 1e-12, relerr(out["mcsor"], want)
        g.destroy()


# orders and widths that do not run as fronts, more sweeps than the level
# tables pipeline at once (64), forward and backward
@pytest.mark.parametrize("nni, nmu, method, name", [
    (91, 121, 1, "middlemt"), (91, 121, 2, "middlemt"), (511, 61, 1, "middle"), (91, 121, 2, "middle"),
    (91, 121, 0, "middle"),
])
def test_level_tables_beyond_one_pipeline(nni, nmu, method, name):
    from x2dhf_amd import gpu
    print(f"{nni}x{nmu} {name} method={method}", flush=True)
    P = synthetic_problem(nni, nmu, seed=12)
    win = pyoracle.putin(nni, nmu, 1, P["fun"])
    want = pyoracle.relax_ordered(nni, nmu, 1, win.copy(), P["lhs"], P["rhs"], P["suppl"][1], P["suppl"][2],
                                  P["coef"][:16], P["coef"][16:21], 1.7, 70, method, name)
    with gpu.Context(0) as ctx:
        g = gpu.Grid(ctx, nni, nmu, P["coef"], P["suppl"], P["vxi"], P["veta"])
        lhs, rhs, w = ctx.upload(P["lhs"]), ctx.upload(P["rhs"]), ctx.upload(win)
        with Ran(ctx) as ran:
            gpu.check(ctx.lib.x2g_relax_ordered(g.h, 1, 1, w.ptr, lhs.ptr, rhs.ptr, 1.7, 70, method,
                                                pyoracle.ORDERINGS[name]))
        assert ran.kernels == {"levels"}
        assert np.array_equal(w.get(), want), relerr(w.get(), want)
        g.destroy()


def test_ordered_call_keeps_the_graphs_of_others():
    """An ordered call that first reserves the workspace of fronts: the graph of
    a colour-sweep call, which does not address it, is replayed as before."""
    from x2dhf_amd import gpu
    res = {}
    for graphs in (0, 1):
        with gpu.Context(0) as ctx:
            p = Problems(ctx, [(169, 241, 3, 0, 0, 0)])
            q = Problems(ctx, [(91, 121, 1, 0, 1, 1)])
            gpu.check(ctx.lib.x2g_set_graphs(ctx.h, graphs))
            c, r, out = gpu.C.c_longlong(), gpu.C.c_longlong(), []
            print(f"graphs={graphs}", flush=True)
            for call in range(4):
                p.relax(1, 4)
                ctx.sync()
            gpu.check(ctx.lib.x2g_graph_counts(ctx.h, c, r))
            before = c.value, r.value
            q.relax(1, 4)
            for call in range(3):
                p.relax(1, 4)
                ctx.sync()
                out.append(p.get())
            gpu.check(ctx.lib.x2g_graph_counts(ctx.h, c, r))
            assert (c.value - before[0], r.value - before[1]) == (0, 3 * graphs)
            res[graphs] = out
            p.close()
            q.close()
    for a, b in zip(res[0], res[1]):
        assert np.array_equal(a, b)


# (shape, kernel, words per point and launch beyond the first, launches of ten sweeps)
@pytest.mark.parametrize("shape, kernel, per_launch", [
    ((91, 121, 700, 1, 0, 0), "chain", False), ((91, 121, 10, 1, 0, 0), "sweep32", True),
    ((169, 241, 2, 0, 0, 0), "sweep64", True), ((61, 91, 2, 0, 0, 0), "resident", False),
    ((61, 91, 2, 0, 1, 1), "front", False), ((61, 91, 2, 0, 1, 2), "levels", False),
    ((361, 61, 2, 0, 0, 0), "strip", True),
])
def test_statistics_count_what_ran(shape, kernel, per_launch):
    """Launches and algorithmic bytes by kernel: a launch of several sweeps is
    one launch that moves its arrays once, and the first sweep of an FP32
    correction does not read its zero source."""
    from x2dhf_amd import gpu
    nni, nmu, count, prec = shape[:4]
    sweeps, iters = 10, 2
    with gpu.Context(0) as ctx:
        p = Problems(ctx, [shape])
        p.relax(1, sweeps)  # tunes the plan
        gpu.check(ctx.lib.x2g_stats_enable(ctx.h, 1))
        with Ran(ctx) as ran:
            p.relax(iters, sweeps)
        st, tot = ctx.kernel_stats(), (gpu._dbl * 6)()
        gpu.check(ctx.lib.x2g_stats_get(ctx.h, tot))
        gpu.check(ctx.lib.x2g_stats_enable(ctx.h, 0))
        assert ran.kernels == set(st) == {kernel}
        launches, ms, nbytes = st[kernel]
        assert launches == ran.n[kernel] and (launches == iters * sweeps) == per_launch
        word, points = (4, 8)[prec == 0], count * (nni - 2) * (nmu - 5)
        assert nbytes == word * points * (4 * launches - prec * iters)
        assert ms > 0 and tuple(tot[3 * prec:3 * prec + 3]) == (launches, ms, nbytes) and tot[3 * (1 - prec)] == 0
        p.close()


def test_problems_on_grids_of_their_own():
    """Chains are slower where each problem has a grid of its own and a workgroup
    holds several: such a batch keeps one launch per sweep, one on a common grid
    does not, and the results are the same."""
    from x2dhf_amd import gpu
    nni, nmu, count = 331, 601, 120
    res = {}
    for own in (False, True):
        print(f"own={own}", flush=True)
        with gpu.Context(0) as ctx:
            P = synthetic_problem(nni, nmu, seed=8)
            grids = [gpu.Grid(ctx, nni, nmu, P["coef"], P["suppl"], P["vxi"], P["veta"])
                     for _ in range(count if own else 1)]
            l, r = ctx.upload(P["lhs"]), ctx.upload(P["rhs"])
            f = ctx.upload(np.tile(P["fun"], count))
            items = [gpu.RelaxItem(f.ptr + 8 * k * nni * nmu, l.ptr, r.ptr, None, 1.9, (1, -1)[k % 2], 1, 1,
                                   k if own else 0) for k in range(count)]
            gh = (gpu._vp * len(grids))(*[g.h.value for g in grids])
            with Ran(ctx) as ran:
                gpu.check(ctx.lib.x2g_relax_batch(ctx.h, gh, (gpu.RelaxItem * count)(*items), count, 1, 10))
            print(ran.n, flush=True)
            assert ran.kernels == ({"sweep32"} if own else {"chain"})
            res[own] = f.get().reshape(count, -1)
            for g in grids:
                g.destroy()
    assert np.array_equal(res[False], res[True])


# the smallest fronts, uneven middles; straight, reversed and mirrored orders
@pytest.mark.parametrize("nni, nmu, method, name", [
    (24, 24, 1, "col-wise"), (24, 25, 1, "middle"), (25, 24, 2, "col-wise"), (31, 41, 1, "rrow-wis"),
    (41, 51, 1, "test2"), (45, 67, 1, "test1"),
])
def test_small_ordered_grids_take_the_faster_path(nni, nmu, method, name):
    """Few small problems run several sweeps on the level tables, one sweep as
    fronts; more problems than CUs, and problems beside a large one, as fronts:
    bit for bit what the oracle gives."""
    from x2dhf_amd import gpu
    code, sweeps, cus = pyoracle.ORDERINGS[name], 20, 256
    with gpu.Context(0) as ctx:
        for count, n, beside, kernel in ((1, sweeps, False, "levels"), (6, sweeps, False, "levels"),
                                         (1, 1, False, "front"), (cus + 1, sweeps, False, "front"),
                                         (2, sweeps, True, "front")):
            print(f"{nni}x{nmu} {name} method={method} count={count} sweeps={n} beside={beside}", flush=True)
            p = Problems(ctx, [(nni, nmu, count, 0, method, code)] + beside * [(121, 161, 1, 0, 1, 1)])
            with Ran(ctx) as ran:
                p.relax(1, n)
            assert ran.kernels == {kernel}, ran.n
            got = p.get()[0].reshape(count, -1)
            P, u = synthetic_problem(nni, nmu, seed=70), p.sets[0][1]
            for k in {0, 1, 2, count - 1} & set(range(count)):
                it = p.arr[k]
                w = pyoracle.putin(nni, nmu, it.isym, u[k])
                pyoracle.relax_ordered(nni, nmu, it.isym, w, P["lhs"], P["rhs"], P["suppl"][it.bkind], P["suppl"][2],
                                       P["coef"][:16], P["coef"][16:21], it.omega, n, method, name)
                assert np.array_equal(got[k], pyoracle.putout(nni, nmu, w)), (k, count)
            p.close()
        P = synthetic_problem(nni, nmu, seed=3)
        win = pyoracle.putin(nni, nmu, 1, P["fun"])
        g = gpu.Grid(ctx, nni, nmu, P["coef"], P["suppl"], P["vxi"], P["veta"])
        lhs, rhs = ctx.upload(P["lhs"]), ctx.upload(P["rhs"])
        for n, kernel in ((1, "front"), (sweeps, "levels")):
            want = pyoracle.relax_ordered(nni, nmu, 1, win.copy(), P["lhs"], P["rhs"], P["suppl"][1], P["suppl"][2],
                                          P["coef"][:16], P["coef"][16:21], 1.8, n, method, name)
            w = ctx.upload(win)
            with Ran(ctx) as ran:
                gpu.check(ctx.lib.x2g_relax_ordered(g.h, 1, 1, w.ptr, lhs.ptr, rhs.ptr, 1.8, n, method, code))
            assert ran.kernels == {kernel}, ran.n
            assert np.array_equal(w.get(), want), n
        g.destroy()
