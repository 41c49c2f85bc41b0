"""Launch descriptors of a relaxation call: what a call stages depends on its
items, not on how often or how long they are relaxed, and every descriptor
stays what it was until the call's last launch has read it.
"""
import numpy as np
import pytest

from oracle import pyoracle
from test_kernels_gpu import synthetic_problem

pytestmark = pytest.mark.gpu


class Batch:
    """count functions of one grid as relax items of one scheme."""

    def __init__(self, ctx, nni, nmu, count, prec=0, method=0, ordering=0, seed=5):
        from x2dhf_amd import gpu
        self.ctx, self.P = ctx, synthetic_problem(nni, nmu, seed=seed)
        P = self.P
        self.grid = gpu.Grid(ctx, nni, nmu, P["coef"], P["suppl"], P["vxi"], P["veta"])
        self.lhs, self.rhs = ctx.upload(P["lhs"]), ctx.upload(P["rhs"])
        self.u = np.tile(P["fun"], (count, 1)) * (1.0 + 0.1 * (np.arange(count) % 5))[:, None]
        self.f = ctx.upload(self.u)
        items = []
        for k in range(count):
            it = gpu.RelaxItem(self.f.ptr + 8 * k * nni * nmu, self.lhs.ptr, self.rhs.ptr, None, 1.8, 1, 1, prec, 0)
            it.method, it.ordering = method, ordering
            items.append(it)
        self.arr, self.n = (gpu.RelaxItem * count)(*items), count
        self.gh = (gpu._vp * 1)(self.grid.h.value)

    def relax(self, maxsor1, maxsor2):
        """Bytes staged by one call from the starting functions; the results."""
        from x2dhf_amd import gpu
        self.f.set(self.u)
        before = self.ctx.counts()["staged"]
        gpu.check(self.ctx.lib.x2g_relax_batch(self.ctx.h, self.gh, self.arr, self.n, maxsor1, maxsor2))
        return self.ctx.counts()["staged"] - before, self.f.get().reshape(self.n, -1)

    def relax_first(self, count):
        """As relax(2, 2) of the first `count` functions."""
        from x2dhf_amd import gpu
        self.f.set(self.u)
        gpu.check(self.ctx.lib.x2g_relax_batch(self.ctx.h, self.gh, self.arr, count, 2, 2))
        return self.f.get().reshape(len(self.u), -1)


# one workgroup per grid, fronts, level tables (their one ordering), the
# strip sweep of either precision
@pytest.mark.parametrize("kw", [
    dict(nni=61, nmu=91, count=4), dict(nni=61, nmu=91, count=4, method=1, ordering=1),
    dict(nni=61, nmu=91, count=4, method=1, ordering=2), dict(nni=169, nmu=241, count=2),
    dict(nni=61, nmu=91, count=4, prec=1),
])
def test_macro_iterations_stage_nothing(kw):
    from x2dhf_amd import gpu
    print(kw, flush=True)
    with gpu.Context(0) as ctx:
        b = Batch(ctx, **kw)
        b.relax(1, 2)  # tunes the plan, builds the tables
        one, _ = b.relax(1, 2)
        many, got = b.relax(7, 2)
        assert many == one, (one, many)
        # seven macro-iterations in one call: as seven calls
        b.f.set(b.u)
        for _ in range(7):
            gpu.check(ctx.lib.x2g_relax_batch(ctx.h, b.gh, b.arr, b.n, 1, 2))
        assert np.array_equal(b.f.get().reshape(b.n, -1), got)
        b.grid.destroy()


def test_more_chained_sweeps_stage_nothing_more():
    """400 sweeps of a large FP32 batch stage what 200 do, and leave what one
    launch per sweep leaves (an odd number, so that a launch is shorter)."""
    from x2dhf_amd import gpu
    with gpu.Context(0) as ctx:
        b = Batch(ctx, 91, 121, 350, prec=1)
        out = {}
        for sweeps in (200, 400, 401):
            print(sweeps, flush=True)
            n = ctx.counts()["chain"]
            out[sweeps] = b.relax(1, sweeps)
            n = ctx.counts()["chain"] - n
            assert n > 1 and n < sweeps
        assert out[400][0] == out[200][0], (out[200][0], out[400][0])
        gpu.check(ctx.lib.x2g_set_sweep_plan(4, 0, 0))
        try:
            _, want = b.relax(1, 401)
        finally:
            gpu.check(ctx.lib.x2g_set_sweep_plan(0, 0, 0))
        assert np.array_equal(out[401][1], want)
        b.grid.destroy()


def test_descriptors_of_one_call_beyond_the_ring():
    """45 000 ordered functions in one call: their descriptors take more than
    the 16 MiB ring, and the first staged are read again in the second
    macro-iteration.  Then a small call, which gives the outgrown ring back."""
    from x2dhf_amd import gpu
    nni, nmu, n = 24, 24, 45000
    with gpu.Context(0) as ctx:
        b = Batch(ctx, nni, nmu, n, method=1, ordering=0)
        P, want = b.P, []
        for k in range(5):
            u = b.u[k]
            for _ in range(2):
                w = pyoracle.putin(nni, nmu, 1, u)
                pyoracle.relax_ordered(nni, nmu, 1, w, P["lhs"], P["rhs"], P["suppl"][1], P["suppl"][2],
                                       P["coef"][:16], P["coef"][16:21], 1.8, 2, 1, "col-wise")
                u = pyoracle.putout(nni, nmu, w)
            want.append(u)
        print(f"{n} items", flush=True)
        staged, got = b.relax(2, 2)
        assert staged > 16 << 20
        assert np.array_equal(got.reshape(n // 5, 5, -1), np.broadcast_to(want, (n // 5, 5, nni * nmu)))
        for count in (7, n, 7):
            got = b.relax_first(count)
            assert np.array_equal(got[:count], np.tile(want, (n // 5, 1))[:count]), count
        b.grid.destroy()
