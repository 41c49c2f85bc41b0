"""bench.py's traffic summary and roofline line name the kernels that ran (host
arithmetic; counter files as rocprofv3 writes them)."""
import json
import os
import sys

import pytest

from conftest import ROOT

sys.path.insert(0, ROOT)
import bench  # noqa: E402

COPY = 1201 * 1201 * 8 / 1024.0  # KiB


def counters(path, names, kib):
    with open(path, "w") as f:
        f.write('"Dispatch_Id","Kernel_Name","Counter_Name","Counter_Value"\n')
        for i, n in enumerate(names):
            f.write(f'{i + 1},"{n}","C",{kib(i, n)}\n')


def dispatches(*sweeps):
    return (["x2g::k_lincomb(double*, double const*, double, x2g_term const*, int, long)"] * 3 +
            ["x2g::k_residual_rows<true>(x2g::ResDesc const*)"] + [n for n, k in sweeps for _ in range(k)])


CHAIN = "x2g::k_chain_f32(x2g::ChainPack const*, x2g::ChainSeg const*, x2g::ChainWg const*, int, int)"
F32 = "void x2g::k_sweep<float, 1, 528, 2>(x2g::SweepDesc<float> const*, x2g::SweepSeg const*, int const*, int, int)"
F64 = F32.replace("float, 1, 528, 2", "double, 1, 352, 4").replace("<float>", "<double>")


def value(kernel_kib):
    def f(i, n):
        if "k_lincomb" in n:
            return COPY / 2  # a counter of half the bytes: factor 2
        return next((v / 2 for k, v in kernel_kib.items() if k in n), 1.0)
    return f


@pytest.mark.parametrize("probe, runs", [("n2", [(CHAIN, 5), (F64, 10)]), ("n2", [(F32, 10), (F64, 10)]),
                                         ("stream", [(CHAIN, 5), (F32, 10)])])
def test_summary_of_the_probes(tmp_path, monkeypatch, probe, runs):
    out = tmp_path / "traffic.json"
    monkeypatch.setattr(bench, "TRAFFIC", str(out))
    monkeypatch.setattr(bench, "TRAFFIC_STREAM", str(out))
    fetch, write = tmp_path / "f.csv", tmp_path / "w.csv"
    kib = {"k_chain_f32": 3e5, "k_sweep<float": 8e5, "k_sweep<double": 16e5}
    counters(fetch, dispatches(*runs), value(kib))
    counters(write, dispatches(*runs), value({k: v / 4 for k, v in kib.items()}))
    bench.traffic_summary(str(fetch), str(write), probe, 16)
    got = json.load(open(out))
    points = 352 * 329 * 596 if probe == "n2" else sum(c * (n - 2) * (m - 5) for n, m, c in bench.STREAM_PROBE)
    want = {{CHAIN: "k_chain_f32", F32: "k_sweep<float>", F64: "k_sweep<double>"}[n]: k for n, k in runs}
    assert set(got["kernels"]) == set(want)
    for name, k in got["kernels"].items():
        # an FP32 correction's first launch does not read its source
        assert k["launches"] == want[name] - ("double" not in name)
        words = 32.0 if "double" in name else 16.0
        assert k["algorithmic_bytes_per_launch"] == words * points
        assert k["hbm_bytes_per_launch"] == pytest.approx(1.25 * 1024 * kib[name.rstrip(">")])
    # the roofline of the kernel that took most of the time, with its own ratio
    name = {"k_chain_f32": "chain", "k_sweep<float>": "sweep32"}[next(iter(k for k in got["kernels"] if "double" not in k))]
    stats = {name: (100.0, 50.0, 4e10), "sweep64": (10.0, 1.0, 1e8)}
    roof = bench.sweep_roofline(stats, str(out))
    assert roof["kernel"] == bench.KERNELS[name] and roof["launches"] == 100
    assert roof["achieved"] == pytest.approx(4e10 / 0.05 / 1e9) and roof["avg_launch_us"] == pytest.approx(500.0)
    assert roof["traffic"] == pytest.approx(got["kernels"][roof["kernel"]]["traffic_over_algorithmic"] * 4e8)
    assert set(roof["all_kernels"]) == {bench.KERNELS[name], "k_sweep<double>"}
    # a kernel the probe did not run has no ratio
    other = bench.sweep_roofline({"resident": (1.0, 1.0, 1e8)}, str(out))
    assert other["kernel"] == "k_resident" and other["traffic"] is None
    assert bench.sweep_roofline({})["kernel"] is None


def test_recorded_ratios_name_their_kernels():
    for path in (bench.TRAFFIC, bench.TRAFFIC_STREAM):
        got = json.load(open(path))
        assert "k_chain_f32" in got["kernels"], path
        for k in got["kernels"].values():
            assert 0.5 < k["traffic_over_algorithmic"] < 4.0, path


def test_a_step_is_a_share_of_one_stream(monkeypatch, capsys):
    """Without --count the timed work is one stream, whatever the steps: 64
    requests, or 4 a step; with it, a stream of that many per step.  Energies
    compare equal where both servings of a request stopped on a NaN."""
    from types import SimpleNamespace as Ns
    nan = float("nan")
    for steps, count, streams, per in ((1, None, 1, 64), (10, None, 1, 64), (20, None, 1, 80), (3, 5, 3, 5)):
        sizes = []

        def serve_stream(reqs, prec, stats=False, graphs=False, groups=1):
            sizes.append(len(reqs))
            res = [dict(stop="not a number", etot=nan) if k == 3 else
                   dict(stop="orbital energy threshold", etot=-1.0 - k) for k in range(len(reqs))]
            return [Ns(result=r, latency=1.0) for r in res], 2.0, {}

        monkeypatch.setattr(bench, "serve_stream", serve_stream)
        argv = ["bench.py", "--steps", str(steps), "--warmup", "2", "--no-cpu", "--no-plain"]
        monkeypatch.setattr(sys, "argv", argv + (["--count", str(count)] if count else []))
        bench.bench_stream(bench.parse())
        line = json.loads(capsys.readouterr().out.strip().splitlines()[-1])
        # two warm-up streams, then as served, in FP64, with graphs, in two groups
        assert sizes[2:] == [per] * 4 * streams and max(sizes[:2]) <= 8
        assert line["steps"] == steps and line["requests"] == streams * per
        assert line["config"]["requests_per_step"] == streams * per / steps
        assert line["ms_per_step"] == pytest.approx(2000.0 * streams / steps)
        assert line["graph_replay"]["energies_identical_to_eager"]
        assert line["two_groups_graph_replay"]["energies_identical_to_eager"]
