"""Launch shapes left to choose: the packing and the table placement depend on
the number of runs, the results do not.  Every run's outputs equal those of
the widest packing with the tables in global memory, bit for bit, on both
sides of the rule's turning points (a wave per SIMD, two, three; few lanes,
many; with digests and without; models whose slots are tested one after
another), and so do the importance sampler's.
"""
from __future__ import annotations

import numpy as np
import pytest

import cusmc_amd as cs
from cusmc_amd import generators as G

from _models import large_model

pytestmark = pytest.mark.gpu

PER_RUN = ("flag", "value", "steps", "transitions", "time")


def _query(name):
    if name == "csma":
        net = cs.ParsedNetwork.from_string(large_model("CSMA_100.xml"), "Process0.SUCCESS")
        return net, cs.reach_query(2.0, max_steps=60)
    kind, n = name.split("-")
    if kind == "race":
        net = cs.ParsedNetwork.from_string(G.race_network(int(n))[0], "")
        return net, cs.var_query(net.variable_id("count"), 3.0, threshold=2, max_steps=60)
    if kind == "fischer":
        net = cs.ParsedNetwork.from_string(G.fischer_network(int(n))[0], "P0.cs")
        return net, cs.reach_query(8.0, max_steps=60)
    net = cs.ParsedNetwork.from_string(G.sir_network(int(n), 0.3, 0.1)[0], "")
    return net, cs.var_query(net.variable_id("I"), 4.0, threshold=3, max_steps=60)


def _same(a, b, what):
    for k in a:
        x, y = a[k], b[k]
        if x.dtype == np.float64:
            x, y = x.view(np.uint64), y.view(np.uint64)
        assert np.array_equal(x, y), (what, k)


@pytest.mark.parametrize("name,n_runs", [
    ("race-1", [1, 1000, 70_000]), ("race-8", [63, 1025, 17_000, 140_000]), ("race-40", [1023, 8200, 70_000]),
    ("fischer-16", [5, 4097, 70_000]), ("fischer-100", [3000, 20_000]), ("sir-77", [1024, 5001, 33_000]),
    ("sir-300", [2050, 9000]), ("csma", [300, 5000]),
])
def test_chosen_launch_equals_widest(name, n_runs):
    net, q = _query(name)
    sim = cs.GpuSimulator(net)
    try:
        wide = min(64, 1 << (net.n_components - 1).bit_length())
        for n in n_runs:
            for per_run in (PER_RUN, PER_RUN + ("digest",)):
                print(f"[gpu launch] {name} runs={n} outputs={len(per_run)}", flush=True)
                a = sim.run(q, seed=4, n_runs=n, run_begin=2, per_run=per_run)
                b = sim.run(q, seed=4, n_runs=n, run_begin=2, lanes_per_run=wide, per_run=per_run)
                _same(a.per_run, b.per_run, (name, n))
                assert (a.hits, a.steps, a.transitions, a.truncated) == (b.hits, b.steps, b.transitions, b.truncated)
    finally:
        sim.close()


@pytest.mark.parametrize("n,n_runs", [(12, 40_000), (100, 9000), (100, 300), (400, 5000)])
def test_sampler_packing_does_not_change_results(n, n_runs, monkeypatch):
    net = cs.ParsedNetwork.from_string(G.sir_network(n, 0.15, 0.1, initial_infected=1)[0], "")
    q = cs.var_query(net.variable_id("I"), 5.0, threshold=max(2, n // 8))
    sim = cs.GpuSimulator(net)
    try:
        out = []
        for lanes in (None, str(min(64, 1 << (n - 1).bit_length()))):
            if lanes:
                monkeypatch.setenv("SMC_IS_LANES", lanes)
            s = cs.ImportanceSampler(sim, q, hidden=64)
            rng = np.random.default_rng(3)
            s.set_params(rng.normal(0.0, 0.1, s.get_params().shape).astype(np.float32))
            for use_mlp in (False, True):
                print(f"[gpu launch] sampler n={n} runs={n_runs} lanes={lanes} mlp={use_mlp}", flush=True)
                out.append(s.sample(seed=2, n_runs=n_runs, use_mlp=use_mlp).per_run)
            s.close()
        _same(out[0], out[2], (n, n_runs, "base law"))
        _same(out[1], out[3], (n, n_runs, "proposal"))
    finally:
        sim.close()
