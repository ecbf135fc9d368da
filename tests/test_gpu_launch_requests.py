"""Launch shapes that a caller names: what is honoured, what is refused, and
that results do not depend on it."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import cusmc_amd as cs
from cusmc_amd import _capi as A
from cusmc_amd import generators as G

import oracle

from _models import E_ADD, RawNetwork

pytestmark = pytest.mark.gpu

PER_RUN = ("flag", "value", "steps", "transitions", "time")


def _same(a, b, what):
    assert a.keys() == b.keys()
    for k in a:
        assert a[k].tobytes() == b[k].tobytes(), (what, k)


@pytest.mark.parametrize("waves", [1, 7, 1 << 20, 2**31 - 1])
def test_any_number_of_waves(waves):
    """From one wave to the largest number, many runs: the workgroups follow
    what a CU holds, the grid what the runs fill."""
    net = cs.ParsedNetwork.from_string(G.race_network(40)[0], "")
    q = cs.var_query(net.variable_id("count"), 3.0, threshold=2, max_steps=20)
    sim = cs.GpuSimulator(net)
    try:
        n = 30_000 if waves > 100 else 2000
        ref = sim.run(q, seed=4, n_runs=n, per_run=PER_RUN)
        for tables in (0, 1, 2):
            for lanes in (64, 8):
                print(f"[gpu requests] waves={waves} tables={tables} lanes={lanes}", flush=True)
                r = sim.run(q, seed=4, n_runs=n, lanes_per_run=lanes, waves=waves, tables=tables, per_run=PER_RUN)
                _same(r.per_run, ref.per_run, (waves, tables, lanes))
                assert r.waves <= max(8, -(-n // (64 // lanes)) + 8)
    finally:
        sim.close()


def _distinct(n_locs):
    """One component of n_locs locations that share no record: a ring with a
    rate of its own each, and constants of its own in every edge."""
    net = RawNetwork()
    v = net.var(0.0)
    first = net.component([dict(type=0, rate=net.lit(1.0 + l / 4096.0)) for l in range(n_locs)])
    for l in range(n_locs):
        net.edge(first + l, first + (l + 1) % n_locs, upds=[(v, net.expr(E_ADD, net.ref(v), net.lit(float(1 + l))))])
    return net.build()


# locations, and whether tables = 1 and tables = 2 are accepted: staged; within
# the counted bytes but not in LDS; the locations past them; the edges past them
@pytest.mark.parametrize("n_locs,one,two", [(500, True, True), (1200, True, True), (1900, False, True),
                                            (5000, False, False)])
def test_named_tables_are_staged_or_refused(n_locs, one, two):
    net = _distinct(n_locs)
    q = cs.var_query(0, 20.0, estimate=True)
    sim = cs.GpuSimulator(net)
    try:
        n = 500
        with_digest = PER_RUN + ("digest",)
        ref = sim.run(q, seed=2, n_runs=n, lanes_per_run=1, per_run=with_digest)
        for tables, accepted in ((1, one), (2, two)):
            print(f"[gpu requests] locations={n_locs} tables={tables}", flush=True)
            if accepted:
                r = sim.run(q, seed=2, n_runs=n, lanes_per_run=1, tables=tables, per_run=PER_RUN)
                _same(r.per_run, {k: ref.per_run[k] for k in PER_RUN}, (n_locs, tables))
            else:
                with pytest.raises(A.SmcError) as e:
                    sim.run(q, seed=2, n_runs=n, lanes_per_run=1, tables=tables, per_run=PER_RUN)
                assert e.value.code == A.SMC_E_LIMIT
            # digest runs take tables from anywhere
            r = sim.run(q, seed=2, n_runs=n, lanes_per_run=1, tables=tables, per_run=with_digest)
            _same(r.per_run, ref.per_run, (n_locs, tables, "digest"))
    finally:
        sim.close()


def test_autotuner_names_only_what_a_launch_does(monkeypatch):
    """Tables that do not fit in LDS are not a choice of the autotuner's."""
    monkeypatch.setenv("SMC_TUNE_CACHE", "off")
    for n_locs, staged in ((4, None), (1200, 0), (5000, 0)):
        net = _distinct(n_locs)
        sim = cs.GpuSimulator(net)
        try:
            print(f"[gpu requests] autotune locations={n_locs}", flush=True)
            best = sim.autotune(cs.var_query(0, 20.0, estimate=True), sample_runs=4096)
            assert best.tables in (0, 1) if staged is None else best.tables == staged
        finally:
            sim.close()


@pytest.mark.parametrize("n_comp,lanes,n_vars", [(16, 1, 116), (16, 16, 1746), (2, 1, 116), (40, 4, 450)])
def test_as_many_variables_as_a_packing_holds(n_comp, lanes, n_vars):
    """Variables of the packed runs up to the limit of 60,000 bytes: with the
    state words, and a digest run's locations, a wave takes more than 64 KB of
    LDS.  One variable more is refused."""
    def network(n):
        net = RawNetwork()
        vs = [net.var(float(k % 7)) for k in range(n)]
        for c in range(n_comp):
            first = net.component([dict(type=0, rate=net.lit(1.0 + c)), dict(type=0, rate=net.lit(2.0))])
            a, b = vs[(37 * c + 5) % n], vs[n - 1 - c % 2]
            net.edge(first, first + 1, upds=[(a, net.expr(E_ADD, net.ref(a), net.ref(b)))])
            net.edge(first + 1, first, upds=[(b, net.expr(E_ADD, net.ref(b), net.lit(1.0)))])
        return net.build()

    n = 300
    with_digest = PER_RUN + ("digest",)
    net = network(n_vars)
    q = cs.var_query(n_vars - 1, 3.0, estimate=True)
    _, want = oracle.run(net, q, seed=6, n_runs=n, threads=8, per_run=with_digest)
    sim = cs.GpuSimulator(net)
    try:
        for tables in (0, 1):
            print(f"[gpu requests] components={n_comp} lanes={lanes} variables={n_vars} tables={tables}", flush=True)
            r = sim.run(q, seed=6, n_runs=n, lanes_per_run=lanes, tables=tables, per_run=with_digest)
            _same(r.per_run, want, (n_comp, lanes, tables))
    finally:
        sim.close()
    more = network(n_vars + 2)
    sim = cs.GpuSimulator(more)
    try:
        with pytest.raises(A.SmcError) as e:
            sim.run(q, seed=6, n_runs=n, lanes_per_run=lanes)
        assert e.value.code == A.SMC_E_LIMIT
    finally:
        sim.close()


@pytest.mark.parametrize("n_vars,stays", [(145, 7), (147, 6)])
def test_waves_left_to_choose_are_resident(n_vars, stays):
    """A wave whose LDS, handed out in parts of 1280 bytes, fits a compute unit
    one time less than its bytes do: sixteen runs of 145 and of 147 variables
    take 18 and 19 parts of 128."""
    net = RawNetwork()
    vs = [net.var(0.0) for _ in range(n_vars)]
    for c in range(64):
        first = net.component([dict(type=0, rate=net.lit(1.0 + c))])
        net.edge(first, first, upds=[(vs[c], net.expr(E_ADD, net.ref(vs[c]), net.lit(1.0)))])
    net = net.build()
    q = cs.var_query(63, 3.0, estimate=True)
    n = 60_000
    sim = cs.GpuSimulator(net)
    try:
        print(f"[gpu requests] variables={n_vars}", flush=True)
        r = sim.run(q, seed=8, n_runs=n, lanes_per_run=4, tables=0, per_run=PER_RUN)
        assert r.waves == stays * torch.cuda.get_device_properties(0).multi_processor_count
        _same(r.per_run, sim.run(q, seed=8, n_runs=n, lanes_per_run=64, per_run=PER_RUN).per_run, n_vars)
    finally:
        sim.close()
