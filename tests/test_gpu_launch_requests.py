"""Launch shapes that a caller names: what is honoured, what is refused, and
that results do not depend on it."""
from __future__ import annotations

import numpy as np
import pytest

import cusmc_amd as cs
from cusmc_amd import generators as G

pytestmark = pytest.mark.gpu

PER_RUN = ("flag", "value", "steps", "transitions", "time")


def _same(a, b, what):
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
