"""Delay windows without an end: invariants whose constant bound is infinite
or the largest double, or whose clock was set to minus infinity.  A component
under one still draws a uniform delay, from [0, largest double], so its event
crosses every time bound; runs in which nothing else races end with it.

Trajectory digests, times and FP64 likelihood ratios equal the canonical
oracle's at one, two and several slots per lane: there is no tolerance.
"""
from __future__ import annotations

import math

import numpy as np
import pytest

import cusmc_amd as cs

import oracle

from _models import E_ADD, E_DIV, E_MUL, E_SUB, RawNetwork

pytestmark = pytest.mark.gpu

LE, LT = 0, 1
PER_RUN = ("flag", "value", "steps", "transitions", "digest", "time")
BOUNDS = [math.inf, 1.7976931348623157e308, math.inf, 2.0, math.inf]


def _network(n_comp, live):
    """Component c: l0 under x <= BOUNDS[c] (strict for odd c) -> l1, a race at
    rate 1 that sets the clock to minus infinity -> l2 under a finite bound,
    which that leaves without an end.  `live`: one more component that races
    on, so that runs go through all three."""
    net = RawNetwork()
    g = net.var(0.0)
    for c in range(n_comp):
        x = net.var(0.0, clock=True)
        first = net.component([
            dict(type=0, invs=[(LT if c % 2 else LE, x, net.lit(BOUNDS[c % len(BOUNDS)]))]),
            dict(type=0, rate=net.lit(1.0)),
            dict(type=0, invs=[(LE, x, net.lit(3.0))])], init=c % 2)
        inc = [(g, net.expr(E_ADD, net.ref(g), net.lit(1.0)))]
        net.edge(first, first + 1, upds=inc)
        minus_inf = net.expr(E_DIV, net.lit(-1.0), net.lit(0.0)) if c % 3 == 1 else net.lit(-math.inf)
        net.edge(first + 1, first + 2, upds=inc + [(x, minus_inf)])
        net.edge(first + 2, first, upds=inc)
    if live:
        first = net.component([dict(type=0, rate=net.lit(2.0))])
        net.edge(first, first, upds=[(g, net.expr(E_ADD, net.ref(g), net.lit(1.0)))])
    return net.build()


def _equal(a, b, what):
    if a.dtype == np.float64:
        a, b = a.view(np.uint64), b.view(np.uint64)
    assert np.array_equal(a, b), what


@pytest.mark.parametrize("n_comp,live", [(1, False), (2, True), (5, False), (12, True), (40, False)])
def test_windows_without_an_end_match_oracle(n_comp, live):
    net = _network(n_comp, live)
    q = cs.var_query(0, 6.0, threshold=3, max_steps=200)
    n_runs = 200
    _, ro = oracle.run(net, q, seed=3, n_runs=n_runs, threads=8, per_run=PER_RUN)
    # without a racer that goes on, some run's last event comes out of such a window
    assert (ro["time"].max() > 1e300) == (not live)
    sim = cs.GpuSimulator(net)
    try:
        P = 1 << (n_comp + live - 1).bit_length()
        for S in sorted({min(P, 64), max(1, P // 2), max(1, P // 4), max(1, P // 16)}):
            for tab in (0, 1):
                print(f"[gpu windows] n={n_comp} live={live} lanes={S} tables={tab}", flush=True)
                r = sim.run(q, seed=3, n_runs=n_runs, lanes_per_run=S, tables=tab, per_run=PER_RUN)
                for k in PER_RUN:
                    _equal(r.per_run[k], ro[k], (n_comp, S, tab, k))
        theta = np.random.default_rng(1).uniform(-1.0, 1.0, net.net.n_locations).astype(np.float32)
        s = cs.ImportanceSampler(sim, q, hidden=64)
        try:
            o = oracle.is_run(net, q, seed=3, n_runs=n_runs, theta=theta, early_stop=False, threads=8)
            for lock in (False, True):
                print(f"[gpu windows] sampler n={n_comp} lockstep={lock}", flush=True)
                r = s.sample(seed=3, n_runs=n_runs, theta=theta, lockstep=lock)
                for k in ("digest", "flag", "log2lr", "steps", "time"):
                    _equal(r.per_run[k], o[k], (n_comp, "sampler", lock, k))
        finally:
            s.close()
    finally:
        sim.close()


@pytest.mark.parametrize("n_comp", [1, 2, 5, 40])
def test_clocks_set_from_growing_variables_match_oracle(n_comp):
    """A clock set to minus a variable that squares itself, which reaches
    infinity, under a finite bound; the other components' to a counter's value."""
    net = RawNetwork()
    g = net.var(0.0)
    for c in range(n_comp):
        x, v = net.var(0.0, clock=True), net.var(2.0)
        first = net.component([dict(type=0, invs=[(LE, x, net.lit(3.0))])])
        grow = net.expr(E_MUL, net.ref(v), net.ref(v)) if c % 2 == 0 else net.expr(E_ADD, net.ref(v), net.lit(0.25))
        net.edge(first, first, upds=[(g, net.expr(E_ADD, net.ref(g), net.lit(1.0))), (v, grow),
                                     (x, net.expr(E_SUB, net.lit(0.0), net.ref(v)))])
    net = net.build()
    q = cs.var_query(0, 60.0, estimate=True, max_steps=60 * n_comp)
    n_runs = 200
    _, ro = oracle.run(net, q, seed=3, n_runs=n_runs, threads=8, per_run=PER_RUN)
    sim = cs.GpuSimulator(net)
    try:
        P = 1 << (n_comp - 1).bit_length()
        for S in sorted({min(P, 64), max(1, P // 2), max(1, P // 4), max(1, P // 16)}):
            print(f"[gpu windows] growing n={n_comp} lanes={S}", flush=True)
            r = sim.run(q, seed=3, n_runs=n_runs, lanes_per_run=S, per_run=PER_RUN)
            for k in PER_RUN:
                _equal(r.per_run[k], ro[k], (n_comp, S, k))
    finally:
        sim.close()
