"""The importance sampler's packings: several rows a wave and up to eight slots
a lane, forced and chosen by the number of rows, with exponential rates and
delay windows under a tilt per location, sampling and recording.  Everything
equals the oracle bit for bit.
"""
from __future__ import annotations

import numpy as np
import pytest

import cusmc_amd as cs
from cusmc_amd import generators as G

import oracle

from _models import receiver_goal

pytestmark = pytest.mark.gpu


def _sir(n):
    net = cs.ParsedNetwork.from_string(G.sir_network(n, 0.3, 0.1, initial_infected=2)[0], "")
    return net, lambda bound: cs.var_query(net.variable_id("I"), bound, threshold=max(3, n // 6))


def _fischer(n):
    net = cs.ParsedNetwork.from_string(G.fischer_network(n)[0], "P0.cs")
    return net, cs.reach_query


def _race(n):
    net = cs.ParsedNetwork.from_string(G.race_network(n)[0], "")
    return net, lambda bound: cs.var_query(net.variable_id("count"), bound, threshold=2 * n)


NETS = {"sir100": lambda: _sir(100), "sir250": lambda: _sir(250), "fischer32": lambda: _fischer(32),
        "fischer33": lambda: _fischer(33), "race40": lambda: _race(40)}


def _theta(net):
    return np.random.default_rng(5).uniform(-1.0, 1.0, net.net.n_locations).astype(np.float32)


def _sampler(sim, q, lanes, monkeypatch):
    if lanes:
        monkeypatch.setenv("SMC_IS_LANES", str(lanes))
    s = cs.ImportanceSampler(sim, q, hidden=64)
    monkeypatch.delenv("SMC_IS_LANES", raising=False)
    return s


# rows and the packings: None lets the number of rows choose, and reaches the
# narrowest of those named (two rows a wave from 1024 rows on, four from 2048)
@pytest.mark.parametrize("name,bound,n,lanes", [
    ("sir100", 8.0, 1100, (None, 64, 32)), ("sir100", 4.0, 4100, (None, 16)), ("sir250", 1.5, 1100, (None, 64, 32)),
    ("fischer32", 6.0, 8200, (None, 32, 8, 4)), ("fischer33", 4.0, 2100, (None, 64, 16, 8)),
    ("race40", 2.0, 4200, (None, 16, 8))])
def test_tilted_runs_at_every_packing(name, bound, n, lanes, monkeypatch):
    net, query = NETS[name]()
    q, theta = query(bound), _theta(net)
    sim = cs.GpuSimulator(net)
    try:
        o = oracle.is_run(net, q, seed=9, n_runs=n, theta=theta, threads=0)
        for S in lanes:
            s = _sampler(sim, q, S, monkeypatch)
            for lock in (True, False):
                print(f"[gpu is packings] {name} rows={n} lanes={S} lockstep={lock}", flush=True)
                r = s.sample(seed=9, n_runs=n, theta=theta, lockstep=lock)
                for k in ("digest", "flag", "log2lr", "steps", "transitions", "time"):
                    assert r.per_run[k].tobytes() == o[k].tobytes(), (name, S, lock, k)
            s.close()
    finally:
        sim.close()


def _var_scale(net, q):
    n = net.net
    most = max([float(n.n_components)] + [abs(n.var_init[v]) for v in range(n.n_vars) if n.var_kind[v] != 1])
    return np.array([1.0 / q.time_bound if n.var_kind[v] == 1 else 1.0 / max(1.0, most) for v in range(n.n_vars)],
                    np.float32)


@pytest.mark.parametrize("name,bound,lanes", [
    ("sir100", 12.0, (64, 32, 16)), ("sir250", 4.0, (64, 32)), ("fischer33", 8.0, (64, 32, 16, 8)),
    ("fischer32", 8.0, (32, 16, 4)), ("race40", 3.0, (64, 16, 8))])
def test_recorded_pairs_at_every_packing(name, bound, lanes, monkeypatch):
    """37 replayed runs: several rows a wave, the last wave not full."""
    net, query = NETS[name]()
    q, theta = query(bound), _theta(net)
    runs = np.arange(300, 337, dtype=np.uint64)
    sim = cs.GpuSimulator(net)
    try:
        want = None
        for S in lanes:
            s = _sampler(sim, q, S, monkeypatch)
            print(f"[gpu is packings] record {name} lanes={S}", flush=True)
            got = s.record(runs, seed=4, theta=theta, early_stop=True)
            if want is None:
                per_run = [oracle.is_record(net, q, seed=4, run=int(r), theta=theta, var_scale=_var_scale(net, q),
                                            fpad=s.features_padded, lpad=s.locations_padded, early_stop=True)
                           for r in runs]
                # slots are numbered macro-step-major, run-minor
                order = [(k, p) for k in range(max(len(p[0]) for p in per_run)) for p in per_run if k < len(p[0])]
                want = [np.array([p[part][k] for k, p in order]) for part in range(3)]
            for a, b, part in zip(got, want, "XAB"):
                assert np.array_equal(a, b), (name, S, part)
            s.close()
    finally:
        sim.close()


@pytest.mark.parametrize("live,clock_rate", [(None, False), (1.0, False), (0.5, True)])
def test_goal_entered_by_a_receiver_in_lock_step(live, clock_rate):
    """A goal that broadcast receivers enter at the end of one launch counts by
    the race step of the next: with and without lock step the same hits, the
    plain kernel's without a tilt and the oracle's with one."""
    net = cs.ParsedNetwork.from_string(receiver_goal(live, clock_rate), "")
    q = cs.reach_query(3.0)
    n = 3000
    sim = cs.GpuSimulator(net)
    s = cs.ImportanceSampler(sim, q, hidden=64)
    try:
        plain = sim.run(q, seed=2, n_runs=n, per_run=("flag", "digest", "time"))
        assert 0 < plain.hits < n
        theta = _theta(net)
        tilted = oracle.is_run(net, q, seed=2, n_runs=n, theta=theta, threads=8)
        for lock in (False, True):
            print(f"[gpu is packings] receiver goal live={live} lockstep={lock}", flush=True)
            r = s.sample(seed=2, n_runs=n, lockstep=lock)
            for k in ("flag", "digest", "time"):
                assert r.per_run[k].tobytes() == plain.per_run[k].tobytes(), (lock, k)
            r = s.sample(seed=2, n_runs=n, theta=theta, lockstep=lock)
            for k in ("flag", "digest", "log2lr", "time"):
                assert r.per_run[k].tobytes() == tilted[k].tobytes(), (lock, k, "tilted")
    finally:
        s.close()
        sim.close()
