"""Runs are handed out exactly once, whatever their number, the waves and how
long they take: waves begin with runs of their own, then take more from the
launch's queue, short runs many at a time.  Per-run outputs equal the oracle's
bit for bit; a batch's totals do on every round, with eager work between.
"""
from __future__ import annotations

import numpy as np
import pytest

import cusmc_amd as cs
from cusmc_amd import generators as G

import oracle

from _models import E_ADD, RawNetwork, single_exponential

pytestmark = pytest.mark.gpu

PER_RUN = ("flag", "value", "steps", "transitions", "time")


def _dead():
    net = RawNetwork()
    net.var(3.0)
    net.component([dict(type=0)])
    return net.build(), cs.var_query(0, 2.0, estimate=True)


def _chain(length, n_comp):
    """Components that take `length` steps each and then stand still."""
    net = RawNetwork()
    v = net.var(0.0)
    for c in range(n_comp):
        first = net.component([dict(type=0, rate=net.lit(1.0 + c))] * (length + 1))
        for k in range(length):
            net.edge(first + k, first + k + 1, upds=[(v, net.expr(E_ADD, net.ref(v), net.lit(1.0)))])
    return net.build(), cs.var_query(0, 1e9, estimate=True)


def _one_step():
    return cs.ParsedNetwork.from_string(single_exponential(0.5), ""), cs.reach_query(2.0)


def _race(n):
    net = cs.ParsedNetwork.from_string(G.race_network(n)[0], "")
    return net, cs.var_query(net.variable_id("count"), 1.0, threshold=2)


MODELS = {"dead": _dead, "one step": _one_step, "chain5x1": lambda: _chain(5, 1), "chain2x5": lambda: _chain(2, 5),
          "chain30x1": lambda: _chain(30, 1), "race8": lambda: _race(8)}


@pytest.mark.parametrize("name,numbers", [
    ("dead", (1, 63, 64, 65, 262_145, 1_500_001)), ("one step", (1, 64, 1025, 65_537, 262_144, 262_145, 700_001)),
    ("chain5x1", (1023, 300_000)), ("chain2x5", (8191, 70_000)), ("chain30x1", (20_000, 400_003)),
    ("race8", (33, 8193, 60_001))])
def test_every_run_once(name, numbers):
    net, q = MODELS[name]()
    sim = cs.GpuSimulator(net)
    try:
        wide = min(64, 1 << (net.net.n_components - 1).bit_length())
        n = max(numbers)
        _, want = oracle.run(net, q, seed=8, run_begin=3, n_runs=n, threads=8, per_run=PER_RUN)
        for n in numbers:
            for launch in (dict(), dict(lanes_per_run=wide, waves=7), dict(lanes_per_run=1, tables=1), dict(waves=5000)):
                if launch.get("waves") == 7 and n > 70_000:
                    continue  # (seven waves take seconds)
                print(f"[gpu queue] {name} runs={n} {launch}", flush=True)
                r = sim.run(q, seed=8, run_begin=3, n_runs=n, per_run=PER_RUN, **launch)
                for k in PER_RUN:
                    assert r.per_run[k].tobytes() == want[k][:n].tobytes(), (name, n, launch, k)
                assert (r.steps, r.transitions) == (want["steps"][:n].sum(), want["transitions"][:n].sum())
    finally:
        sim.close()


@pytest.mark.parametrize("sizes", [(1,), (1, 64, 5000), (100_000, 3, 20_000, 63)])
def test_batch_rounds(sizes):
    items, nets = [], []
    for k, name in enumerate(sorted(MODELS)):
        net, q = MODELS[name]()
        nets.append((net, q))
        items.append((cs.GpuSimulator(net), q, 50 + k, sizes[k % len(sizes)]))
    batch = cs.Batch(items)
    try:
        for rnd in range(4):
            print(f"[gpu queue] batch sizes={sizes} round={rnd}", flush=True)
            res, _ = batch.run(1)
            items[0][0].run(items[0][1], seed=1, n_runs=100)  # eager work between the rounds
            for (net, q), (_, _, seed, n), r in zip(nets, items, res):
                o, _ = oracle.run(net, q, seed=seed, run_begin=rnd * n, n_runs=n, threads=8)
                assert (r.hits, r.steps, r.transitions) == (o.hits, o.steps, o.transitions), (rnd, n)
    finally:
        batch.close()
        for sim, *_ in items:
            sim.close()
