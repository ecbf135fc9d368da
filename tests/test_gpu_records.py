"""Record classes and the race step's paths: networks made of instances of a
few templates, with private variables in every place a record names one
(rates, invariant bounds, guards, weights, updates), constant comparisons at
the edges of the `==` tolerance, one and several invariants and blocking
conjuncts, and receive edges of every kind (one channel unguarded, guarded,
two channels, non-commuting, beyond the 32nd edge, weights summing past 2^31).

Every run's trajectory digest equals the canonical oracle's, at each launch
shape: there is no tolerance.
"""
from __future__ import annotations

import numpy as np
import pytest

import cusmc_amd as cs

import oracle

from _models import E_ADD, E_MUL, E_SUB, RawNetwork

pytestmark = pytest.mark.gpu

LE, LT, GE, GT, EQ, NE = range(6)
PER_RUN = ("flag", "value", "steps", "transitions", "digest", "time")


def _template(rng, clock_rate):
    """Choices shared by the instances of one template."""
    return dict(seed=int(rng.integers(1 << 30)), clock_rate=clock_rate, n_locs=int(rng.integers(3, 6)))


def _instance(net, tpl, g, x_shared):
    """One component: private integer p, k and clock x, and edges over them
    and the shared variables g.  The template's own generator draws the
    structure, so instances differ in their private variables only."""
    rng = np.random.default_rng(tpl["seed"])
    p, k = net.var(0.0), net.var(1.0)
    x = net.var(0.0, clock=True)
    lit, ref, ex = net.lit, net.ref, net.expr
    locs = []
    for _ in range(tpl["n_locs"]):
        kind = rng.integers(0, 7)
        if kind == 0:
            locs.append(dict(type=0, rate=lit(float(rng.choice([0.0, 0.5, 2.0])))))
        elif kind == 1:
            locs.append(dict(type=0, rate=ex(E_ADD, lit(0.5), ex(E_MUL, lit(0.25), ref(k)))))
        elif kind == 2:
            locs.append(dict(type=0, rate=ex(E_ADD, lit(0.5), ref(g[0]))))
        elif kind == 3:
            locs.append(dict(type=0, invs=[(int(rng.choice([LE, LT])), x, lit(float(rng.integers(0, 3))))]))
        elif kind == 4:
            locs.append(dict(type=0, invs=[(LE, x, ex(E_ADD, ref(k), lit(1.0))), (LT, x_shared, lit(4.0))]))
        elif kind == 5:
            locs.append(dict(type=3))  # urgent
        else:
            rate = ex(E_ADD, lit(0.5), ref(x)) if tpl["clock_rate"] else lit(1.5)
            locs.append(dict(type=0, rate=rate, invs=[(LE, x, lit(1.0))]))
    first = net.component(locs)

    def guard():
        op = int(rng.choice([LE, LT, GE, GT, EQ]))
        what = rng.integers(0, 6)
        if what == 0:
            return (op, p, lit(float(rng.integers(0, 4))))
        if what == 1:  # within and just past the tolerance of ==
            return (op, g[1], lit(float(rng.choice([0.0, 1e-5, 2e-5, -1e-5, 5e-6]))))
        if what == 2:
            return (int(rng.choice([LE, GE, GT])), x, lit(float(rng.choice([0.0, 0.5, 1.0]))))
        if what == 3:
            return (op, g[0], ref(p))
        if what == 4:
            return (LE, x_shared, ex(E_ADD, lit(1.0), ref(k)))
        return (NE, p, lit(7.0))

    def update(commuting):
        what = rng.integers(0, 5)
        if commuting or what == 0:
            return (g[0], ex(E_ADD, ref(g[0]), lit(1.0))) if rng.random() < 0.5 else \
                (g[0], ex(E_SUB, ref(g[0]), lit(1.0)))
        if what == 1:
            return (g[1], ex(E_ADD, ref(g[1]), lit(float(rng.choice([5e-6, -5e-6, 1e-5])))))
        if what == 2:
            return (x, lit(float(rng.choice([0.0, 0.25]))))
        if what == 3:
            return (p, ex(E_ADD, ref(p), ref(k)))
        return (k, ex(E_SUB, lit(2.0), ref(k)))

    n = tpl["n_locs"]
    for l in range(n):
        for _ in range(int(rng.integers(1, 4))):
            gs = [guard() for _ in range(int(rng.choice([0, 0, 1, 1, 2])))]
            ups = [update(False) for _ in range(int(rng.integers(0, 3)))]
            w = -1 if rng.random() < 0.5 else (lit(float(rng.integers(0, 5))) if rng.random() < 0.7 else ref(k))
            net.edge(first + l, first + int(rng.integers(0, n)), channel=int(rng.choice([0, 0, 1, 2])), weight=w,
                     guards=gs, upds=ups)
        kind = rng.integers(0, 8)
        dst = lambda: first + int(rng.integers(0, n))  # noqa: E731
        if kind == 0:    # one channel, unguarded, two edges
            for wt in (1.0, float(rng.choice([0.0, 9.0]))):
                net.edge(first + l, dst(), channel=-1, weight=lit(wt), upds=[update(True)])
        elif kind == 1:  # three edges
            for wt in (2.0, 0.0, 3.0):
                net.edge(first + l, dst(), channel=-2, weight=lit(wt))
        elif kind == 2:  # guarded
            net.edge(first + l, dst(), channel=-1, guards=[guard()], upds=[update(True)])
            net.edge(first + l, dst(), channel=-1, weight=lit(3.0))
        elif kind == 3:  # two channels
            net.edge(first + l, dst(), channel=-1, upds=[update(True)])
            net.edge(first + l, dst(), channel=-2)
        elif kind == 4:  # updates that read each other
            net.edge(first + l, dst(), channel=-1, upds=[(g[0], ex(E_ADD, ex(E_MUL, ref(g[0]), lit(0.5)), ref(k)))])
        elif kind == 5:  # receive edges past the 32nd of the list
            for _ in range(34):
                net.edge(first + l, first + l, channel=3, guards=[(GT, p, lit(1e9))])
            net.edge(first + l, dst(), channel=-2, upds=[update(True)])
        elif kind == 6:  # weights summing past 2^31
            for _ in range(2):
                net.edge(first + l, dst(), channel=-1, weight=lit(2147483647.0))


def _network(seed, n_comp, clock_rate):
    rng = np.random.default_rng(seed)
    net = RawNetwork()
    g = [net.var(0.0), net.var(0.0)]
    x_shared = net.var(0.0, clock=True)
    tpls = [_template(rng, clock_rate and t == 0) for t in range(3)]
    for c in range(n_comp):
        _instance(net, tpls[int(rng.integers(0, 3))], g, x_shared)
    return net.build()


@pytest.mark.parametrize("n_comp,clock_rate", [(1, False), (3, False), (6, True), (17, False), (70, False)])
def test_template_networks_bit_exact_vs_oracle(n_comp, clock_rate):
    for seed in range(6):
        net = _network(1000 * n_comp + seed, n_comp, clock_rate)
        q = cs.var_query(0, 4.0, is_max=seed % 2 == 0, estimate=True, max_steps=400)
        n_runs = 96
        _, ro = oracle.run(net, q, seed=seed, n_runs=n_runs, run_begin=5, threads=8, per_run=PER_RUN)
        sim = cs.GpuSimulator(net)
        try:
            P = 1 << (n_comp - 1).bit_length()
            lanes = sorted({min(P, 64), max(1, P // 16), max(1, P // 4)})
            for S in lanes:
                for occ, tab in ((0, 0), (3, 1)):
                    print(f"[gpu records] n={n_comp} seed={seed} lanes={S} occupancy={occ} tables={tab}", flush=True)
                    r = sim.run(q, seed=seed, n_runs=n_runs, run_begin=5, lanes_per_run=S, occupancy=occ, tables=tab,
                                per_run=PER_RUN)
                    for k in PER_RUN:
                        a, b = r.per_run[k], ro[k]
                        if a.dtype == np.float64:
                            a, b = a.view(np.uint64), b.view(np.uint64)
                        assert np.array_equal(a, b), (n_comp, seed, S, occ, tab, k)
        finally:
            sim.close()


@pytest.mark.parametrize("edges", [
    [(1, 2147483647)] * 2, [(1, 2147483647), (1, 1), (1, 2147483647)], [(1, 2147483647), (2, 1), (1, 2147483647)],
    [(1, 2147483647)] * 32, [(1, 3), (2, 2147483647)] * 16, [(1, 2147483647)] * 33])
@pytest.mark.parametrize("guarded", [False, True])
def test_heavy_receivers_bit_exact_vs_oracle(edges, guarded):
    """Weights that sum past 31 and 32 bits, on one channel and on two, with as
    many edges as are tested together and one more."""
    net = RawNetwork()
    v = [net.var(0.0) for _ in range(4)]
    up = lambda k: [(v[k], net.expr(E_ADD, net.ref(v[k]), net.lit(1.0)))]  # noqa: E731
    first = net.component([dict(type=0, rate=net.lit(2.0))])
    for channel in (1, 2):
        net.edge(first, first, channel=channel)
    for c in range(20):
        first = net.component([dict(type=0), dict(type=0)])
        for l in range(2):
            for k, (channel, weight) in enumerate(edges):
                net.edge(first + l, first + (k + l) % 2, channel=-channel, weight=net.lit(float(weight)), upds=up(k % 4),
                         guards=[(LE, v[0], net.lit(150.0))] if guarded and k == 1 else [])
    net = net.build()
    q = cs.var_query(1, 100.0, estimate=True, max_steps=100)
    _, ro = oracle.run(net, q, seed=3, n_runs=200, threads=8, per_run=PER_RUN)
    sim = cs.GpuSimulator(net)
    try:
        for S in (2, 8, 32):
            print(f"[gpu records] edges={len(edges)} guarded={guarded} lanes={S}", flush=True)
            r = sim.run(q, seed=3, n_runs=200, lanes_per_run=S, per_run=PER_RUN)
            for k in PER_RUN:
                assert np.array_equal(r.per_run[k].view(np.uint8), ro[k].view(np.uint8)), (S, k)
    finally:
        sim.close()
