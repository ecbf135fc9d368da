"""Importance sampling on networks whose locations nearly fill the advance
kernel's LDS (12 bytes of tilts each): accepted up to the same size whatever the
packing, with clock bounds (delay windows) or without.  Runs under a tilt per
location and recorded pairs equal the oracle's bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

import cusmc_amd as cs
from cusmc_amd import _capi as A

import oracle

from test_gpu_large_tables import ADD, CONSTRAINT, EDGE, LE, LIT, LOCATION, UPDATE, VAR, ArrayNetwork, _expr

pytestmark = pytest.mark.gpu


def _network(n_comp, per, bounded):
    """Instances of a ring of `per` locations, every third one under a bound of
    a shared clock, which some edges reset; every edge counts."""
    n = n_comp * per
    k = np.arange(n) % per
    head = [(ADD, 2, 3, -1, 0.0), (LIT, -1, -1, 0, 0.0), (VAR, -1, -1, 0, 0.0), (LIT, -1, -1, 0, 1.0)]
    ex = [(LIT, -1, -1, 0, 0.05 + j / 64.0) for j in range(per)] + [(LIT, -1, -1, 0, 40.0 + j) for j in range(per)]
    locations = np.zeros(n, LOCATION)
    locations["rate"] = len(head) + k
    locations["edge_first"], locations["edge_count"] = np.arange(n), 1
    edges = np.zeros(n, EDGE)
    edges["src"], edges["dst"] = np.arange(n), np.arange(n) - k + (k + 1) % per
    edges["weight"], edges["upd_count"] = -1, np.where(k % 5 == 0, 2, 1)
    constraints = np.zeros(per, CONSTRAINT)
    constraints["op"], constraints["uses_variable"], constraints["var"], constraints["lhs"] = LE, 1, 1, -1
    constraints["rhs"] = len(head) + per + np.arange(per)
    if bounded:
        locations["inv_first"], locations["inv_count"] = k, k % 3 == 1
    net = ArrayNetwork(var_init=[0.0, 0.0], first_loc=np.arange(n_comp + 1) * per, init_loc=np.arange(n_comp) * per,
                       locations=locations, edges=edges, constraints=constraints,
                       updates=np.array([(0, 0), (1, 1)], UPDATE), exprs=_expr(head + ex))
    net._keep[0][1] = 1  # variable 1 is a clock
    return net


def _theta(net):
    return np.random.default_rng(3).uniform(-1.0, 1.0, net.net.n_locations).astype(np.float32)


# lanes: the packing asked for (SMC_IS_LANES), or the sampler's
@pytest.mark.parametrize("n_comp,per,bounded,lanes", [
    (512, 25, True, None), (300, 43, True, None), (512, 25, False, None), (128, 99, True, "16"), (256, 50, True, "32"),
    (64, 180, True, "8"), (16, 640, True, None)])
def test_tilt_per_location_at_the_limit(n_comp, per, bounded, lanes, monkeypatch):
    net = _network(n_comp, per, bounded)
    q = cs.var_query(0, 4.0, threshold=200, max_steps=60)
    if lanes:
        monkeypatch.setenv("SMC_IS_LANES", lanes)
    sim = cs.GpuSimulator(net)
    s = cs.ImportanceSampler(sim, q, hidden=64)
    try:
        n, theta = 150, _theta(net)
        o = oracle.is_run(net, q, seed=5, n_runs=n, theta=theta, threads=8)
        for lock in (False, True):
            print(f"[gpu is large] {n_comp}x{per} bounded={bounded} lanes={lanes} lockstep={lock}", flush=True)
            r = s.sample(seed=5, n_runs=n, theta=theta, lockstep=lock)
            for k in ("digest", "flag", "log2lr", "steps", "time"):
                assert r.per_run[k].tobytes() == o[k].tobytes(), (n_comp, lanes, lock, k)
    finally:
        s.close()
        sim.close()


def test_recorded_pairs_at_the_limit():
    net = _network(512, 24, True)
    q = cs.var_query(0, 1.0, threshold=100, max_steps=12)
    sim = cs.GpuSimulator(net)
    s = cs.ImportanceSampler(sim, q, hidden=64)
    try:
        theta = _theta(net)
        runs = np.arange(20, 25, dtype=np.uint64)
        print("[gpu is large] record", flush=True)
        X, Aa, B = s.record(runs, seed=9, theta=theta, cap=256)
        scale = np.array([1.0 / 512, 1.0 / q.time_bound], np.float32)
        per_run = [oracle.is_record(net, q, seed=9, run=int(r), theta=theta, var_scale=scale, fpad=s.features_padded,
                                    lpad=s.locations_padded, cap=64) for r in runs]
        order = [(k, p) for k in range(max(len(p[0]) for p in per_run)) for p in per_run if k < len(p[0])]
        assert len(X) == len(order)
        for got, part in ((X, 0), (Aa, 1), (B, 2)):
            assert np.array_equal(got, np.array([p[part][k] for k, p in order])), part
    finally:
        s.close()
        sim.close()


def test_refused_past_the_limit():
    net = _network(512, 27, True)
    sim = cs.GpuSimulator(net)
    try:
        with pytest.raises(A.SmcError) as e:
            cs.ImportanceSampler(sim, cs.var_query(0, 4.0, threshold=20), hidden=64)
        assert e.value.code == A.SMC_E_LIMIT
    finally:
        sim.close()
