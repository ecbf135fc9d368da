"""Networks whose tables are larger than the narrow forms of an index hold.
Runs equal the canonical oracle's, bit for bit."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import cusmc_amd as cs
from cusmc_amd import _capi as A

import oracle

pytestmark = pytest.mark.gpu

LE, GE = 0, 2
LIT, VAR, ADD = 0, 1, 3
PER_RUN = ("flag", "value", "steps", "transitions", "digest", "time")

CONSTRAINT = np.dtype([(k, np.int32) for k in ("op", "uses_variable", "var", "lhs", "rhs")])
EXPR = np.dtype([(k, np.int32) for k in ("op", "a", "b", "c", "var", "reserved")] + [("value", np.float64)])
LOCATION = np.dtype([(k, np.int32) for k in ("type", "rate", "inv_first", "inv_count", "edge_first", "edge_count")])
EDGE = np.dtype([(k, np.int32) for k in ("src", "dst", "channel", "weight", "guard_first", "guard_count", "upd_first",
                                         "upd_count")])
UPDATE = np.dtype([(k, np.int32) for k in ("var", "expr")])


class ArrayNetwork:
    """A network given as the arrays of smc_network."""

    def __init__(self, *, var_init, first_loc, init_loc, locations, edges, constraints, updates, exprs):
        as_ = lambda a, t: np.ascontiguousarray(a, dtype=t)  # noqa: E731
        self._keep = [as_(np.zeros(len(var_init)), np.int32), as_(var_init, np.float64), as_(first_loc, np.int32),
                      as_(init_loc, np.int32), as_(locations, LOCATION), as_(edges, EDGE),
                      as_(constraints, CONSTRAINT), as_(updates, UPDATE), as_(exprs, EXPR)]
        k = self._keep
        ptr = [a.ctypes.data_as(t) for a, (_, t) in zip(k, A.Network._fields_[8:])]
        self.net = A.Network(len(init_loc), len(var_init), len(k[4]), len(k[5]), len(k[6]), len(k[7]), len(k[8]), 0, *ptr)
        self.net_ptr = C.pointer(self.net)


def _expr(items):
    """(op, a, b, var, value) rows."""
    out = np.zeros(len(items), EXPR)
    for i, (op, a, b, var, value) in enumerate(items):
        out[i] = (op, a, b, -1, var, 0, value)
    return out


def _runs_equal(net, q, n_runs, lanes, **launch):
    _, ro = oracle.run(net, q, seed=11, n_runs=n_runs, threads=8, per_run=PER_RUN)
    sim = cs.GpuSimulator(net)
    try:
        for S in lanes:
            print(f"[gpu large tables] lanes={S} {launch}", flush=True)
            r = sim.run(q, seed=11, n_runs=n_runs, lanes_per_run=S, per_run=PER_RUN, **launch)
            for k in PER_RUN:
                a, b = r.per_run[k], ro[k]
                if a.dtype == np.float64:
                    a, b = a.view(np.uint64), b.view(np.uint64)
                assert np.array_equal(a, b), (S, k)
    finally:
        sim.close()
    return ro


def test_guard_records_past_24_bits():
    """266 edges of 65,535 guards each, no two edges' alike: 17.4 million
    records.  The runs use the last six edges, of which one is enabled."""
    per_edge, fillers, filler_edges, tested = 65535, 5, 52, 6
    n_guarded = fillers * filler_edges + tested
    # expressions: 0 the variable w, 1 and 2 the updates of v, then per edge
    # the constant its second guard compares with
    ex = [(VAR, -1, -1, 1, 0.0), (LIT, -1, -1, 0, 1.0), (LIT, -1, -1, 0, 2.0)]
    consts = np.zeros(n_guarded, EXPR)
    consts["op"] = LIT
    enabled = n_guarded - tested + 3
    k = np.arange(n_guarded)
    consts["value"] = np.where(k == enabled, 0.0, -1.0 - k)  # v <= value, with v at 0
    exprs = np.concatenate([_expr(ex), consts])
    g = np.zeros((n_guarded, per_edge), CONSTRAINT)
    g["op"], g["uses_variable"], g["var"], g["lhs"], g["rhs"] = LE, 1, 0, -1, 0  # v <= w
    g["op"][:, 0], g["rhs"][:, 0] = GE, 3 + enabled                                # v >= 0
    g["rhs"][:, 1] = 3 + k
    locations, edges = [], []
    at = 0
    for l in range(fillers + 1):
        n = filler_edges if l < fillers else tested
        locations.append((0, -1, 0, 0, len(edges), n + 1))
        for _ in range(n):
            edges.append((l, fillers + 1, 0, -1, at * per_edge, per_edge, at % 2, 1))
            at += 1
        edges.append((l, l, 0, 4, 0, 0, 0, 0))  # unguarded, of weight below 0: never blocked, never picked
    locations.append((0, -1, 0, 0, len(edges), 0))
    net = ArrayNetwork(var_init=[0.0, 5.0], first_loc=[0, fillers + 2], init_loc=[fillers],
                       locations=np.array(locations, LOCATION), edges=np.array(edges, EDGE), constraints=g.ravel(),
                       updates=np.array([(0, 1), (0, 2)], UPDATE), exprs=exprs)
    ro = _runs_equal(net, cs.var_query(0, 50.0, estimate=True, max_steps=40), 24, [1])
    assert set(ro["value"]) == {2.0} and set(ro["transitions"]) == {1}
