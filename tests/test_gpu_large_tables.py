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


def test_more_record_classes_than_a_state_word_holds_beside_a_base():
    """Two components of 131,100 locations, all different: variables keep their
    own indices and a state word holds the class alone."""
    n_comp, L, rates = 2, 131100, 256
    n = n_comp * L
    l = np.arange(n) % L
    c = np.arange(n) // L
    # expressions: 0 the first update, 1 the second, then rates, then guard bounds
    head = [(ADD, 2, 3, -1, 0.0), (ADD, 2, 4, -1, 0.0), (VAR, -1, -1, 0, 0.0), (LIT, -1, -1, 0, 1.0),
            (LIT, -1, -1, 0, -1.0)]
    bounds = -(-L // rates)
    ex = np.zeros(rates + n_comp * bounds, EXPR)
    ex["op"] = LIT
    ex["value"][:rates] = 0.5 + np.arange(rates) / 64.0
    ex["value"][rates:] = np.arange(n_comp * bounds) - 3.0
    locations = np.zeros(n, LOCATION)
    locations["rate"] = len(head) + l % rates
    locations["edge_first"], locations["edge_count"] = 2 * np.arange(n), 2
    edges = np.zeros(2 * n, EDGE)
    edges["src"] = np.repeat(np.arange(n), 2)
    edges["weight"] = -1
    edges["dst"][0::2] = c * L + (5 * l + 1) % L
    edges["dst"][1::2] = c * L + (l + 12345) % L
    edges["guard_first"][0::2], edges["guard_count"][0::2] = np.arange(n), 1   # v <= a bound of its own
    edges["upd_first"], edges["upd_count"] = np.tile([0, 1], n), 1
    g = np.zeros(n, CONSTRAINT)
    g["op"], g["uses_variable"], g["var"], g["lhs"] = LE, 1, 0, -1
    g["rhs"] = len(head) + rates + c * bounds + l // rates
    net = ArrayNetwork(var_init=[0.0], first_loc=[0, L, n], init_loc=[0, L + 7], locations=locations, edges=edges,
                       constraints=g, updates=np.array([(0, 0), (0, 1)], UPDATE), exprs=np.concatenate([_expr(head), ex]))
    ro = _runs_equal(net, cs.var_query(0, 30.0, estimate=True), 200, [1, 2])
    assert len(set(ro["value"])) > 3


@pytest.mark.parametrize("n_comp,length", [(3, 65), (7, 100), (40, 90)])
def test_chains_of_equal_locations(n_comp, length):
    """Instances of a chain of equal locations, each adding to one variable, the
    last link back to the first: classes by place."""
    n = n_comp * length
    k = np.arange(n) % length
    c = np.arange(n) // length
    ex = _expr([(ADD, 1, 2, -1, 0.0), (VAR, -1, -1, 0, 0.0), (LIT, -1, -1, 0, 1.0), (LIT, -1, -1, 0, 2.0)])
    locations = np.zeros(n, LOCATION)
    locations["rate"] = np.where(k == length - 1, 3, -1)
    locations["edge_first"], locations["edge_count"] = np.arange(n), 1
    edges = np.zeros(n, EDGE)
    edges["src"], edges["dst"] = np.arange(n), c * length + (k + 1) % length
    edges["weight"], edges["upd_first"], edges["upd_count"] = -1, 0, 1
    net = ArrayNetwork(var_init=[0.0], first_loc=np.arange(n_comp + 1) * length, init_loc=np.arange(n_comp) * length,
                       locations=locations, edges=edges, constraints=np.zeros(0, CONSTRAINT),
                       updates=np.array([(0, 0)], UPDATE), exprs=ex)
    P = 1 << (n_comp - 1).bit_length()
    for tables in (0, 1):
        ro = _runs_equal(net, cs.var_query(0, 120.0, estimate=True), 64, sorted({P, max(1, P // 8)}), tables=tables)
    assert ro["value"].min() > n_comp * length / 2
