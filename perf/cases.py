"""The measured work of this framework: model checking calls of every size a
user makes, through the public entry points of `cusmc_amd`.

A case names a kind of call and its sizes:

  run    one GpuSimulator.run(): `n_runs` simulations of one query, reduced on
         the GPU.  `tuned`: the program autotuned the model beforehand (long
         studies do); without it the call runs as the `cusmc` command line
         runs, with the launch left to the library.  `per_run`: which per-run
         outputs the program asks for ("", "value" or "all", which includes
         the trajectory digests of a parity check).
  batch  one round of a Batch of `n_sir` epidemics and `n_fischer` protocol
         instances of uneven width.
  sample one ImportanceSampler.sample() under the MLP proposal.
  mlp    one ImportanceSampler.mlp_eval(): the proposal network forward and
         its parameter gradient.
  learn  a rare-event study from nothing: create the sampler, train it by
         cross-entropy, estimate to a relative width.

Networks come from cusmc_amd.generators and from the UPPAAL fixtures of the
test-suite; the Philox seed of a call comes from the case's seed.
"""
from __future__ import annotations

import gzip
import math
from pathlib import Path

import numpy as np

import cusmc_amd as cs
from cusmc_amd import generators as G

MODELS = Path("tests") / "golden" / "models"

# UPPAAL fixtures: file, location query, query variable, components, and the
# race steps and lane-operations of one run at the time bound given (averages
# of the sequential reference simulation: one lane-operation per 64-bit
# add, multiply, compare or select, 100 per random block).
FIXTURES = {
    "weight": ("UppaalWeightTest.xml", "Template.l3", None, 60.0, 24.3, 3.4e3),
    "fischer10": ("fischer_10_29.xml", "P0.cs", None, 300.0, 228.7, 1.03e5),
    "fischermulti": ("fischermulti.xml", "", 0, 100.0, 146.2, 4.7e4),
    "covid32": ("agentBaseCovid_32_1.xml", "", "inf", 100.0, 124.2, 4.7e4),
    "covid100": ("large/agentBaseCovid_100_1.0.xml.gz", "", "inf", 100.0, 365.8, 3.4e5),
    "covid350": ("large/agentBaseCovid_350.xml.gz", "", "inf", 100.0, 1288.8, 3.7e6),
    "aloha25": ("aloha_25.xml", "", "nt", 100.0, 28338.6, 5.2e7),
    "csma100": ("large/CSMA_100.xml.gz", "Process0.SUCCESS", None, 100.0, 155.2, 1.02e6),
    "fischer100": ("large/fischer_100_29.xml.gz", "P0.cs", None, 100.0, 263.2, 7.9e5),
}

PER_RUN = {"": (), "value": ("flag", "value"),
           "all": ("flag", "value", "steps", "transitions", "digest", "time")}
BYTES_PER_RUN = {"": 17, "value": 17, "all": 33}

# no drawn case costs more lane-operations than this (the widest listed one)
MOST_OPS = 1.6e11


def listed() -> list[dict]:
    return [
        # the smallest call: a one-component model, a thousand runs; what a
        # script that sweeps a parameter pays per point
        dict(name="weight_1k", kind="run", model="weight", n=1, n_runs=1000, tuned=False, per_run=""),
        # eight racing components, ten thousand runs: a quick look at a small
        # model; few runs for the width of the GPU
        dict(name="race8_10k", kind="run", model="race", n=8, n_runs=10_000, tuned=False, per_run=""),
        # Fischer mutual exclusion with 32 processes, a million runs: the
        # repository's headline benchmark
        dict(name="fischer32_1m", kind="run", model="fischer", n=32, n_runs=1_000_000, tuned=True, per_run=""),
        # slotted aloha, 25 stations: broadcasts, clock bounds, and runs of
        # some thirty thousand steps
        dict(name="aloha25_1k", kind="run", model="aloha25", n=25, n_runs=1024, tuned=False, per_run="value"),
        # CSMA/CA with 100 processes and 900 variables at the command line's
        # default number of runs
        dict(name="csma100_16k", kind="run", model="csma100", n=100, n_runs=16_384, tuned=False, per_run=""),
        # the agent-based covid model at the command line's defaults, asking
        # for each run's peak
        dict(name="covid350_16k", kind="run", model="covid350", n=350, n_runs=16_384, tuned=False, per_run="value"),
        # agent SIR with 350 agents: broadcast waves over hundreds of receivers
        dict(name="sir350_200k", kind="run", model="sir", n=350, n_runs=200_000, tuned=True, per_run=""),
        # an odd-sized epidemic with every per-run output: a parity check
        dict(name="sir77_all", kind="run", model="sir", n=77, n_runs=5001, tuned=False, per_run="all"),
        # a parameter study: 48 uneven instances in one captured round
        dict(name="batch_48", kind="batch", n_sir=24, n_fischer=24, n_runs=2000),
        # fifty thousand lock-step runs under a proposal network
        dict(name="sample_50k", kind="sample", n=100, n_runs=50_000),
        # the proposal network alone: tilts and parameter gradient of a batch
        # of states
        dict(name="mlp_8k", kind="mlp", n=100, rows=8192),
        # the whole rare-event study, training included
        dict(name="learn_20k", kind="learn", n=100, n_runs=20_000, rounds=2, epochs=6, batch=32_768),
    ]


def _log_int(rng, lo, hi) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    """One more case: networks of 1 to 512 components, a thousand to a million
    runs, tuned or not, with and without per-run outputs."""
    kind = rng.choice(["run"] * 7 + ["batch", "sample", "mlp", "learn"])
    if kind == "run":
        model = rng.choice(["race", "fischer", "fischer", "sir", "sir"] + sorted(FIXTURES))
        c = dict(kind=kind, model=model, n=1, n_runs=1, tuned=rng.random() < 0.3,
                 per_run=rng.choice(["", "", "value", "all"]))
        if model == "race":
            c["n"] = _log_int(rng, 2, 64)
        elif model == "fischer":
            c["n"] = _log_int(rng, 4, 128)
        elif model == "sir":
            c["n"] = _log_int(rng, 16, 512)
        most = MOST_OPS / _run_cost(c)[1]
        c["n_runs"] = _log_int(rng, 300, max(600.0, min(most, 1e6)))
        return c
    if kind == "batch":
        return dict(kind=kind, n_sir=rng.randint(3, 32), n_fischer=rng.randint(3, 32), n_runs=_log_int(rng, 300, 3000))
    if kind == "sample":
        return dict(kind=kind, n=_log_int(rng, 20, 120), n_runs=_log_int(rng, 1000, 60_000))
    if kind == "mlp":
        return dict(kind=kind, n=_log_int(rng, 20, 120), rows=_log_int(rng, 64, 10_000))
    return dict(kind=kind, n=_log_int(rng, 40, 100), n_runs=_log_int(rng, 4000, 20_000), rounds=rng.randint(1, 2),
                epochs=rng.randint(2, 6), batch=_log_int(rng, 8000, 32_768))


def _run_cost(case) -> tuple[float, float]:
    """Race steps and lane-operations of one run (averages measured with the
    sequential reference simulation, interpolated over the width)."""
    n = case["n"]
    if case["model"] == "race":
        return 35.0 * n, 35.0 * n * (160.0 + 59.5 * n)
    if case["model"] == "fischer":
        return 62.0 * n ** 0.41, 62.0 * n ** 0.41 * (160.0 + 13.5 * n)
    if case["model"] == "sir":
        return 1.05 * n, 1.05 * n * (380.0 + 5.0 * n)
    return FIXTURES[case["model"]][4:6]


def _fixture_text(model) -> tuple[str, str]:
    name, locq = FIXTURES[model][:2]
    data = (MODELS / name).read_bytes()
    return (gzip.decompress(data) if name.endswith(".gz") else data).decode(), locq


def _network(case):
    """The parsed network and query of a run case."""
    model, n = case["model"], case["n"]
    if model == "race":
        net = cs.ParsedNetwork.from_string(G.race_network(n)[0], "")
        return net, cs.var_query(net.variable_id("count"), 100.0, threshold=5 * n - 1)
    if model == "fischer":
        net = cs.ParsedNetwork.from_string(G.fischer_network(n)[0], "P0.cs")
        return net, cs.reach_query(300.0)
    if model == "sir":
        net = cs.ParsedNetwork.from_string(G.sir_network(n, 0.3, 0.1)[0], "")
        return net, cs.var_query(net.variable_id("I"), 100.0, threshold=max(1, int(0.3 * n)) - 1)
    text, locq = _fixture_text(model)
    net = cs.ParsedNetwork.from_string(text, locq)
    var, bound = FIXTURES[model][2:4]
    if var is None:
        return net, cs.reach_query(bound)
    vid = net.variable_id(var) if isinstance(var, str) else var
    return net, cs.var_query(vid, bound, is_max=model != "fischermulti", estimate=True)


def _totals(r) -> dict:
    return dict(n_runs=r.n_runs, hits=r.hits, estimate=r.estimate, clt_half=r.clt_half, steps=r.steps,
                transitions=r.transitions, truncated=r.truncated, sum=r.sum, sumsq=r.sumsq, vmin=r.vmin, vmax=r.vmax)


# ------------------------------------------------------------ rare events

def _rare(n):
    """The rare-event query on an epidemic of n agents, one infected: a peak
    that the base law reaches with a probability near 1e-5 or below."""
    net = cs.ParsedNetwork.from_string(G.sir_network(n, 0.15, 0.1, initial_infected=1)[0], "")
    return net, cs.var_query(net.variable_id("I"), 50.0, threshold=int(0.9 * n) - 1)


HIDDEN = 128


def _mlp_shape(n) -> tuple[int, int, int, int]:
    """Features (three locations per agent, three variables, time), and
    features, outputs and locations padded to 64."""
    feats = 3 * n + 3 + 1
    up = lambda v: -(-v // 64) * 64  # noqa: E731
    return feats, up(feats), up(3), up(3 * n)


def _mlp_params(n, seed) -> np.ndarray:
    """A proposal as training leaves one: hidden layers at He scale, output
    tilts that speed infections up and recoveries down, varying with the
    state.  Flat [W1 b1 W2 b2 W3 b3]."""
    feats, fpad, opad, _ = _mlp_shape(n)
    rng = np.random.default_rng(seed)
    w1 = np.zeros((fpad, HIDDEN), np.float32)
    w1[:feats] = rng.normal(0.0, math.sqrt(2.0 / feats), (feats, HIDDEN))
    w2 = rng.normal(0.0, math.sqrt(2.0 / HIDDEN), (HIDDEN, HIDDEN)).astype(np.float32)
    w3 = np.zeros((HIDDEN, opad), np.float32)
    w3[:, :3] = rng.normal(0.0, 0.05, (HIDDEN, 3))
    b3 = np.zeros(opad, np.float32)
    b3[:3] = (0.5, -0.6, 0.0)
    zero = np.zeros(HIDDEN, np.float32)
    return np.concatenate([w1.ravel(), zero, w2.ravel(), zero, w3.ravel(), b3])


def _mlp_inputs(case, seed) -> tuple[np.ndarray, np.ndarray]:
    """States as the sampler meets them (one-hot agents, counts over n, time
    over the bound) and an output gradient."""
    n, rows = case["n"], case["rows"]
    feats, fpad, _, lpad = _mlp_shape(n)
    rng = np.random.default_rng(seed + 1)
    x = np.zeros((rows, fpad), np.float32)
    at = rng.integers(0, 3, (rows, n))
    x[np.arange(rows)[:, None], 3 * np.arange(n)[None, :] + at] = 1.0
    for k in range(3):
        x[:, 3 * n + k] = (at == k).sum(1) / n
    x[:, feats - 1] = rng.random(rows)
    g = np.zeros((rows, lpad), np.float32)
    g[:, :3 * n] = rng.normal(0.0, 1.0, (rows, 3 * n))
    return x, g


# ------------------------------------------------------------ the interface

def prepare(case, seed):
    kind = case["kind"]
    if kind == "run":
        net, q = _network(case)
        sim = cs.GpuSimulator(net)
        if case["tuned"]:
            sim.autotune(q, seed=1, sample_runs=max(1024, min(case["n_runs"] // 4, 16384)))
        return dict(case=case, sim=sim, q=q, seed=seed)
    if kind == "batch":
        specs = G.batch_instances(case["n_sir"], case["n_fischer"])
        items = []
        for k, sp in enumerate(specs):
            net = cs.ParsedNetwork.from_string(sp["xml"], sp["loc_query"])
            q = (cs.var_query(net.variable_id(sp["var"]), sp["time_bound"], threshold=sp["threshold"])
                 if sp["kind"] == "sir" else cs.reach_query(sp["time_bound"]))
            items.append((cs.GpuSimulator(net), q, 1000 * seed + k, case["n_runs"]))
        return dict(case=case, batch=cs.Batch(items))
    net, q = _rare(case["n"])
    sim = cs.GpuSimulator(net)
    if kind == "learn":
        return dict(case=case, sim=sim, q=q, seed=seed)
    sampler = cs.ImportanceSampler(sim, q, hidden=HIDDEN)
    sampler.set_params(_mlp_params(case["n"], seed))
    if kind == "sample":
        return dict(case=case, sampler=sampler, seed=seed)
    x, g = _mlp_inputs(case, seed)
    return dict(case=case, sampler=sampler, x=x, g=g)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "run":
        r = state["sim"].run(state["q"], seed=state["seed"], n_runs=case["n_runs"], per_run=PER_RUN[case["per_run"]])
        out = _totals(r)
        out.update({"run_" + k: v for k, v in r.per_run.items()})
        return out
    if kind == "batch":
        res, st = state["batch"].run(1)
        keys = ("hits", "steps", "transitions", "truncated", "estimate", "sum", "sumsq")
        out = {k: np.array([getattr(r, k) for r in res]) for k in keys}
        out["runs"] = st.runs
        return out
    if kind == "sample":
        r = state["sampler"].sample(seed=state["seed"], n_runs=case["n_runs"], use_mlp=True)
        return dict(r.per_run, hits=r.hits, estimate=r.estimate, ess=r.ess, steps=r.steps, transitions=r.transitions)
    if kind == "mlp":
        theta, grad = state["sampler"].mlp_eval(state["x"], state["g"])
        return dict(theta=theta, grad=grad)
    s = cs.ImportanceSampler(state["sim"], state["q"], hidden=HIDDEN, rounds=case["rounds"],
                             runs_per_round=case["n_runs"], epochs=case["epochs"], learning_rate=1e-2,
                             seed=state["seed"])
    rounds = s.train()
    est = s.estimate(seed=state["seed"] + 1, batch_runs=case["batch"], max_runs=case["batch"], rel_target=0.1)
    out = dict(params=s.get_params(), n_runs=est.n_runs, hits=est.hits, estimate=est.estimate, ess=est.ess,
               steps=est.steps, transitions=est.transitions)
    for k in ("level", "elites", "hits", "estimate", "ess", "pairs"):
        out["round_" + k] = np.array([r[k] for r in rounds])
    s.close()
    return out


def work(case) -> dict:
    """What the call cannot do without: the lane-operations of its race steps
    (and the matrix products of its proposal network), its inputs read once
    and its results written once."""
    kind = case["kind"]
    if kind == "run":
        steps, ops = _run_cost(case)
        return dict(bytes=case["n_runs"] * BYTES_PER_RUN[case["per_run"]], flops=case["n_runs"] * ops)
    if kind == "batch":
        total = 0.0
        for sp in G.batch_instances(case["n_sir"], case["n_fischer"]):
            total += _run_cost(dict(model=sp["kind"], n=sp["n"]))[1]
        return dict(bytes=case["n_runs"] * 17 * (case["n_sir"] + case["n_fischer"]), flops=case["n_runs"] * total)
    feats, fpad, _, lpad = _mlp_shape(case["n"])
    forward = 2.0 * (feats * HIDDEN + HIDDEN * HIDDEN + HIDDEN * 3)
    if kind == "mlp":
        params = 4 * (fpad * HIDDEN + HIDDEN * HIDDEN)
        return dict(bytes=case["rows"] * 4 * (fpad + 2 * lpad) + 2 * params, flops=3 * forward * case["rows"])
    n = case["n"]
    ops = 1.05 * n * (380.0 + 5.0 * n)
    macro = 1.9 * n  # transitions that end a macro-step
    if kind == "sample":
        return dict(bytes=case["n_runs"] * 37, flops=case["n_runs"] * (ops + macro * forward))
    runs = case["rounds"] * case["n_runs"] + case["batch"]
    pairs = case["rounds"] * 0.12 * case["n_runs"] * macro
    return dict(bytes=4 * fpad * HIDDEN + 37 * case["batch"],
                flops=runs * (ops + macro * forward) + case["epochs"] * pairs * 3 * forward)


def exact(case, seed):
    """The proposal network in 64 bits; simulated runs have no other value
    than their own."""
    if case["kind"] != "mlp":
        return None
    n, clamp = case["n"], 4.0
    feats, fpad, opad, lpad = _mlp_shape(n)
    p = _bf16(_mlp_params(n, seed))
    raw = _mlp_params(n, seed).astype(np.float64)
    x, g = _mlp_inputs(case, seed)
    x = _bf16(x)
    at = 0
    parts = []
    for shape, rounded in (((fpad, HIDDEN), True), ((HIDDEN,), False), ((HIDDEN, HIDDEN), True), ((HIDDEN,), False),
                           ((HIDDEN, opad), True), ((opad,), False)):
        size = int(np.prod(shape))
        parts.append((p if rounded else raw)[at:at + size].reshape(shape))
        at += size
    w1, b1, w2, b2, w3, b3 = parts
    h1 = np.maximum(x @ w1 + b1, 0.0)
    h2 = np.maximum(h1 @ w2 + b2, 0.0)
    out = np.clip(h2 @ w3 + b3, -clamp, clamp)
    out[:, 3:] = 0.0
    theta = np.zeros((case["rows"], lpad))
    go = np.zeros_like(out)
    for k in range(3):
        theta[:, k:3 * n:3] = out[:, k:k + 1]
        go[:, k] = g[:, k:3 * n:3].astype(np.float64).sum(1) * (np.abs(out[:, k]) < clamp)
    d2 = (go @ w3.T) * (h2 > 0.0)
    d1 = (d2 @ w2.T) * (h1 > 0.0)
    grad = np.concatenate([(x.T @ d1).ravel(), d1.sum(0), (h1.T @ d2).ravel(), d2.sum(0), (h2.T @ go).ravel(),
                           go.sum(0)])
    return dict(theta=theta, grad=grad)


def _bf16(v: np.ndarray) -> np.ndarray:
    """Rounded to bfloat16 (nearest even), as float64."""
    u = np.ascontiguousarray(v, np.float32).view(np.uint32).astype(np.uint64)
    u = (u + 0x7FFF + ((u >> np.uint64(16)) & np.uint64(1))) & np.uint64(0xFFFF0000)
    return u.astype(np.uint32).view(np.float32).astype(np.float64)
