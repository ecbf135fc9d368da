"""The lowering of networks to the run kernel's tables, run on the CPU in a
build that stops at undefined behaviour."""
from __future__ import annotations

import gzip
import math
import shutil
import subprocess
from pathlib import Path

import pytest

from cusmc_amd import generators as G

ROOT = Path(__file__).resolve().parent.parent
CSRC = ROOT / "cusmc_amd" / "csrc"
MODELS = ROOT / "tests" / "golden" / "models"


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    """Lowers the given model texts; the lines printed for each."""
    out = tmp_path_factory.mktemp("compile_check")
    exe = out / "compile_check"
    subprocess.run([shutil.which("g++") or "g++", "-std=c++17", "-O1", "-g", "-ffp-contract=off",
                    "-fsanitize=undefined", "-fno-sanitize-recover=all", f"-I{ROOT / 'include'}", f"-I{CSRC}",
                    str(ROOT / "tests" / "compile_check.cpp"),
                    *[str(CSRC / s) for s in ("compile.cpp", "network.cpp", "uppaal.cpp")], "-o", str(exe)], check=True)

    def run(*texts):
        files = []
        for k, t in enumerate(texts):
            files.append(out / f"model{k}.xml")
            files[-1].write_text(t)
        r = subprocess.run([str(exe), *map(str, files)], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True)
        assert r.returncode == 0, r.stderr[-2000:]
        models = []
        for line in r.stdout.splitlines():
            if line.startswith("model "):
                models.append([])
            models[-1].append(line.split())
        return models
    return run


def _guarded(guards):
    """One component with an edge per guard on the integer variable v."""
    edges = "".join(f"""<transition><source ref="id0"/><target ref="id0"/><label kind="guard">{g}</label></transition>"""
                    for g in guards)
    return f"""<?xml version="1.0" encoding="utf-8"?>
<nta><declaration>int v = 0;</declaration>
<template><name>T</name><declaration></declaration>
<location id="id0"><name>l0</name></location><init ref="id0"/>{edges}</template><system>system T;</system></nta>"""


def test_equality_intervals(check):
    """`v == r` holds on the doubles within 1e-5 of r: the interval's ends pass
    the test and their neighbours outside do not."""
    values = [0, 1, -1, 2, 7, -7, 1000000, 2147483647, -2147483648]
    lines = check(_guarded([f"v == {r}" for r in values]))[0]
    got = [(float.fromhex(a), float.fromhex(b)) for kind, a, b in (l for l in lines if l[0] == "interval")]
    assert len(got) == len(values)
    for r, (lo, hi) in zip(values, got):
        assert lo <= r <= hi
        assert abs(lo - r) <= 1e-5 and abs(hi - r) <= 1e-5, r
        assert abs(math.nextafter(lo, -math.inf) - r) > 1e-5 and abs(math.nextafter(hi, math.inf) - r) > 1e-5, r


def test_models_lower_without_undefined_behaviour(check):
    texts = [(f.read_text() if f.suffix == ".xml" else gzip.decompress(f.read_bytes()).decode())
             for f in sorted(MODELS.glob("*.xml")) + sorted((MODELS / "large").glob("*.gz"))]
    texts += [G.race_network(8)[0], G.fischer_network(32)[0], G.sir_network(77, 0.3, 0.1)[0]]
    for lines in check(*texts):
        assert int(lines[0][2]) > 0


def _chains(components, length, last=""):
    """Instances of a template whose locations are a chain of equal ones; `last`:
    a guard on the final edge of the first component alone."""
    tpls, names = [], []
    for c in range(components):
        loc = "".join(f'<location id="id{c * 1000 + k}"><name>l{c}_{k}</name></location>' for k in range(length))
        tr = "".join(f"""<transition><source ref="id{c * 1000 + k}"/><target ref="id{c * 1000 + k + 1}"/>"""
                     + (f'<label kind="guard">{last}</label>' if last and c == 0 and k == length - 2 else "")
                     + "</transition>" for k in range(length - 1))
        tpls.append(f"""<template><name>T{c}</name><declaration></declaration>{loc}<init ref="id{c * 1000}"/>{tr}
</template>""")
        names.append(f"T{c}")
    return f"""<?xml version="1.0" encoding="utf-8"?>
<nta><declaration>int v = 0;</declaration>{"".join(tpls)}<system>system {", ".join(names)};</system></nta>"""


@pytest.mark.parametrize("length", [63, 64, 65, 66, 67, 100, 300])
def test_chains_of_equal_locations_share_records(check, length):
    """Equal locations of a chain differ by how far they are from its end, which
    takes a pass a link to find out; instances share their records whatever the
    length (record 0 stands for no component)."""
    one, eight, odd = check(_chains(1, length), _chains(8, length), _chains(8, length, last="v == 0"))
    assert int(one[0][4]) == length + 1
    assert int(eight[0][2]) == 8 * length and int(eight[0][4]) == length + 1
    # one instance leads to another guard: its records are its own, but for those past the guard
    assert length + 2 < int(odd[0][4]) <= 2 * length + 1


def _receivers(edges):
    """A sender and two components that receive on the given (channel, weight) edges."""
    tpls = ["""<template><name>S</name><declaration></declaration><location id="id0"><name>s</name></location>
<init ref="id0"/><transition><source ref="id0"/><target ref="id0"/><label kind="synchronisation">a!</label></transition>
<transition><source ref="id0"/><target ref="id0"/><label kind="synchronisation">b!</label></transition></template>"""]
    for c in (1, 2):
        tr = "".join(f"""<transition><source ref="id{c}0"/><target ref="id{c}0"/><label kind="synchronisation">{ch}?</label>
<label kind="assignment">n = n + {k % 3}</label>{f'<label kind="probability">{w}</label>' if w else ""}</transition>"""
                     for k, (ch, w) in enumerate(edges))
        tpls.append(f"""<template><name>R{c}</name><declaration></declaration><location id="id{c}0"><name>r</name></location>
<init ref="id{c}0"/>{tr}</template>""")
    return f"""<?xml version="1.0" encoding="utf-8"?>
<nta><declaration>broadcast chan a, b; int n = 0;</declaration>{"".join(tpls)}<system>system S, R1, R2;</system></nta>"""


def test_commuting_receivers_fire_together(check):
    """Receivers whose edges add integers fire all at once, with up to 32 edges
    and whatever their constant weights sum to."""
    cases = [[("a", 1), ("a", 3)], [("a", 2147483647)] * 2, [("a", 1)] * 32, [("a", 1)] * 3, [("a", 2), ("b", 2147483647)] * 16]
    for case, lines in zip(cases, check(*map(_receivers, cases))):
        kinds = [l[1] for l in lines if l[0] == "receives"]
        assert kinds == ["together"], case


@pytest.mark.parametrize("declared,updates,window", [
    ("", "x = 0", "inline"), ("int v = 7;", "x = v", "inline"), ("int v = 7;", "x = v - 2 * v", "inline"),
    ("int v = 7; int w = 1;", "v = v + 3, w = v * v, x = w", "inline"), ("int v; int w;", "v = w, w = v, x = w", "inline"),
    ("int v; int w;", "v = w + 1, w = v, x = w", "general"), ("int v = 2;", "v = v * v, x = v", "general"),
    ("int v = 2;", "v = v + v, x = v", "general"), ("int v = 2;", "x = v / 2", "general"),
    ("clock y;", "x = y", "general"), ("", "x = x + 1", "general"), ("int v = 2;", "v = x, x = v", "general"),
    ("int " + ", ".join(f"v{k}" for k in range(200)) + ";",
     ", ".join(f"v{k + 1} = v{k} + 1" for k in range(199)) + ", x = v199", "general"),
    ("int " + ", ".join(f"v{k}" for k in range(6)) + ";",
     ", ".join(f"v{k + 1} = v{k} + 1" for k in range(5)) + ", x = v5", "inline")])
def test_windows_known_to_end(check, declared, updates, window):
    """A window under one constant bound is read off its record where the values
    that its clock is set to are known to be moderate."""
    model = f"""<?xml version="1.0" encoding="utf-8"?>
<nta><declaration>clock x; {declared}</declaration><template><name>T</name><declaration></declaration>
<location id="id0"><name>l</name><label kind="invariant">x &lt;= 3</label></location><init ref="id0"/>
<transition><source ref="id0"/><target ref="id0"/><label kind="assignment">{updates.replace(">", "&gt;")}</label></transition>
</template><system>system T;</system></nta>"""
    assert [l[1] for l in check(model)[0] if l[0] == "window"] == [window]
