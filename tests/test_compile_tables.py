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
