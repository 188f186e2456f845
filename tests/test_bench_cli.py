"""bench.py's command-line contract, without a GPU: one GPU only, sane step counts."""
from __future__ import annotations

import importlib.util
import json
import subprocess
import sys
import types

from conftest import ROOT


def run_bench(*args):
    return subprocess.run([sys.executable, str(ROOT / "bench.py"), *args], capture_output=True, text=True, timeout=120)


def test_more_than_one_gpu_is_refused_with_a_message():
    r = run_bench("--gpus", "2")
    assert r.returncode == 2
    line = json.loads(r.stdout.strip().splitlines()[-1])
    assert "one GPU" in line["error"]


def test_step_counts_are_checked():
    for args in (("--steps", "0"), ("--warmup", "-1")):
        r = run_bench(*args)
        assert r.returncode == 2 and "--steps must be >= 1" in r.stderr, args


def load_bench():
    spec = importlib.util.spec_from_file_location("bench", ROOT / "bench.py")
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


class PlannedJob:
    """What the labels of a benchmark line are made from, as the headline job plans it."""

    def __init__(self, split, path=2, w_nab=157):
        self._split, self._path, self._w = split, path, w_nab

    def info(self):
        return types.SimpleNamespace(n=20000, m=1000, kt=16)

    def plan(self):
        return {"H": {"nab": 16, "path": self._path}, "W": {"nab": self._w, "path": self._path}}

    def split(self):
        return self._split


def test_traffic_is_that_of_the_kernels_that_ran():
    # A profile's bytes go with the kernels it was taken of, and with no others.
    bench = load_bench()
    label = bench.partial_kernels(PlannedJob(False))
    assert label == "k_partial_mfma<16,1,4> (H half), k_partial_mfma<16,2,2> (W half)"
    assert bench.measured_traffic(label) > 81_344_000
    for other in (PlannedJob(True), PlannedJob(False, w_nab=313), PlannedJob(False, path=1)):
        label = bench.partial_kernels(other)
        assert "k_partial_mfma<16,2,2>" not in label and bench.measured_traffic(label) is None
