"""bench.py's stdout line stays short enough to be read from the end of a
captured output, whatever was measured, and keeps the contract's keys as they
are (no GPU)."""
import importlib.util
import json
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CONTRACT = ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step",
            "higher_is_better", "scaling", "vs_baseline", "dtype", "data", "config")


@pytest.fixture(scope="module")
def bench():
    spec = importlib.util.spec_from_file_location("bench_module", os.path.join(ROOT, "bench.py"))
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


def _out(sections):
    roof = {"kernel": "k", "bound": "hbm", "achieved": 3182.812345678, "peak": 8000.0, "unit": "GB/s",
            "frac": 0.3978515432, "traffic": 2634695305, "ms_per_step": 0.4923212345,
            "measured": "x" * 250, "algorithmic": "y" * 60}
    roof["kernels"] = {k: dict(roof) for k in ("gather", "deposit_J", "dht")}
    leg = {"value": 8028133699.71845, "ms_per_step": 2.070438861846924, "roofline": roof}
    big = {"n%d" % i: {"avg_us": i / 7, "note": "z" * 120, "GB/s": i / 3} for i in range(60)}
    out = {"metric": "particle-steps/s", "value": 5994982506.543188, "unit": "particle-steps/s",
           "n_gpus": 1, "steps": 20, "warmup": 5, "ms_per_step": 11.142277717590332,
           "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f64",
           "data": "synthetic (seeded plasma with the workload's density profile, Gaussian laser)",
           "config": {"workload": "w" * 100, "Nz": 4096, "dt": 0.020000000001}}
    out.update({k: dict(leg, more=big) for k in sections})
    return out


@pytest.mark.parametrize("sections", [(), ("roofline", "mixed"),
                                      ("roofline", "mixed", "secondary", "kernels", "configs",
                                       "differentiable", "diagnostics", "cpu_baseline")])
def test_line_is_short_and_keeps_the_contract(bench, sections):
    out = _out(sections)
    whole = json.dumps(out)
    line = json.dumps(bench.headline(out))
    assert len(line) <= bench.LINE_MAX <= 8000 and "\n" not in line
    got = json.loads(line)
    for k in CONTRACT:
        assert got[k] == out[k], k
    assert json.dumps(out) == whole  # the measured results are left as they were


def test_sections_are_rounded_not_changed(bench):
    out = _out(("mixed",))
    m = bench.headline(out)["mixed"]
    assert m["ms_per_step"] == 2.0704 and m["value"] == 8.0281e9
    r = m["roofline"]
    assert r["frac"] == 0.39785 and "measured" not in r
    assert set(r["kernels"]) == {"gather", "deposit_J", "dht"}
    assert r["kernels"]["dht"]["achieved"] == 3182.8
