"""The bench prints one JSON line that a reader of a bounded tail of its output gets whole."""

import json
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)

import bench  # noqa: E402


def test_the_line_is_short_and_keeps_the_headline_exact():
    entry = {"n": 36, "fp32": "PRIMARY_SUCCESS", **{k: 1.2345678901234567e-07 for k in ("e", "g", "x", "x_refined", "e_refined")}}
    headline = {"metric": bench.METRIC, "value": 37554.512345678, "unit": "Mtet-evals/s", "n_gpus": 1, "steps": 20, "warmup": 5,
                "ms_per_step": 0.034912345678, "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
                "dtype": "f32", "data": "synthetic", "config": {"n_tets": 1310720}}
    out = {**headline, "roofline": {"frac": 0.123456789}, "combined": {"fp32_s": 1.0, "per_instance": [entry] * 64,
                                                                      "fp32_refined": {"branch_switches": [{"instance": 3}]}}}
    line = bench.contract_line(out)
    assert "\n" not in line and len(line) <= 10000
    j = json.loads(line)
    assert {k: j[k] for k in headline} == headline
    assert abs(j["roofline"]["frac"] - 0.123456789) <= 1e-6 and j["combined"]["fp32_s"] == 1.0
    assert "per_instance" not in j["combined"] and j["combined"]["fp32_refined"]["branch_switches"] == [{"instance": 3}]
    assert len(out["combined"]["per_instance"]) == 64  # the caller's dictionary is left as it is
