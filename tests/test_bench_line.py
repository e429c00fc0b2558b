"""bench.py's printed line: short enough for a captured output's tail, with the headline's fields whole."""
import json
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)

import bench  # noqa: E402


def test_printed_line_is_short_and_whole():
    leg = {"workload": "x" * 300, "value": 1.23456789012345e6, "unit": "systems/s", "identical": True, "worst": float("inf"),
           "by_size": {str(n): {"ms": 1.0 / 3.0 * n, "note": "y" * 100, "accuracy": {"frac": 0.999, "max": 1e-4}}
                       for n in range(30)}, "list": list(range(100))}
    head = {"metric": "ODE systems/sec @ rel err<=1e-3 vs FP64; p50/p99 request latency", "value": 21.7e6 / 3,
            "unit": "systems/s", "n_gpus": 1, "steps": 20, "warmup": 5, "ms_per_step": 48.1234567,
            "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f32",
            "data": "synthetic (seeded)", "config": {"workload": "z" * 120, "nsys": 1 << 20},
            "latency_ms": {"p50": 48.1, "p99": 49.2, "request": "one step (all systems)"}}
    for legs in (0, 1, 5, 20):
        line = {**head, **{f"leg{i}": leg for i in range(legs)}}
        text = bench.compact(line)
        assert len(text) <= bench.LINE_MAX and "\n" not in text
        got = json.loads(text, parse_constant=lambda c: 1 / 0)  # (no Infinity or NaN)
        assert {k: got[k] for k in head} == head
        if legs == 5:
            assert got["leg0"]["value"] == 1.23457e6 and got["leg0"]["identical"] is True
