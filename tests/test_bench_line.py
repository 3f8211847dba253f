"""bench.py's one line stays short (readers keep its end only) and holds the
headline figures, whatever the record's other parts grow to."""
import json
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


def test_the_line_is_short_and_complete():
    long = {f"field_{k}": {"max": 0.12345678901234567, "text": "x" * 200} for k in range(100)}
    out = {k: 1.2345678901234567 for k in bench.LINE_KEYS}
    out["config"] = {"workload": "w" * 400, "step": "s" * 400, "cells_total": 1, "tiles": [0, 0]}
    for part, keys in bench.LINE_PARTS.items():
        out[part] = dict({k: 1.2345678901234567 for k in keys}, report=long)
    out["serving"] = {"workload": "w" * 500,
                      "sweep": [dict({k: 1.2345678901234567 for k in bench.SERVING_KEYS}, more=long) for _ in range(4)]}
    out["mixed_vs_fp64_error"] = long
    text = json.dumps(bench.headline(out))
    assert len(text) < 5000
    line = json.loads(text)
    for k in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
              "vs_baseline", "dtype", "data", "config"):
        assert line[k] == out[k]
    assert set(line["roofline"]) == set(bench.LINE_PARTS["roofline"]) and len(line["serving"]) == 4
    out["serving"] = out["accuracy"] = out["cpu_baseline"] = None  # legs left out
    assert "serving" not in bench.headline(out) and "accuracy" not in bench.headline(out)
