"""bench.py prints one line that a reader with a small buffer gets whole: the headline, its
configuration and the rooflines, of the other sections their plain figures."""
import json
from pathlib import Path

import bench

ROOT = Path(__file__).resolve().parent.parent


def test_result_line_is_short_and_complete():
    out = json.loads((ROOT / "profiles" / "c2_bench_line.json").read_text())  # a whole run's result
    line = bench.result_line(out)
    text = json.dumps(line)
    assert "\n" not in text and len(text) < 8000 < len(json.dumps(out))
    for k in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
              "vs_baseline", "dtype", "data", "config", "roofline", "roofline_sort_pass", "cpu_baseline"):
        assert line[k] == out[k], k
    for leg, key in (("c3_dynamic", "ms_per_frame"), ("instances", "ms_per_frame"), ("c4_batched", "ms_per_batch")):
        assert line[leg][key] == out[leg][key]
    assert line["c4_batched"]["wavefront"]["ms_per_batch"] == out["c4_batched"]["wavefront"]["ms_per_batch"]
    assert line["c5_serving"]["p99_within_50ms"]["mrays"] == out["c5_serving"]["p99_within_50ms"]["mrays"]


def test_result_line_without_the_optional_legs():
    out = {"metric": "m", "value": 1.0, "config": {"triangles": 1}, "kernels": {"trace": {"ms": 1.0}},
           "cpu_baseline": None, "c4_batched": {"ms_per_batch": 2.0}}
    assert bench.result_line(out) == {"metric": "m", "value": 1.0, "config": {"triangles": 1}, "cpu_baseline": None,
                                      "c4_batched": {"ms_per_batch": 2.0}}
