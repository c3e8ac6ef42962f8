"""bench.py's result line: one short JSON object with the contract's keys, whatever else was measured."""
import json

import bench

KEYS = ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling", "vs_baseline",
        "dtype", "data", "config", "roofline")


def result(n_other):
    row = {"case": "c" * 120, "config": "cfg3", "kernel": "k" * 60, "launches": 1, "us_per_call": 4.769, "GB_per_s": 3744.7,
           "TFLOP_per_s": 7.036, "algorithmic_bytes": 17858560,
           "roofline": {"bound": "hbm", "achieved": 3744.7, "peak": 8000.0, "unit": "GB/s", "frac": 0.4681}}
    case = {**row, "M": 1, "hbm_frac": 0.5, "mfma_frac": 0.1, "us_samples": [7.0] * 64}
    return {**{k: "x" for k in KEYS}, "value": 3733.5, "roofline": row["roofline"], "cases": [dict(case) for _ in range(3)],
            "cases_checkpoint_layout_ops": [case] * 8, "other_configs": [row] * n_other, "extra_configs": [row] * 50,
            "cpu_baseline": {"value": 4.0, "unit": "GB/s"}}


def test_line_is_short_and_whole():
    text = bench.headline(result(40))
    line = json.loads(text)
    assert len(text) <= bench.MOST_LINE_BYTES and "\n" not in text
    assert all(k in line for k in KEYS) and line["value"] == 3733.5
    assert "other_configs" not in line and "extra_configs" not in line
    assert line["cases"][0]["us_per_call"] == 4.769 and "us_samples" not in line["cases"][0]
    assert line["cpu_baseline"] == {"value": 4.0, "unit": "GB/s"}


def test_details_leave_before_the_figures():
    full = result(4)
    full["cases"] = full["cases"] * 40
    text = bench.headline(full)
    line = json.loads(text)
    assert len(text) <= bench.MOST_LINE_BYTES and all(k in line for k in KEYS) and "cases" not in line
