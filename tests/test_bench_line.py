"""bench.py's last line is JSON and short enough to survive in a log that keeps only its end; the rest is printed ahead of it."""
import json

import bench


def full_line():
    configs = {k: {unit: 123456.78, "us": 1.0, "kernel": "k" * 60, "verified": True} for k, unit in bench.SHORT_CONFIGS}
    configs["c5_decode_f32_fused_level3"] = {"error": "RuntimeError: " + "x" * 500}
    return {
        "metric": "GB/s (reductions) vs HBM roofline", "value": 6448.42, "unit": "GB/s", "n_gpus": 1, "steps": 20, "warmup": 5, "ms_per_step": 0.02081,
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "config": {"workload": "w" * 130, "algorithmic_bytes_per_step": 134217732, "kernel": {"strategy": "grid_reduce", "grid_dim": 256, "block_dim": 256, "lds_bytes": 0, "scratch_bytes": 1024}},
        "roofline": {**{k: 1234.567 for k in bench.SHORT_ROOFLINE}, "traffic_source": bench.TRAFFIC_SOURCE, "kernel": "u" * 70, "configs": configs, "launch_floor_model": {"a": 1}},
        "result": -2635.91455078125, "truth_f64": -2635.9143512828937, "runs": [{"ms_per_step": 0.02, "kernel_us": 20.0}] * 3,
        "cpu_baseline": {"value": 52.411, "unit": "GB/s", "cores": 1, "kind": "port", "sample": "4686 passes of the full workload in 12.0 s (" + "s" * 200 + ")", "host_cpus": 16},
        "extras": {**{f"row_{i}": {"us": 1.0, "note": "n" * 300} for i in range(40)}, "broken": {"error": "RuntimeError: " + "x" * 500}},
        "sustained": {"after_s": 0.5, "us_per_step": 21.757},
    }


def test_last_line_is_short_and_holds_the_headline():
    line = full_line()
    text = json.dumps(bench.short_line(line))
    assert len(text) < 2000 and "\n" not in text
    out = json.loads(text)
    for key in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling", "vs_baseline", "dtype", "data", "config"):
        assert out[key] == line[key], key
    assert out["roofline"]["frac"] == line["roofline"]["frac"] and out["cpu_baseline"]["value"] == 52.411
    assert out["configs"]["c5_decode_f32_fused_level3 tok/s"] == "error" and out["configs"]["c3_bmm_f32_8x1024^3 TFLOP/s"] == 123456.78
    assert out["failed"] == ["broken"]


def test_details_hold_everything_else():
    line = full_line()
    got = dict(bench.details(line))
    assert {f"extras.{k}" for k in line["extras"]} <= set(got) and {f"roofline.configs.{k}" for k in line["roofline"]["configs"]} <= set(got)
    assert got["roofline"]["launch_floor_model"] == {"a": 1} and got["runs"] == line["runs"] and got["sustained"] == line["sustained"]
    assert not any(name.startswith("{") for name in got)
