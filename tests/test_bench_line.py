"""bench.py's result line (CPU): the keys of a result, short, with the long records
on stderr."""
import json

import bench

KEYS = ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
        "vs_baseline", "dtype", "data", "config")


def test_result_line_is_short_and_whole(capsys):
    result = {k: k for k in KEYS}
    result.update({k: [{"us": 1.0, "text": "x" * 300}] * 30 for k in bench.RECORDS})
    result["roofline"] = {"frac": 0.4}
    result["cpu_baseline"] = {"value": 0.055, "unit": "TFLOP/s", "legs": [{"text": "x" * 300}] * 30}
    line = json.loads(bench.report(result))
    assert set(line) == {*KEYS, "roofline", "cpu_baseline"}
    assert line["cpu_baseline"] == {"value": 0.055, "unit": "TFLOP/s"}
    assert len(json.dumps(line)) < 4096
    records = {}
    for ln in capsys.readouterr().err.splitlines():
        records.update(json.loads(ln.removeprefix("[bench] record ")))
    assert records == {**{k: result[k] for k in bench.RECORDS}, "cpu_baseline_legs": result["cpu_baseline"]["legs"]}


def test_result_without_baseline():
    assert json.loads(bench.report({"value": 1, "cpu_baseline": None})) == {"value": 1, "cpu_baseline": None}
