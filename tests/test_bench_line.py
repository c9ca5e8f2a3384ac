"""What the benchmark prints: a short line on standard output, so that it is whole in the last kilobytes of it."""
import json

import bench


def test_the_line_is_short_and_nothing_is_lost():
    contract = {"metric": "m" * 90, "value": 3010.0, "unit": "GB/s", "n_gpus": 1, "steps": 20, "warmup": 5, "ms_per_step": 0.58,
                "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f32", "data": "synthetic",
                "config": {"workload": "w" * 150, "step_bytes": 1, "step_elements": 2, "seed": 3},
                "roofline": {"kernel": "k" * 60, "traffic_source": "t" * 150}, "parity_gate": "ok"}
    rows = {f"row{i}": {"ms_median": 0.1, "timing": "t" * 60} for i in range(80)}
    cpu = {"value": 1.0, "unit": "GB/s", "sample": "s" * 200}
    line, details = bench.split_report({**contract, "parity": rows, "launches": rows, "breakdown": rows,
                                        "cpu_baseline": {**cpu, "configs": rows}})
    assert line == {**contract, "cpu_baseline": cpu} and len(json.dumps(line)) < 4000
    assert details == {"parity": rows, "launches": rows, "breakdown": rows, "cpu_baseline_configs": rows}
    assert bench.split_report({**contract, "cpu_baseline": None, "breakdown": {}}) == (
        {**contract, "cpu_baseline": None}, {"breakdown": {}})
