"""bench.py's command line on the CPU: it compiles and refuses more than one GPU before it
touches a device (the driver runs it at round end; a syntax error would lose the bench)."""

from __future__ import annotations

import py_compile
import subprocess
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_bench_compiles():
    py_compile.compile(str(ROOT / "bench.py"), doraise=True)


def test_bench_refuses_several_gpus_without_a_device():
    result = subprocess.run([sys.executable, str(ROOT / "bench.py"), "--gpus", "2"], cwd=ROOT,
                            capture_output=True, text=True, timeout=120)
    assert result.returncode == 2
    assert "one GPU" in result.stderr


def test_printed_line_keeps_its_figures_and_fits_a_log_tail():
    import json

    import bench

    stats = {"median_us": 1234.567, "min_us": 1230.123, "max_us": 1250.321, "samples_us": [1234.567] * 11, "GB/s": 1234.56,
             "GB/s_best": 1240.12, "copies": 29, "hbm_frac": 0.3489}
    groups = dict(stats, per_group_us={"q+k+v": 12.345, "o": 12.345, "gate+up": 123.456, "down": 45.678})
    details = {f"C{i}_a_configuration_with_a_long_name_{i}": dict(stats) for i in range(60)}
    details.update({f"C5_layer_{i}": dict(groups) for i in range(6)}, measurement_order=list(details),
                   torch={"torch": "2.10", "cases": {f"mm_{i}": dict(stats) for i in range(8)}})
    cpu = {"ms": 12.345, "GB/s": 1.234, "GFLOP/s": 12.345, "single_thread_ms": 123.456, "single_thread_GB/s": 0.1,
           "sample": "1/4 of each matrix's rows per call; ms scaled to the full call", "numerics": "x" * 60}
    result = {"metric": bench.METRIC, "value": 4000.0, "config": {"workload": "w" * 300, "step_us": dict(stats)},
              "roofline": {"timing": "t" * 1000}, "details": details,
              "cpu_baseline": {"value": 8.0, "per_config": {f"config_{i}": dict(cpu) for i in range(8)}}}
    line = bench.printed(result)
    assert "\n" not in line and len(line) < 8000, len(line)
    read = json.loads(line)
    assert read["metric"] == bench.METRIC and read["value"] == 4000.0
    assert read["details"]["C5_layer_0"] == {"median_us": 1234.567, "GB/s": 1234.56, "per_group_us": groups["per_group_us"]}
    assert read["details"]["torch"]["cases"]["mm_3"]["median_us"] == 1234.567
    assert read["cpu_baseline"]["per_config"]["config_0"]["ms"] == 12.345
    assert result["details"]["C5_layer_0"]["samples_us"]  # the record itself is left whole
