"""bench.py's result line: the fields a reader of the line relies on, unrounded where
they are the result, and a length that does not grow with the steps (a record that
keeps the last 8,000 characters of the output holds it whole)."""
import json

import pytest

import bench


def record(steps, extras):
    its = [9 + s % 3 for s in range(steps)]
    rows = [dict(step=s, p_rel_l2=1.2345678901234567e-12 * (s + 1), fp64_its=9, mixed_its=9 + s % 2,
                 fp64_rel_res=3.1058564714192846e-10, mixed_rel_res=5.1333247187859e-10,
                 fp64_maxdiv=2.5844546183806016e-09, mixed_maxdiv=2.5812408806736342e-09) for s in range(steps)]
    lat = dict(n=50, p50_ms=29.612345678901234, p99_ms=87.11234567890123, mean_ms=31.01234567890123)
    serve = dict(cases=50, step_latency=lat, cell_updates_per_s=173312345.67890123, makespan_s=2.5712345678901234,
                 bytes_peak=35970351104, failed=0, max_its=its * 5)
    phases = dict(momentum_ms=23.123456789012345, poisson_ms=59.12345678901234, poisson_ms_per_iteration=6.5692729765569)
    leg = dict(precision="mixed16", steps_per_s=10.964912280701755, ms_per_step=91.2, its=its,
               cell_updates_per_s=367920175.43859649, **phases)
    names = [f"{a}_{b}" for a in ("serving", "ensemble", "serving_batched", "ensemble_batched") for b in ("mixed", "fp64")]
    roof = dict(bound="hbm", model="m" * 80, V=363, its=its, bytes_per_step=1.1e11, achieved=4012.3456789, peak=8000.0,
                unit="GB/s", frac=0.50154320986)
    cpu = dict(value=0.006979207878889192, unit="steps/s", cores=16, kind="port", sample="s" * 250,
               cell_updates_per_s=234183.35618605162)
    return {
        "metric": bench.METRIC, "value": 10.964912280701755, "unit": "steps/s", "n_gpus": 1, "steps": steps, "warmup": 5,
        "ms_per_step": 91.20000000000073, "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "f64/f32", "data": "synthetic", "config": dict(workload="w" * 120, cells=33554432, **bench.SOLVER),
        "fp64": leg, "mixed": leg, "mixed_over_fp64": 1.7612345678901234,
        "mixed_fp32": dict(leg, over_fp64=1.5, accuracy=rows) if extras else None,
        "mixed_fp32_4level_rb": (dict(leg, mg_levels=4, semi_coarsening=[0, 0, 0], **bench.STATED_PC["solver"],
                                      over_fp64=1.1, accuracy=rows) if extras else None),
        "shard_share_8way": dict(leg, cells=[512, 256, 32], mg_levels=8, dt=6e-5) if extras else None,
        "host_exchange_ms_per_step": 52.123456789, "pcie_inclusive_mixed_ms_per_step": 143.323456789,
        "accuracy": rows if extras else [],
        "ensemble_latency_ms": {f"{n}_{q}": 29.612345678901234 for n in names for q in ("p50", "p99")} if extras else None,
        "serving": {n: serve for n in names} if extras else None,
        "roofline": dict(bound="hbm", kernel="k" * 130, launches=1080, avg_us=253.0123456789, bytes_per_launch=1.2317e9,
                         achieved=4868.123456789, peak=8000.0, unit="GB/s", frac=0.60851543, traffic=1.4e9),
        "step_roofline": {"fp64": roof, "mixed": roof, "mixed_fp32": roof}, "cpu_baseline": cpu, "cpu_baseline_1core": cpu,
        "gpu_mixed_over_cpu": 1571.1, "gpu_mixed_over_cpu_1core": 2005.9,
    }


@pytest.mark.parametrize("steps,extras", [(3, True), (20, True), (1000, True), (3, False)])
def test_result_line_is_short_and_whole(steps, extras):
    rec = record(steps, extras)
    line = bench.result_line(rec)
    assert "\n" not in line and len(line) < 6000, len(line)
    out = json.loads(line)
    assert set(out) == set(rec)
    for k in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
              "vs_baseline", "dtype", "data", "config"):
        assert out[k] == rec[k], k
    assert abs(out["roofline"]["frac"] - rec["roofline"]["frac"]) < 1e-5
    if extras:
        assert out["fp64"]["its"] == [9, 11] and out["accuracy"]["steps"] == steps
        assert out["accuracy"]["p_rel_l2"] == pytest.approx(1.2345678901234567e-12 * steps, rel=1e-4)
