"""bench.py's printed line: its headline keys as they are, and short enough to be
whole in the last 8000 characters of a log."""

import json

import bench


def _record():
    kernels = {name: {"us": 10.123, "GB/s": 12345.6, "frac_hbm": 0.12345, "TFLOP/s": 123.45,
                      "frac_mfma_f16": 0.12345, "algorithmic_bytes": 234917888,
                      "flops": 234881024, "replicas": 12, "shape": "x[1,4096] W[6144,4096]",
                      "launches_per_graph": 96, "traffic_bytes": 234917888.0}
               for name, _ in bench.sweep_workloads()}
    trace = {name: {"call_us": 9.279, "kernel_us": {"gemv_kernel<1, 1, 1, 8, false, 8>": 9.279}}
             for name in kernels}
    decomp = {name: {**{k: 123.456 for k in (
        "t_stream_us", "t_graph_us", "t_fused_us", "delta_launch_us", "B_us", "residual_us",
        "t_fused_graph_us", "residual_graph_us")}, "delta_launch_ci": [1.0, 2.0],
        "bound": "launch-bound", "dominant": "launch", "total_bytes": 10**9,
        "eliminable_bytes": 10**6, "fused_extra_bytes": 0, "fused_check": {"ok": True},
        "samples_us": {k: [123.456] * 30 for k in ("stream", "graph", "fused")}}
        for name, _ in bench.DECOMP_WORKLOADS}
    return {
        "metric": bench.METRIC, "value": 6768.9, "unit": "GB/s", "n_gpus": 1, "steps": 20,
        "warmup": 5, "ms_per_step": 0.034705, "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "f16", "data": "synthetic", "config": {"workload": "x" * 120},
        "roofline": {"bound": "hbm", "kernel": "k" * 60, "traffic": 1.0}, "kernels": kernels,
        "f4_two_launch_parts": {"f4_L8192": {"split_us": 1.0, "merge_us": 2.0}},
        "roofline_by_kernel": bench.roofline_by_kernel(kernels, {}, trace, trace),
        "decomposition": decomp,
        "cpu_baseline": {"value": 400.0, "unit": "GB/s", "cores": 16, "kind": "port",
                         "sample": "s" * 160, "us_per_call": 100.0, "cpu_model": "c" * 40,
                         "rows": {"f1_cfg1": {"us_per_call": 90.0},
                                  "f4_L8192": {"us_per_call": 80000.0}}}}


def test_printed_line_is_short_and_whole():
    rec = _record()
    line = json.dumps(bench.short_record(rec))
    assert len(json.dumps(rec)) > 8000 and len(line) < 7000, len(line)
    short = json.loads(line)
    for key in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step",
                "higher_is_better", "scaling", "vs_baseline", "dtype", "data", "config"):
        assert short[key] == rec[key]
    assert set(short["kernels_us_gbs"]) == set(rec["kernels"])
    assert short["decomposition"]["f1_cfg1"]["t_fused_us"] == 123.456
    head = {k: rec[k] for k in list(rec)[:14]}
    assert bench.short_record(head) == head
