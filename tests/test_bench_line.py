"""The benchmark's printed line: whoever keeps only the last few KiB of a run's output must still have all of it."""
import importlib.util
import json
import os


def test_the_printed_line_stays_short_and_keeps_the_headline():
    path = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bench.py")
    spec = importlib.util.spec_from_file_location("bench", path)
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    names = ["ns"] + bench.DEFAULT_EXTRA.split(",")
    detail = {"us_per_call": 22.767, "kernel_us_avg_events": 22.727, "roofline_frac": 0.6615, "plan": {"note": "n" * 300}, "parity": {"note": "p" * 400}}
    probe = {"us_per_launch": 18.553, "note": "n" * 200}
    ceiling = {"stream_read": [dict(probe)] * 4, "stream_read_best_us": 18.5, "empty_grid": probe, "loads_only": probe, "compute_only": probe,
               "timeline_us": {"first_wave_start_to_last_store": 22.3, "note": "t" * 1500}}
    rows = {"stream_read": probe, "loads_only": probe, "compute_only": probe}
    out = {"metric": "HBM GB/s", "value": 2210.0, "unit": "GB/s", "n_gpus": 1, "steps": 20, "warmup": 5, "ms_per_step": 0.004,
           "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f16", "data": "synthetic", "config": {"name": "ns"},
           "roofline": {"frac": 0.28, "by_workload": {n: [22.727, 0.6615, 1] for n in names}},
           "other_workloads": {n: detail for n in names}, "all_parity_ok": True,
           "ceilings": {"ns": ceiling, "c5": ceiling, "c4:m8": rows, "c5:m16": rows, "c1": None}}
    line = bench.short_line(out)
    assert len(json.dumps(line)) < 6000 and len(json.dumps(out)) > 20000
    assert {k: v for k, v in line.items() if k not in ("ceilings", "other_workloads")} == \
        {k: v for k, v in out.items() if k not in ("ceilings", "other_workloads")}
    assert line["other_workloads"]["c5"] == {"us_per_call": 22.767}
    assert line["ceilings"]["c5"]["stream_read"] == 18.5 and line["ceilings"]["c4:m8"]["loads_only"] == 18.553
