"""bench.py's result line: the headline's numbers in full, the further
sections' to six digits and without their lists of single measurements."""
import json
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))


def test_line(capsys):
    import bench
    run = {"rate": 16.0, "latency_p99_s": 0.30373972468857824, "requests": 101, "order": "fifo",
           "fp64_replays": [{"err": 1.0}] * 40}
    out = {"metric": "m", "value": 252345678901.2345, "ms_per_step": 0.0664212345678, "steps": 20,
           "roofline": {"frac": 0.1234567890123, "three_step_kernel": {"kernel_avg_us": 1 / 3}},
           "timing": {"timed_loop_us_per_step": 66.123456789},
           "batched": {"value": 228289742418.0047, "autotuned": {
               "rows": 48, "table": [{"rate": 1.0 * k} for k in range(300)]}},
           "serving": {"rates": [run, run]},
           "cpu_baseline": None, "bench_wall_s": 141.123456789}
    text = bench.line(out)
    assert "\n" not in text and len(text) < 1200
    d = json.loads(text)
    for key in ("metric", "value", "ms_per_step", "steps", "roofline", "timing", "bench_wall_s",
                "cpu_baseline"):
        assert d[key] == out[key], key
    assert list(d) == list(out)
    assert d["batched"] == {"value": 228290000000.0, "autotuned": {"rows": 48}}
    for r in d["serving"]["rates"]:
        assert r == {"rate": 16.0, "latency_p99_s": 0.30374, "requests": 101, "order": "fifo"}
    # all of it is in the log
    err = capsys.readouterr().err
    assert '"fp64_replays"' in err and '"table"' in err
