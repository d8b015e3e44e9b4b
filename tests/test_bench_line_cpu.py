"""bench.py's printed line: the headline first, and no longer than what a reader of its last 12 KB holds
whole, however many points the sweeps have."""
import json

import bench


def test_line_holds_the_headline_and_not_the_sweeps():
    head = {"metric": bench.METRIC, "value": 1180.21, "unit": "frames/s", "n_gpus": 1, "steps": 50, "warmup": 5,
            "ms_per_step": 0.8473, "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "x" * 60,
            "data": "synthetic", "config": {"workload": "w" * 300}}
    # the remaining entries at about their size (9 KB together) and sweeps of 19 points
    rest = {k: {"note": "n" * 700} for k in ("learned", "plain_tile_lists", "reference_estimator", "roofline",
                                            "roofline_culling", "batched_views", "shadow_passes", "cpu_baseline")}
    point = {"spp": 8, "relmse": 0.000692, "frames_per_s": 1642.15,
             "kernels_ms": {"cull_global": 0.03, "gather": 0.1, "denoise": 0.2, "direct_light_concurrent": 0.04},
             "atrous_at_equal_relmse": {"brackets": [{"spp": 1.0}] * 20}}
    line = bench.line_of(head | rest | {k: [point] * 19 for k in bench.SWEEPS})
    got = json.loads(line)
    assert "\n" not in line and len(line) < 10000
    assert {k: got[k] for k in head} == head and list(got)[:len(head)] == list(head)
    assert all(got[k] == v for k, v in rest.items())
