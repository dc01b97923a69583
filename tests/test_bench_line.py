"""The line that bench.py prints is short enough to be read back whole and
keeps what a reader of it needs; the full report may be as long as it is."""
import importlib.util
import json
import os

from conftest import ROOT


def load_bench():
    spec = importlib.util.spec_from_file_location("bench_under_test", os.path.join(ROOT, "bench.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def full_report():
    x = 1234567890123.456789
    lat = {"p50_ms": x, "p99_ms": x, "mean_ms": x, "max_ms": x, "queries": 1000}
    row = dict(lat, rate_per_s=10000, elapsed_s=x, leaves_per_s=x, batches=100, mean_batch=x,
               by_depth={d: dict(lat, queued_p99_ms=x) for d in range(3, 8)})
    roof = {"bound": "valu", "achieved": x, "peak": x, "unit": "T int32 lane-ops/s", "frac": x, "traffic": x,
            "kernel": "k", "launches": 18, "avg_launch_ms": x, "valu_insts_per_board": x, "valu_source": "s" * 80,
            "peak_note": "n" * 200, "hbm": {"achieved": x, "peak": x, "unit": "GB/s", "frac": x, "note": "n" * 200}}
    table = [{"slider": "kogge_stone", "dedup": True, "blocks_per_cu": 8, "split_depth": 0, "ms_on_512_sample": x}] * 48
    run = {"tt_gb": 16, "depth": 9, "perft": 1, "s": x, "effective_leaves_per_s": x, "boards_per_ply": [10**12] * 9,
           "table_access": {k: x for k in "abcdef"}}
    return {"metric": "m" * 80, "value": x, "unit": "leaves/s", "n_gpus": 1, "steps": 20, "warmup": 5, "ms_per_step": x,
            "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "u64", "data": "synthetic",
            "config": {"workload": "w" * 120, "leaves_per_step": 10**11, "slider": "kogge_stone", "exact": True},
            "variants": {v: {"leaves_per_s": x, "ms_per_step": x} for v in "abcd"},
            "merged": {"leaves_per_s": x, "ms_per_step": x}, "roofline": roof,
            "leaf_totals": {k: 10**10 for k in ("launches", "items", "parents", "grandparents", "ms")},
            "counters": dict({"measured": True, "valu_insts_per_board": x}, **{"c%d" % i: x for i in range(40)}),
            "calib": {"copy": {"gb_per_s_read_plus_write": x}, "issue_probes": {"k%d" % i: {"r": x} for i in range(16)},
                      "cus": 256},
            "batch": {"workload": "w" * 80, "ms": x, "leaves_per_s": x, "autotuned": table[0], "autotune_table": table,
                      "speedup_vs_plain_loop": x, "exact": True},
            "tt": {"workload": "w" * 120, "runs": [run] * 4, "exact": True},
            "serve": {"rates": [row] * 6, "burst_without_table": row, "burst_vs_plain": x, "exact": True},
            "cpu_baseline": {"value": x, "unit": "leaves/s", "cores": 16, "kind": "port", "sample": "s" * 120,
                             "single_thread": {"value": x, "sample": "s" * 60}, "cpu_model": "c" * 40, "nproc": 256},
            "served_p50_ms": x, "served_p99_ms": x}


def test_line_is_short_and_keeps_the_contract():
    full = full_report()
    text = json.dumps(load_bench().summary(full))
    assert len(json.dumps(full)) > 15000  # what could not be read back
    assert len(text) < 7000 and "\n" not in text
    line = json.loads(text)
    for k in ("metric", "unit", "n_gpus", "steps", "warmup", "higher_is_better", "scaling", "vs_baseline", "dtype",
              "data", "config"):
        assert line[k] == full[k]
    assert abs(line["value"] / full["value"] - 1) < 1e-5 and abs(line["ms_per_step"] / full["ms_per_step"] - 1) < 1e-5
    assert line["roofline"]["bound"] == "valu" and len(line["serve"]["rates"]) == 6


def test_legs_that_did_not_run_are_absent():
    full = full_report()
    for k in ("counters", "calib", "batch", "tt", "serve"):
        del full[k]
    line = load_bench().summary(full)
    assert not {"counters", "calib", "batch", "tt", "serve", "leafmodes"} & set(line)
