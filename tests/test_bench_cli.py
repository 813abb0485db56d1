"""bench.py's command-line contract and its CPU baseline, on the CPU.

- `--gpus N` above 1 exits with status 2 and says that only one GPU is
  measured (no GPU is touched before that check).
- An unknown `--secondary` name is a usage error.
- The printed line holds the contract's keys and stays short, however many
  rounds the secondary figures hold.
- The CPU baseline (the oracle's gather + SDPA path, timed) returns the
  fields the bench line's `cpu_baseline` object carries.
"""

import importlib.util
import json
import subprocess
import sys
import types
from pathlib import Path

import torch

ROOT = Path(__file__).resolve().parents[1]


def run_bench(*args):
    return subprocess.run([sys.executable, str(ROOT / "bench.py"), *args], capture_output=True, text=True,
                          timeout=120)


def test_more_than_one_gpu_is_refused_with_a_message():
    r = run_bench("--gpus", "2")
    assert r.returncode == 2
    assert "one GPU" in r.stderr and r.stdout == ""


def test_unknown_secondary_is_a_usage_error():
    r = run_bench("--secondary", "config9")
    assert r.returncode == 2 and "unknown secondary config9" in r.stderr


def load_bench():
    spec = importlib.util.spec_from_file_location("bench_under_test", ROOT / "bench.py")
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    return bench


def test_the_line_is_short_whatever_the_rounds():
    bench = load_bench()
    systems = ("contiguous", "paged-gather", "paged-direct", "paged-direct-graph", "contiguous-direct",
               "contiguous-direct-graph")
    pairs = [f"{a}_minus_{b}" for a in systems for b in systems]
    deltas = {p: {"per_round_delta_ms": [0.123456] * 21, "mean_delta_ms": -0.0012, "ci95_ms": [-0.0012, 0.0012]}
              for p in pairs}
    contexts = ("16", "64", "256", "1024")
    secondary = {
        "config1_e2e_decode": {
            "summary": {s: {"decode_median_ms": 27.0671} for s in systems}, "paired_deltas": deltas,
            "tokens_identical": True, "rounds": 21, "placement_sampled": True,
            "cpu": {"summary": {s: {"decode_median_ms": 27.0671} for s in systems[:2]}, "torch_threads": 16,
                    "cpu_model": "AMD EPYC 9575F 64-Core Processor", "tokens_equal_gpu": True},
            "parity": {"engine_cache": "paged-direct", "max_abs_logit_diff": 0.0003662109375,
                       "max_rel_logit_diff": 7.314807589864358e-05, "greedy_tokens_compared": 64,
                       "first_greedy_mismatch": None, "tokens_equal_reference_engine": True}},
        "config1_context_sweep": {"median_step_ms": {s: {c: 2.0942 for c in contexts} for s in systems},
                                  "paging_cost_ms": {c: deltas for c in contexts}, "rounds": 21,
                                  "placement_sampled": True},
        "config3_append_gather": {"cells": [deltas] * 3},
    }
    roofline = {"bound": "hbm", "kernel": "k" * 120, "achieved": 6451.2, "peak": 8000.0, "unit": "GB/s", "frac": 0.8064,
                "traffic": 786338398, "algorithmic_bytes_per_launch": 785196504, "avg_duration_us": 121.71,
                "median_duration_us": 122.08, "duration_source": "d" * 170}
    main_res = {"value": 6436.123, "ms_per_step": 0.12204, "partition_tokens": 8192, "attn_bytes": 785000000,
                "append_bytes": 393216, "roofline": roofline}
    cpu = {"value": 15.775, "unit": "GB/s", "cores": 16, "kind": "port", "sample": "s" * 200, "ms_per_pass": 5.24}
    args = types.SimpleNamespace(steps=20, warmup=5)
    text = bench.result_line(args, main_res, cpu, secondary, 255385)
    assert "\n" not in text and len(text) <= bench.LINE_LIMIT
    line = json.loads(text)
    assert {"metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
            "vs_baseline", "dtype", "data", "config", "roofline", "cpu_baseline", "per_token_decode_ms"} == line.keys()
    assert line["per_token_decode_ms"]["paged-direct"] == 27.0671
    assert len(bench.result_line(args, main_res, None, {}, 255385)) <= bench.LINE_LIMIT


def test_cpu_baseline_reports_its_sample():
    bench = load_bench()
    from moe_engine import workloads

    w = workloads.make_workload([40, 7, 0, 100, 16, 3, 64, 1, 33], block_size=16, dtype=torch.bfloat16, seed=2,
                                device="cpu")
    res = bench.cpu_baseline(torch, w, 0.05)
    assert res["kind"] == "port" and res["unit"] == "GB/s"
    assert res["value"] > 0 and res["cores"] == torch.get_num_threads()
    # every 8th sequence: 0 and 8
    assert "sequences [0, 8]" in res["sample"] and "73 tokens" in res["sample"]
    assert res["ms_per_pass"] > 0
