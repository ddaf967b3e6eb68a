"""CPU checks of bench.py's command line: the benchmark measures one GPU, so a
request for several exits with a message before any device work, and the result
line of a whole run stays short enough for a reader that keeps 16 KB of output."""
import json
import subprocess
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_more_than_one_gpu_is_refused():
    res = subprocess.run([sys.executable, str(ROOT / "bench.py"), "--gpus", "2", "--steps", "1", "--warmup", "0"],
                         capture_output=True, text=True, timeout=120)
    assert res.returncode == 2
    assert "one GPU only" in res.stderr
    assert res.stdout == ""


def test_help_lists_the_driver_flags():
    res = subprocess.run([sys.executable, str(ROOT / "bench.py"), "--help"], capture_output=True, text=True,
                         timeout=120)
    assert res.returncode == 0
    for flag in ("--gpus", "--steps", "--warmup"):
        assert flag in res.stdout


def test_result_line_is_short():
    import bench
    shape = {"I": 4096, "N": 12288, "K": 6}
    timed = {"us": 1234.567, "median_pass_us": 1234.567, "passes": 11, "launches": 3, "rotation_copies": 128,
             "timed_steps": 4096, "replay_matches_eager": False, "packed_GBps": 12345.6, "pct_hbm_peak": 12.3,
             "call_floor_us": 123.456, "call_floor_shape": [[1024, 16, 4096], [1024, 16, 4096]],
             "call_floor_launches": "gate/up bytes, then down bytes, each in its fastest shape",
             "pct_call_floor": 12.3, "pct_read_ceiling": 12.3, "fp16_library_us": 1234.567,
             "fp16_library_pct_peak": 12.3, "speedup_vs_fp16_library": 12.34, "TFLOPs": 1234.5, "pct_fp16_peak": 12.3}
    products = ("TFLOPs", "pct_fp16_peak", "fp16_library_pct_peak")
    gemv = {**shape, "R": 8, **{k: v for k, v in timed.items() if k not in products}}
    head = {**gemv, "warmup_launches": 4096, "oracle_pass": True, "oracle_maxabs": 1.234e-05,
            "oracle_nrmse": 1.234e-07, "oracle_gate": "x" * 200}
    ceil = {"GBps": 6387.5, "pct_hbm_peak": 79.8, "shape": [1024, 16, 4096], "us": 168.1, "bytes": 1 << 30}
    cpu = {"kind": "port", "sample": "x" * 200, **{f"field_{i}": 123456.789 for i in range(12)}}
    grouped = {"groups": 16, "fold": "owner", **gemv}
    moe = {"experts": 64, "H": 1536, "rows": 8, "top_k": 8, "distinct_experts": 39, "packed_bytes": 1 << 28, **gemv}
    gemm = [{**shape, "M": m, **{k: v for k, v in timed.items() if "floor" not in k and k != "packed_GBps"}}
            for m in (128, 512, 2048)] * 6
    out = bench.result_line(head, ceil, cpu, [gemv] * 24, gemm, [grouped] * 16, moe, 512)
    assert out["value"] == head["packed_GBps"] and out["steps"] == 4096 and out["warmup"] == 512
    assert len(out["sweep_gemv"]) == 24 and len(out["sweep_gemm"]) == 18 and len(out["grouped_o_a"]) == 16
    assert out["cells_replay_match_eager"] is False
    assert len(json.dumps(out)) < 12000
    full = dict(out, sweep_gemv=[gemv] * 24, sweep_gemm=gemm, grouped_o_a=[grouped] * 16)
    assert len(json.dumps(full)) > 16000   # what the whole cells would take
    none = bench.result_line(head, ceil, None, [], [], [], None, 0)
    assert none["moe_k2"] is None and none["cpu_baseline"] is None and none["sweep_gemv"] == []
