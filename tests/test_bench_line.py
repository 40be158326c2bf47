"""The benchmark's printed line: what it keeps, and that it stays short."""
import json

import bench


def _entry(config, qtype, m, k, n, gemm):
    roofline = {"bound": "hbm", "achieved": 4001.2, "peak": 8000.0, "unit": "GB/s", "frac": 0.5001, "algorithmic_bytes": 1}
    e = {"config": config, "qtype": qtype, "m": m, "k": k, "n": n, "us": 100.123, "gbps": 4001.2, "roofline": roofline,
         "cpu_baseline": {"unit": "GB/s", "scalar": 0.2, "sample": "x" * 150}}
    return dict(e, f32_mode={"us": 56.2}) if gemm else e


def test_printed_line_is_short_and_keeps_its_values():
    """With every configs point and embedded objects of their usual size the
    line takes less than 8000 characters (its log keeps that many), and the
    contract's fields, times and rates are unchanged."""
    points = {"gemv": bench.GEMV_POINTS, "gemv_row_major": bench.RM_POINTS, "gemm": bench.GEMM_POINTS}
    configs = {kind: [_entry(c, bench.QNAME[q], m, k, n, kind == "gemm") for c, q, k, n, ms in pts for m in ms]
               for kind, pts in points.items()}
    configs.update(device="d", note="x" * 600)
    nested = {"metric": "m" * 50, "value": 829.14, "unit": "TFLOP/s", "n_gpus": 1, "steps": 50, "warmup": 20,
              "ms_per_step": 0.24864, "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
              "dtype": "f16 operands, f32 accumulation", "data": "x" * 100, "note": "x" * 150,
              "config": {"workload": "w" * 45, "m": 2048, "k": 4096, "n": 12288, "device": "d" * 30, "step": "s" * 50},
              "roofline": {"bound": "mfma", "achieved": 829.14, "peak": 2500.0, "unit": "TFLOP/s", "frac": 0.33}}
    line = dict(nested, configs=configs, gemm={"q4_k": nested, "q8_0": nested}, gemm_f32={"q4_k": nested},
                gemv_q8_0=dict(nested, cpu_baseline={"scalar": 1.9, "sample": "x" * 200}), f32_matmul_head=nested,
                e2e=dict(nested, dtype="x" * 60, detail="x" * 900), through_abi={"value": 1249.8, "note": "x" * 150},
                cpu_baseline={"value": 0.2, "sample": "x" * 200})
    short = bench.short_line(line)
    assert len(json.dumps(short, separators=(",", ":"))) < 8000
    for key in nested:
        assert short[key] == line[key]
    assert short["gemm"]["q4_k"]["value"] == 829.14 and short["gemm"]["q4_k"]["roofline"] == nested["roofline"]
    assert short["configs"]["gemv"][0] == [0, "q8_0", 1, 4096, 4096, 100.123, 0.5001]
    assert {kind: len(rows) for kind, rows in short["configs"].items()} == {k: len(v) for k, v in configs.items()
                                                                           if k in points}
