"""bench.py's result line, checked without a GPU."""
import argparse
import json
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)

import bench  # noqa: E402


def _roofline(kernel):
    f = dict(kernel=kernel, bound="mfma", achieved=1012.3, peak=2500.0, unit="TFLOP/s", frac=0.4049, traffic=2062736411.0,
             algorithmic_flops_per_launch=981040431104.0, us_per_launch=1087.84, mfma_busy_pct_counters=36.93)
    f["vendor_gemm"] = dict(shape_mnk=[4096, 28672, 4096], TFLOPs=1215.5, frac_of_peak=0.4862, kernel_frac_of_vendor=0.8329)
    return f


def test_result_line_fits_the_kept_end_of_the_output(capsys):
    """Readers keep the last 8 KB of the output and take its JSON line: with a
    record of every workload the bench runs, the line is one JSON object under
    that, and the full records on stderr are not JSON lines by themselves."""
    shape = {k: v for k, v in bench.QWEN3_INT4.items()}
    head = bench.Workload("qwen3_30b_a3b_moe_layer_int4_g128_decode", tokens=16, **shape)
    res = dict(tokens_per_s=315123.456789, ms_per_step=0.0507712345, us_per_layer=50.7712345, mean_active_experts=83.125,
               layer_hbm_frac=0.5123456789, breakdown_us={k: 12.3456789 for k in ("route+group", "gate_up", "down", "combine")})
    r = dict(res, workload="qwen3_30b_a3b_moe_layer_int8_pc_prefill_zipf", tokens=4096, probe="qwen3_int8", steps=400,
             warmup=40, roofline=_roofline("gemm2_i8_kernel (gate_up, int8_per_channel, T=4096)"),
             roofline_alt=_roofline("gemm2_i8_kernel (gate_up, int8_per_channel, T=4096)"))
    c = dict(workload=r["workload"], tokens=4096, value=4040.002, unit="tokens/s", cores=16, kind="port", median_s=0.25347,
             min_s=0.24981, cpu_model="x" * 60, sample="x" * 300)
    line = bench.result_line(head, argparse.Namespace(steps=400, warmup=40, tokens=16, layers=8), res,
                             _roofline("gemv_kernel (gate_up, int4_g128, T=16)"), [c] * 13, [r] * 14)
    text = json.dumps(line)
    assert len(text) < 6500, len(text)
    for key in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
                "vs_baseline", "dtype", "data", "config", "roofline", "cpu_baseline"):
        assert key in line
    bench.detail(r)
    for out in capsys.readouterr().err.splitlines():
        assert not out.startswith("{")


def test_counter_rows_join_the_kernel_that_they_were_taken_on():
    """A counter row goes beside a kernel's time only if it was taken on that
    kernel's present form; every committed row is."""
    table = bench.counter_table()
    assert table
    for key, row in table.items():
        phase = key.split(":")[2].replace("shared_", "").replace("_layer_call", "")
        name = row["kernel"].split("::")[1].split("<")[0]
        assert bench.counters_apply(row, name, phase), key
        assert not bench.counters_apply(row, name, "down" if phase == "gate_up" else "gate_up")
    assert not bench.counters_apply({"kernel": "nkt::gemm2_i4_kernel<0, false>"}, "gemm2_i4_kernel", "gate_up")
    assert not bench.counters_apply({"kernel": "nkt::gemm2_kernel<1, 0, 8>"}, "gemm2_kernel", "gate_up")
    assert not bench.counters_apply({}, "gemv_kernel", "gate_up")
