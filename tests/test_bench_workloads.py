"""bench.py's table of streaming-operator workloads: names and oracle passes (host side only, no GPU)."""
import os
import sys

import torch

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench
from oracle import quant_ref as q, bitpack_ref as bp


def test_stream_workload_table_is_complete():
    ops = bench._stream_ops()
    assert set(ops) == set(bench.STREAM_WORKLOADS) and len(bench.STREAM_WORKLOADS) == len(set(bench.STREAM_WORKLOADS))
    assert all(name.startswith("stream_") for name in ops)
    assert not set(ops) & (set(bench.WORKLOADS) | set(bench.MOE_WORKLOADS))


def test_stream_workload_oracle_passes_run_on_host_inputs():
    """Every oracle pass of the table accepts host tensors shaped like its operator's device inputs (2048 rows
    here; the pass itself takes the first 1024)."""
    torch.manual_seed(0)
    ops = bench._stream_ops()
    N, K = 2048, 512
    x, w = torch.randn(N, K).bfloat16(), torch.randn(N, K) * 0.02
    nib = torch.randint(0, 16, (N, K), dtype=torch.uint8)
    yf, sf = q.weight_quant_fp8(w)
    yi, si = q.weight_quant_int8(w)
    qq, s, s4, z4 = q.w4a8_weight_quant_levels(w.half())
    as_t = lambda a: torch.from_numpy(a)
    host = {
        "stream_act_quant_fp8": (x,), "stream_act_quant_int8": (x,), "stream_act_quant_int8_per_token": (x,),
        "stream_weight_quant_fp8": (w,), "stream_weight_quant_int8": (w,),
        "stream_weight_dequant_fp8": (yf, sf), "stream_weight_dequant_int8": (yi, si),
        "stream_weight_dequant_w4a8": (as_t(bp.pack_rows(qq.numpy(), 4, 32)[0]), s, s4, z4),
        "stream_quantize_w4a16_nk": (w.half(),),
        "stream_pack_rows_4in32": (nib,), "stream_pack_cols_4in32": (nib,),
        "stream_unpack_rows_4in32": (as_t(bp.pack_rows(nib.numpy(), 4, 32)[0]),),
        "stream_unpack_cols_4in32": (as_t(bp.pack_cols(nib.numpy(), 4, 32)[0]),),
        "stream_silu_and_mul": (torch.randn(N, 256).bfloat16(), torch.sort(torch.randint(0, 8, (N,)))[0]),
    }
    assert set(host) == set(ops)
    for name, args in host.items():
        assert ops[name][2](*args) is not None, name


def _record(name, unit):
    """A record of the form bench.record() returns, every number as long as it gets."""
    return {"workload": name, "M": 4096, "N": 128256, "K": 14336, "us_per_launch": 12345.67, "us_per_launch_min": 12345.67,
            "us_per_launch_max": 12345.67, "timed_replays": 7, "preroll_ms": 1234.5, "preroll_replays": 12345,
            "cache_flushed_before_each_replay": True, "us_per_launch_without_flush": 12345.67, "tflops": 12345.67, "gbs": 12345.6,
            "alg_bytes": 10 ** 12, "flops": 1.234567890123456e+16, "weight_copies_rotated": 123, "wall_ms_per_step": 1234.5678,
            "roofline": {"bound": "mfma", "achieved": 12345.6, "peak": 5000.0, "unit": unit, "frac": 0.1234, "traffic": 10 ** 12},
            "cpu_baseline": {"value": 12.3456, "unit": unit, "cores": 16, "kind": "port", "cpu_model": "x" * 60, "sample": "x" * 250,
                             "matmul_only_value": 12.3456}}


def test_the_printed_line_fits_what_a_reader_keeps():
    """The longest default run and the longest run of the streaming operators, and the keys a reader looks for."""
    import json
    head = {"metric": "m" * 80, "value": 12345.67, "unit": "TFLOP/s", "n_gpus": 1, "steps": 20000, "warmup": 20000,
            "ms_per_step": 12.34567, "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "fp8_e4m3",
            "data": "synthetic", "config": {"k%d" % i: "v" * 20 for i in range(20)}}
    calib = {"a_name_of_the_usual_length_of_a_rate_%d" % i: 12345.6 for i in range(16)}
    for names, unit in ((bench.HEADLINE_SET, "TFLOP/s"), (bench.STREAM_WORKLOADS, "GB/s")):
        r = _record(names[0], unit)
        out = dict(head, roofline=r["roofline"], cpu_baseline=r["cpu_baseline"], calibration=calib,
                   cases=[_record(n, unit) for n in names])
        line = bench.result_line(out)
        assert len(line) < bench.MAX_LINE and "\n" not in line
        got = json.loads(line)
        assert all(got[k] == v for k, v in head.items()) and got["roofline"] == r["roofline"]
        assert [c["workload"] for c in got["cases"]] == list(names)
        assert all(c["us"] == 12345.67 and c["unit"] == unit and c["frac"] == 0.1234 for c in got["cases"])
