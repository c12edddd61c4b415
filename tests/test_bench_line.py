"""The benchmark's printed line: one JSON object that fits the last 8 KB of the output with its
progress lines, whatever the length of the report's launch lists."""
import json

import pytest

import bench

LAUNCHES = [[f"fast_rows_tr R{n} c32*H>c16 merged", 0.03641234567, 151519232] for n in range(64)]
ROOF = {"bound": "hbm", "achieved": 3706.8, "peak": 8000.0, "unit": "GB/s", "frac": 0.4633, "traffic": 135008570,
        "traffic_source": "t" * 80, "kernel": "pass 0: onchip (R=65536, lines/tile=1, c16 in / c16 out)",
        "algorithmic_bytes_per_launch": 134217728, "avg_launch_ms": 0.03621, "launch_time": "t" * 130,
        "copy_gbs": 4999.7, "frac_of_copy": 0.7414, "same_size_copy": {"us": 19.46, "timing": "t" * 60},
        "frac_of_same_size_copy": 0.5375, "launches": LAUNCHES}
CPU = {"value": 4.944814810989007, "unit": "GFLOP/s", "cores": 1, "kind": "port", "sample": "t" * 160,
       "all_cores": {"value": 12.725430016036412, "unit": "GFLOP/s", "cores": 16}, "host_cpu": "AMD EPYC"}
CONTRACT = {"metric": "m" * 80, "value": 37026.46, "unit": "GFLOP/s", "n_gpus": 1, "steps": 200, "warmup": 20,
            "ms_per_step": 0.03625, "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
            "dtype": "fp16", "data": "synthetic: " + "t" * 60, "config": {"workload": "t" * 60, "shape": [65536],
                                                                          "batch": 256, "io": "c16 in / c16 out"}}


def config():
    return {"workload": "t" * 260, "value": 27571.3, "unit": "GFLOP/s", "ms_per_exec": 0.2434, "steps": 200,
            "precision": "t" * 50, "rel_l2": 0.00029357811921128024, "rel_max": 0.00044924146483123033,
            "passes": LAUNCHES, "pass_avg_ms": [0.05840711116790771, 0.06326711654663086], "roofline": dict(ROOF),
            "plain_fp32": {"gflops": 14784.0, "ms_per_exec": 0.45393, "rel_l2": 1.5463333209113838e-07},
            "ratio_vs_plain_fp32": 1.865, "comparators": {"a": LAUNCHES}, "cpu_baseline": dict(CPU)}


def report():
    mode = {"p50_ms": 0.0482, "p99_ms": 0.3303, "req_per_s": 2002.0, "gflops": 1373.0, "launches": 61478,
            "saturation_req_per_s": 31150.2, "coalesced": 14271, "paired": 298, "peak_bytes": 68719474688}
    return dict(CONTRACT, rel_l2=0.000293280114516455, passes=LAUNCHES, pass_timing="t" * 120, schedule={"a": 1},
                settle="t" * 200, roofline=dict(ROOF), cpu_baseline=dict(CPU), mfma=[{"kernel": "onchip", "frac": 0.2}],
                comparators={k: {"gflops": 14026.265718196986, "ms_per_exec": 0.095690279006958, "rel_l2": 1.39e-07,
                                 "timing": "t" * 100, "pass_timing": "t" * 200, "launches": LAUNCHES}
                             for k in "abcdef"},
                reference_api={"tcfftExec": {"ms_per_exec": 0.03201, "gflops": 41929.6, "accuracy_sample": "t" * 80},
                               "doit": {"ms_per_exec": 0.03358, "ok": True, "timing": "t" * 100}},
                configs={k: config() for k in ("c1", "c3", "c4")},
                serve={"workload": "t" * 110, "requests": 60057, "split": dict(mode), "plain_fp32": dict(mode),
                       "equal_p99": {"p99_bound_ms": 2.0, "probes": LAUNCHES, "ratio": 3.445,
                                     "sustained_req_per_s": {"split": 26515.8, "plain_fp32": 7697.7}}})


def test_printed_line_fits(capsys, tmp_path):
    whole = report()
    bench.emit(whole, str(tmp_path / "report.json"))
    out = capsys.readouterr().out
    assert out.count("\n") == 1 and len(out) < 6144
    line = json.loads(out)
    for k, v in CONTRACT.items():
        assert line[k] == v
    for part in [line] + list(line["configs"].values()):
        assert part["value"] and part["roofline"]["frac"] == ROOF["frac"] and part["cpu_baseline"]["value"] > 0
    assert line["serve"]["split"]["p99_ms"] == 0.3303 and line["serve"]["equal_p99"]["ratio"] == 3.445
    assert json.loads((tmp_path / "report.json").read_text()) == whole


@pytest.mark.parametrize("part", ["conv", "serve"])
def test_single_workload_lines(capsys, part):
    whole = report()
    bench.emit(dict(CONTRACT, **{part: config() if part == "conv" else whole["serve"]}), None)
    line = json.loads(capsys.readouterr().out)
    assert line["value"] == CONTRACT["value"] and line[part]
