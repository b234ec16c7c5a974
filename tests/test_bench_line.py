"""bench.py's printed line: the contract's keys, unrounded, in a line short enough
to be read back whole, from a record with everything in it."""
import importlib.util
import json
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def load():
    spec = importlib.util.spec_from_file_location("bench", ROOT / "bench.py")
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


def record():
    x = 12345678901.234567
    batch = {"DOF-updates/s": x, "seconds": x, "device_seconds": x, "device_bytes": 18386431248,
             "tile_shapes": [{"p": p, "candidate": 5, "epb": 1, "us_per_launch": x, "us_default": x}
                             for p in range(4)], "bytes_per_dof_update": 64}
    line = {k: x for k in ("value", "ms_per_step")}
    line.update(metric="DOF-updates/s plain FP64 vs batched mixed-prec; p50/p99 solve latency",
                unit="DOF-updates/s", n_gpus=1, steps=200, warmup=10, higher_is_better=True,
                scaling="weak", vs_baseline=None, dtype="f64",
                data="synthetic (seeded Gaussian blob, seeded constant velocity)",
                config={"workload": "32^3 periodic hexahedra, p=7, 16777216 DOF, SSP-RK3 steps, "
                                    "plain FP64", "NeX": 32, "p": 7, "dof": 16777216, "dt": x,
                        "form": "HIP"},
                roofline={k: x for k in ("achieved", "peak", "frac", "traffic", "traffic_GBs",
                                         "kernel_trace_avg_us", "avg_launch_us", "launches",
                                         "algorithmic_bytes_per_launch", "copy_GBs", "stream_GBs",
                                         "stream_regs_GBs")},
                cpu_baseline={"value": x, "unit": "DOF-updates/s", "cores": 16, "kind": "reference",
                              "sample": "s" * 250, "runs": [x] * 3,
                              "one_core": {"value": x, "steps": 12},
                              "port_same_inputs": {"value": x, "cores": 16, "steps": 12}})
    line["roofline"].update(bound="hbm", unit="GB/s", timing="t" * 120, kernel="k" * 60,
                            autotune_us_per_launch=[x] * 7)
    be = {"instances": 512, "nstep": 50, "HIP": batch, "HIP_MP": batch,
          "per_instance_mp_vs_fp64": {"max_rel_l2": x, "note": "n" * 200},
          "decomposition_p7": {"d" * 80 + str(k): x for k in range(7)},
          "speedup_batched_mp_vs_plain_fp64_p7": x}
    be.update({f"batched_{f}_p7{v}": batch for f in ("HIP", "HIP_MP") for v in ("", "_velocity_fields")})
    per_order = [{"p": p, "form": f, "ne": 128, "dof": 16777216, "avg_launch_us": x,
                  "tile_candidate": 1, "elements_per_workgroup": 16, "DOF-updates/s": x, "alg_GBs": x,
                  "frac_hbm": x, "useful_TFLOPs": x, "frac_mfma_peak": x}
                 for p in range(1, 20) for f in ("HIP", "HIP_MP")]
    burst = {"requests": 60, "DOF-updates/s": x, "makespan_s": x, "p50_latency_s": x, "p99_latency_s": x}
    sv = {"requests": 150, "rate_per_s": 6.0, "seed": 5, "p50_latency_s": x, "p99_latency_s": x,
          "DOF-updates/s": x, "makespan_s": x, "by_class": {}, "server": {}, "capacity_burst": burst,
          "sample_vs_alone": {"checked": 150, "all_same_as_alone": True, "max_rel_l2_1e-5_class": x,
                              "max_rel_fp64_class": x,
                              "requests": [{"request": k, "rel_l2_vs_fp64": x} for k in range(150)]}}
    line["extra"] = {"q_minmax_after": [x, x], "device_timers": {str(k): [x, 600] for k in range(5)},
                     "c2_HIP_MP": {"DOF-updates/s": x, "avg_launch_us": x, "achieved_GBs": x,
                                   "ratio_vs_HIP": x},
                     "pcie_inclusive": {k: x for k in ("steps", "DOF-updates/s", "upload_s", "steps_s",
                                                       "download_s", "host_bytes")},
                     "batched_ensemble": be, "per_order": per_order, "serving": sv,
                     "c3_p15": {"workload": "w" * 60, **{f: {"DOF-updates/s": x, "ms_per_step": x,
                                                             "elements_per_workgroup": 1,
                                                             "tile_candidate": 3}
                                                         for f in ("HIP", "HIP_MP")},
                                "mp_rel_l2_vs_fp64": x, "mp_max_rel_vs_fp64": x,
                                "speedup_mp_vs_fp64": x},
                     "p50_latency_s": x, "p99_latency_s": x}
    return line


def test_line_is_short_and_keeps_the_contract():
    bench, full = load(), record()
    text = json.dumps(bench.short_line(full))
    assert len(text) < bench.MAX_LINE <= 8000, len(text)
    line = json.loads(text)
    for key in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step",
                "higher_is_better", "scaling", "vs_baseline", "dtype", "data", "config"):
        assert line[key] == full[key], key
    assert line["extra"]["p99_latency_s"] and line["roofline"]["bound"] == "hbm"
    assert set(line["extra"]["per_order_us_per_launch"]["HIP"]) == {str(p) for p in range(1, 20)}


def test_line_without_the_extra_legs():
    bench, full = load(), record()
    full["extra"] = {"q_minmax_after": [0.0, 1.0], "device_timers": {}}
    full["cpu_baseline"] = None
    assert json.loads(json.dumps(bench.short_line(full)))["value"] == full["value"]
