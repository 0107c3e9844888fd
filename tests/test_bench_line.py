"""The benchmark's derived figures and its line, without a GPU."""
import json

import bench


def test_policy_peak_prices_each_layer_at_its_instruction():
    """29-256-256-8: 7424 multiply-adds in f32, 67584 as six bf16 products; a
    net below 32 neurons runs in f32 throughout."""
    want = (7424 + 67584) / (7424 / 157.3 + 6 * 67584 / 2516.6)
    assert abs(bench.policy_peak_tflops(29, 256, 8) - want) < 1e-9 and 300 < want < 420
    assert abs(bench.policy_peak_tflops(29, 16, 8) - 157.3) < 1e-9


def _full(name):
    kernel = {k: 123456 for k in ("vgpr", "agpr", "sgpr", "scratch_bytes", "block", "max_steps_per_launch", "lanes_per_world")}
    roof = {"bound": "valu", "achieved": 12.3456, "peak": 157.3, "unit": "TFLOP/s", "frac": 0.07849, "launch_ms": 1.2345,
            "traffic": 12345678, "flops_per_world_step": 1234}
    return {"value": 12345678901.2, "unit": "world-steps/s", "dtype": "f32", "ms_per_step": 0.012345, "finite_worlds": 1.0,
            "gpu_over_cpu": 1234.5, "roofline": roof, "cpu_baseline": {"value": 123456.7, "sample": "x" * 200},
            "event_ms_per_span": [1.2345] * 7, "kernel": kernel, "config": {"workload": name, "note": "x" * 200},
            "parity": {"pass": True, "qdd_rel_err_max": 1.234e-5}, "io": {"load_span_readback_ms": 1.234, "more": "x" * 100}}


def test_line_is_short_and_keeps_the_contract():
    """A reader that keeps the last few thousand characters gets the whole line."""
    contract = {"metric": "m", "value": 1.0, "unit": "u", "n_gpus": 1, "steps": 20, "warmup": 5, "ms_per_step": 0.1,
                "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f32", "data": "synthetic",
                "config": {"workload": "chain7"}}
    sweep = [{"dtype": d, "nworld": 1024 << k, "world_steps_per_s_event": 1.23456789e10, "more": "x" * 300}
             for d in ("f32", "f64") for k in range(9)]
    roof = {"achieved": 1.234, "peak": 360.0, "frac": 0.1234, "launch_ms": 0.12345, "kernel": {"vgpr": 1}}
    line = {**contract, "configs": {n: {"config": {}, "f32": _full(n), "f64": _full(n)} for n in "abcde"},
            "terrain_impulse": _full("t"), "mjcf": {n: _full(n) for n in "abc"}, "world_sweep": sweep,
            "control_loop": {"world_steps_per_s": 1.0, "rollout_ms": {"median": 10.0}, "physics_only_ms": 1.8,
                             "policy_roofline": roof, "obs_roofline": roof, "parity": {"obs": 1e-7}},
            "ppo_update": {**_full("p"), "parity": {"rows": 1}}}
    out = bench.brief_line(line)
    assert all(out[k] == v for k, v in contract.items())
    assert out["configs"]["a"]["f64"]["parity"] == "pass" and out["world_sweep"]["f64"]["1024"] == 1.235e10
    assert len(json.dumps(line)) > 12000 and len(json.dumps(out)) < 6000
