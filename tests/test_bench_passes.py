"""What bench.py reports: the tables of the passes as the loops run them against the
committed counter summaries, and the printed line against the contract."""
import json
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)

import bench  # noqa: E402


@pytest.mark.parametrize("n", [4096, 8192])
@pytest.mark.parametrize("table", ["fp64", "mixed"])
def test_pass_tables_have_measured_traffic(n, table):
    """The counters see at least a pass's algorithmic bytes, and ghost rows and
    columns add under 20 %."""
    bytes_, traffic = ((bench.pass_bytes(n), bench.PASS_TRAFFIC) if table == "fp64" else
                       (bench.MIXED_PASS_BYTES, bench.MIXED_PASS_TRAFFIC))
    assert set(bytes_) == set(traffic)
    for cls, (name, bpc) in bytes_.items():
        kernel, profile = traffic[cls]
        t = bench.measured_traffic(kernel, n, profile)
        if table == "fp64" and n == 8192 and cls in (3, 4):  # profiled at 4096^2 only
            assert t is None
            continue
        assert t and bpc * n * n * 0.99 <= t <= bpc * n * n * 1.2, (name, t / (n * n), bpc)


def _record():
    """A record with every section, and in each what makes it long."""
    kernels = {f"kernel {i}": {k: 0.123456789 for k in (
        "timed_launches", "idle_launches", "avg_launch_ms", "achieved_gbs", "bytes_per_cell",
        "frac", "measured_bytes_per_launch", "measured_gbs", "measured_frac", "traffic_source")}
        for i in range(5)}
    run = {"tl_eps": 1e-10, "s_per_step": 1.23456789012, "iterations_per_step": 6179.0,
           "true_rel_residual": 9.98765432e-11, "meets_target": True, "model_gbs": 4000.123456,
           "kernels": kernels}
    comparison = {"workload": "4096x4096, seeded deck (3 rectangles + 2 circles, seed 2), more",
                  "runs": {k: dict(run) for k in bench.PRECISION_EPS}, "all_meet_target": True,
                  "second_step": {k: dict(run) for k in ("fp64_cg", "mixed_ppcg")},
                  **{f"speedup_{i}": 1.23456789 for i in range(4)}}
    adj = {"J": 0.000271103164, "forward_s_per_step": 0.98412732, "forward_backward_s_per_step":
           2.02289, "forward_iterations_per_step": 602.0, "unconverged_solves": {"max_iters": 0},
           "device_bytes": 1.6773e10, "fd_max_rel_err": 3.3e-6}
    adjoint = {"workload": "2048x2048, 20 steps, seeded deck, per-cell density rho*exp(0.1 xi)",
               "fp64": dict(adj), "mixed": dict(adj), "mixed_vs_fp64_gradient_rel_l2": 7e-10,
               "finite_differences": {"quotients": [{"cell": (1, 2), "fd": 1e-6}] * 32}}
    solver = {"s_per_step": 0.433123456, "iterations_per_step": 10000.0, "model_gbs": 1.0,
              "step_measured_frac": 0.6, "kernels": kernels, "work_launches": {"a": 1}}
    return {
        "metric": "s/timestep + HBM GB/s at 4096^2: FP64 CG vs FP32-refined PPCG @1e-10 residual",
        "value": 0.888123456789, "unit": "s/timestep", "n_gpus": 1, "steps": 20, "warmup": 5,
        "ms_per_step": 888.123456789, "higher_is_better": False, "scaling": "weak",
        "vs_baseline": None, "dtype": "f64", "data": "synthetic",
        "config": {"workload": "4096x4096 FP64 CG timestep, seeded deck, tl_eps 1e-15",
                   "cells": 4096 * 4096, "solver": "cg", "eps": 1e-15,
                   "mean_iterations_per_step": 4050.5},
        "hbm_gbs_step": 5800.0, "model_gbs_step": 7000.0, "cell_iterations_per_s": 7.6e10,
        "roofline": {"bound": "hbm", "kernel": "cg calc_w (w = A p, p = r + beta p, p.w)",
                     "achieved": 5400.123456, "peak": 8000.0, "unit": "GB/s", "frac": 0.675,
                     "traffic": 719898089.0, "traffic_source": "profiles/passes_4096.md"},
        "solvers": {k: dict(solver) for k in ("chebyshev", "ppcg", "jacobi")},
        "small": {"workload": "512x512", "s_per_step": 0.0023, "us_per_iteration": 5.2},
        "achievable_hbm": {"copy_gbs": 6110.1, "triad_gbs": 6170.1, "kernels": "hand-written"},
        "precision_comparison": [dict(comparison), dict(comparison)],
        "adjoint": adjoint, "adjoint_large": adjoint,
        "cpu_baseline": {"value": 19.4, "unit": "s/timestep", "cores": 16, "kind": "reference",
                         "sample": "x" * 300, "host": {"model": "y" * 400},
                         "one_thread": {"sample": "z" * 300}}}


def test_printed_line_is_short_and_whole():
    out = _record()
    line = json.dumps(bench.headline(out))
    assert len(json.dumps(out)) > 15000 and len(line) < 4096 and "\n" not in line
    got = json.loads(line)
    for k in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step",
              "higher_is_better", "scaling", "vs_baseline", "dtype", "data", "config", "roofline"):
        assert got[k] == out[k], k
    assert got["precision_comparison"][0]["mixed_ppcg"] == [1.23457, 9.98765e-11]
    assert got["adjoint"]["fp64"]["forward_s_per_step"] == 0.984127
    assert got["cpu_baseline"]["value"] == 19.4
    # a run with every section off
    small = {k: v for k, v in out.items() if k not in (
        "solvers", "small", "achievable_hbm", "precision_comparison", "adjoint", "adjoint_large",
        "cpu_baseline")}
    assert json.loads(json.dumps(bench.headline(small)))["value"] == out["value"]


def test_host_lines_are_set_aside(capfd):
    """What the native host prints to file descriptor 2 is not in the log, and shown
    after a failure."""
    with bench.host_lines_aside():
        os.write(2, b"Step 1 of the host\n")
        bench.log("logged")
    assert capfd.readouterr().err == "logged\n"
    with pytest.raises(RuntimeError):
        with bench.host_lines_aside():
            os.write(2, b"Error from the host\n")
            raise RuntimeError
    assert "Error from the host" in capfd.readouterr().err
    os.write(2, b"as before\n")
    assert capfd.readouterr().err == "as before\n"
