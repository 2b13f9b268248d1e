"""bench.py's single-pass timing says what it measured: the step time (a folded
step is one launch) as the kernel's, and the events around single launches,
which also hold a launch's dispatch, as a figure of their own."""
import ctypes
import types

import pytest
import torch

from hipims_amd import _lib
from test_bench_cpu import bench  # noqa: F401  (the module under test)

CELLS = 2048 * 2048


def timed(bench, monkeypatch, kernel_ms, total_ms, steps):  # noqa: F811
    class Lib:
        @staticmethod
        def hp_grid_step_fused_timed(desc, n, every, k, t, stream):
            k._obj.value, t._obj.value = kernel_ms, total_ms
            return 0

    monkeypatch.setattr(_lib, "lib", lambda: Lib)
    monkeypatch.setattr(_lib, "stream_ptr", lambda dev: None)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: None)
    g = types.SimpleNamespace(ensure_out=lambda: None, step_fused=lambda n: None, desc=ctypes.c_int(0), device=None)
    return bench.time_fused(g, steps)


@pytest.mark.parametrize("kernel_ms", [0.0645, 0.0545])
def test_sampled_launches_and_mean_step_are_separate(bench, monkeypatch, kernel_ms):  # noqa: F811
    out = timed(bench, monkeypatch, kernel_ms, 60.25, 1000)
    mean = out["total_ms"] / 1000
    assert out["kernels_ms"] == {"k_step_fused": pytest.approx(mean, rel=1e-12)}
    assert out["sampled_launch_ms"] == pytest.approx(kernel_ms, rel=1e-6)
    per_kernel, r = bench.roofline_fields(out["kernels_ms"], mean, 4, False, CELLS, "rainfall_runoff_2048_fp32_order2",
                                          timed_with=out["timed_with"])
    assert r["kernel_ms"] == mean and "mean" in r["timed_with"] and "events around the kernel" not in r["timed_with"]
    assert set(per_kernel) == {"k_walk_step"}


def test_two_pass_keeps_its_label(bench):  # noqa: F811
    _, r = bench.roofline_fields({"k_flux": 0.20, "k_update": 0.05}, 0.26, 8, False, CELLS,
                                 "rainfall_runoff_2048_fp64_order2")
    assert r["timed_with"] == "HIP events around the kernel of every tenth timed step"
