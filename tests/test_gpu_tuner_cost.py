"""The height tuner's own cost: one timed round over its choices, after warm-up
work of at most as much; it leaves the domain as it found it."""
import pytest
import torch

from hipims_amd import autotune
from hipims_amd.grid import GridSolver
from test_gpu_fold import solver, state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("path", ["flux", "fused"])
def test_tuning_work_is_bounded_and_leaves_the_state(cuda, monkeypatch, path, dtype):
    s = solver(300, 200, dtype, True, t=1.0)
    s.step(2)
    s.step_fused(2)
    before = state(s) + [s.D.clone()]
    done = {"step_fused": 0, "flux": 0}

    def counted(name, work):
        real = getattr(GridSolver, name)

        def run(self, *a):
            done[name] += work(*a)
            return real(self, *a)
        monkeypatch.setattr(GridSolver, name, run)

    counted("step_fused", lambda n=1: n)
    counted("flux", lambda: 1)
    monkeypatch.setattr(autotune, "_cache", {})
    best = autotune.tune(s, reps=20, apply=False, path=path)
    choices = autotune.CHOICES[dtype]
    assert best in choices and set(s.tune_timings) == set(choices) and s.tile_rows == 0
    # a choice is run untimed once (four steps, or one pass) and timed over 40 steps or 20 passes
    one_round = len(choices) * (4 + 40 if path == "fused" else 1 + 20)
    assert 0 < done["step_fused" if path == "fused" else "flux"] <= 2 * one_round
    for a, b in zip(before, state(s) + [s.D]):
        assert torch.equal(a, b)
