"""A CFL number of zero, of either sign, gives the same time control in calls
that fold it into the step kernel and in calls of single steps: the folded
minimum orders doubles by their bits, where a negative zero would count as the
largest number."""
import pytest
import torch

from hipims_amd.ensemble import Ensemble
from test_gpu_fold import solver, state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("cfl", [0.0, -0.0])
def test_folded_call_equals_single_steps(cuda, dtype, cfl):
    a, b, c, d = (solver(5, 130, dtype, True, t=1.0, cfl=cfl) for _ in range(4))
    a.step_fused(4)
    for _ in range(4):
        b.step_fused(1)
    Ensemble([c]).step(4)
    e = Ensemble([d])
    for _ in range(2):
        e.step(2)
    for s in (a, c, d):
        for x, y in zip(state(s), state(b)):
            # (a step of length zero is no number in double; those compare as equal)
            torch.testing.assert_close(x, y, rtol=0.0, atol=0.0, equal_nan=True)
