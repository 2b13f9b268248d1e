"""An ensemble call of four steps and more folds every domain's time control
into the step kernel; calls of two steps run it in a launch of its own.  Both
must leave the same bits, as must each domain alone: domains of uneven sizes,
some without mass sums, one that stops inside a call, one stopped before."""
import pytest
import torch

from hipims_amd.ensemble import Ensemble
from test_gpu_fold import solver, state

pytestmark = pytest.mark.gpu

DOMAINS = [dict(ny=1, nx=1, sums=True), dict(ny=70, nx=61, sums=False), dict(ny=40, nx=190, sums=True, t_stop=0.2),
           dict(ny=33, nx=64, sums=True, t_stop=0.05, t=0.06), dict(ny=300, nx=257, sums=True, export_T=0.05)]


def domains(dtype, which=DOMAINS):
    return [solver(dtype=dtype, **d) for d in which]


def same(a, b, what):
    for k, (s, t) in enumerate(zip(a, b)):
        for x, y in zip(state(s), state(t)):
            assert torch.equal(x, y), (what, k)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("which", [DOMAINS, DOMAINS[1:2], DOMAINS[2:3]])
def test_folded_call_equals_calls_of_two(cuda, dtype, which):
    a, b, c = (domains(dtype, which) for _ in range(3))
    ea, eb = Ensemble(a), Ensemble(b)
    for n in (4, 6, 2, 10):
        ea.step(n)
        for _ in range(n // 2):
            eb.step(2)
        for s in c:
            s.step_fused(n)
        same(a, b, n)
        same(a, c, n)
    assert all(s.ctrl_dict()["t"] >= 0.2 for s, d in zip(a, which) if d.get("t_stop") == 0.2)


def test_folded_call_under_graph_replay(cuda):
    a, b = domains(torch.float32), domains(torch.float32)
    ea, eb = Ensemble(a), Ensemble(b)
    ea.capture(6)
    for k in range(4):
        ea.replay()
        eb.step(6)
        same(a, b, k)
        for s in a + b:  # the host writes the state between replays
            s.h *= 1.001
            s.state_written()
