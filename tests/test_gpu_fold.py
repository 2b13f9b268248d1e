"""Calls of several single-pass steps fold the time control into the step
kernel; the same steps one call each run it in launches of its own.  Both must
leave the same bits: state, time control, export and stop handling, mass sums."""
import numpy as np
import pytest
import torch

from helpers import random_state
from hipims_amd import _lib
from hipims_amd.grid import GridSolver

pytestmark = pytest.mark.gpu


def solver(ny, nx, dtype, sums, **kw):
    z, h, qx, qy = random_state(ny, nx, seed=ny + nx, rough=0.1)
    pad = lambda a, v: np.pad(a, 1, constant_values=v)  # noqa: E731
    s = GridSolver(pad(np.full((ny, nx), 40), -9999), pad(h, 0.0), pad(qx, 0.0), pad(qy, 0.0), pad(z, 0.0), 1.0,
                   order=2, dtype=dtype, first_dt=0.01, manning=[0.03], mass_sums=sums, **kw)
    s.set_station_rain(np.array([[0.0, 1e-4], [0.2, 3e-4], [1e6, 1e-4]]))
    return s


def state(s):
    torch.cuda.synchronize()
    return [getattr(s, k).clone() for k in ("h", "qx", "qy", "h_max")] + [s.ctrl[: _lib.CTRL_STOPPED_SYNCED + 1].clone()]


@pytest.mark.parametrize("sums", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("ny,nx", [(1, 1), (5, 130), (70, 61), (700, 640)])
def test_folded_call_equals_single_steps(cuda, ny, nx, dtype, sums):
    a, b = solver(ny, nx, dtype, sums, t=1.0), solver(ny, nx, dtype, sums, t=1.0)
    for n in (3, 4, 7, 2, 5):
        a.step_fused(n)
        for _ in range(n):
            b.step_fused(1)
        for x, y in zip(state(a), state(b)):
            assert torch.equal(x, y), n
    assert a.ctrl_dict()["steps"] == 21


@pytest.mark.parametrize("sums", [True, False])
def test_stop_and_export_inside_a_call(cuda, sums):
    """An export time and the stop time are reached inside the call."""
    for n in (4, 12, 13):
        kw = dict(export_T=0.05, t_stop=0.3)
        a, b = solver(40, 70, torch.float32, sums, **kw), solver(40, 70, torch.float32, sums, **kw)
        for _ in range(3):
            a.step_fused(n)
            for _ in range(n):
                b.step_fused(1)
            for x, y in zip(state(a), state(b)):
                assert torch.equal(x, y), n
        assert a.t >= 0.3 and a.ctrl_dict()["export_n"] >= 2


def test_folded_call_under_graph_replay(cuda):
    a, b = solver(60, 200, torch.float32, True, t=1.0), solver(60, 200, torch.float32, True, t=1.0)
    a.step_fused(2)
    b.step_fused(2)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        a.step_fused(6)
    for _ in range(4):
        g.replay()
        b.step_fused(6)
        for x, y in zip(state(a), state(b)):
            assert torch.equal(x, y)
