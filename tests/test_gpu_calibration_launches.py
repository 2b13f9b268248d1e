"""Calibration runs with fewer launches: the gauges of a frozen run ride on the
next step, the edge cotangents of a reverse step are gathered by the next
step's update.  Both must leave the bits of the separate launches."""
import numpy as np
import pytest
import torch

from hipims_amd import generators as gen
from hipims_amd.adjoint import Calibration
from hipims_amd.grid import GridSolver

pytestmark = pytest.mark.gpu


def solver(dtype, order, n=70):
    c = gen.rainfall_runoff(n, 5.0, seed=99, rain_mmh=150.0, relief=8.0)
    s = GridSolver(c.mask, c.h, c.qx, c.qy, c.z, c.dx, cfl=0.5, order=order, dtype=dtype, first_dt=0.5,
                   manning=c.manning, landuse=c.landuse)
    s.set_station_rain(c.rain_table)
    return s


def gauges_of(s, n):
    rng = np.random.Generator(np.random.PCG64(n))
    valid = np.argwhere(s.raster(s.landuse) != 255)
    return valid[rng.choice(len(valid), size=n, replace=False)]


@pytest.mark.parametrize("ck", [1, 4, 9])
@pytest.mark.parametrize("n_gauges", [1, 64, 65, 130])
def test_frozen_run_records_the_recorded_runs_depths(cuda, n_gauges, ck):
    s = solver(torch.float64, 2)
    cal = Calibration(s, gauges_of(s, n_gauges), 9, ck, obs=torch.zeros(10, n_gauges))
    th = cal.theta0()
    cal.run(th)
    first = cal.hist.clone()
    cal.hist.fill_(-1.0)
    cal.run(th)
    assert torch.equal(cal.hist, first)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("steps", [1, 2, 7])
def test_gather_in_the_next_update_changes_no_bits(cuda, dtype, order, steps):
    res = []
    for defer in (True, False):
        s = solver(dtype, order)
        cal = Calibration(s, gauges_of(s, 20), steps, 1, obs=torch.zeros(steps + 1, 20), reverse="separate")
        if not defer:
            cal.adesc.gauge_of = None  # the loss by a kernel of its own, after the gather
        cal.run(cal.theta0())
        g = cal.gradient()
        assert g.abs().max() > 0
        res.append([g] + [t.clone() for t in cal.lam])
    for a, b in zip(*res):
        assert torch.equal(a, b)
