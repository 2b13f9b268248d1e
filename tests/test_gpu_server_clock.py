"""A server step reads the clock with the export flag: the lists it keeps hold
what the model's t and dt hold, also around exports, and a model whose own
step method stands in for the library's is still called."""
import numpy as np
import pytest
import torch

from hipims_amd import generators as gen
from hipims_amd.server import Simulation
from hipims_amd.SWE_CUDA import Godunov

pytestmark = pytest.mark.gpu


class Wrapped(Godunov):
    calls = 0

    def time_friction_euler_update_cuda(self, device):
        self.calls += 1
        super().time_friction_euler_update_cuda(device)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("export_dt", [1.0e9, 20.0])
def test_clock_lists(cuda, tmp_path, dtype, export_dt):
    c = gen.rainfall_runoff(40, 5.0, rain_mmh=300.0, relief=3.0)
    T = lambda a: torch.as_tensor(np.asarray(a))  # noqa: E731
    sims = []
    for cls in (Godunov, Wrapped):
        out = tmp_path / cls.__name__
        out.mkdir()
        num = cls(cuda, c.dx, c.cfl, export_dt, t=0.0, export_n=0, firstTimeStep=1.0, tensorType=dtype)
        num.setOutPutPath(str(out))
        num.init__fluidField_tensor(T(c.mask), T(c.h), T(c.qx), T(c.qy), T(c.h + c.z), T(c.z), cuda)
        num.set__frictionField_tensor(c.manning, cuda)
        num.set_landuse(T(c.mask), T(c.landuse), cuda)
        num.set_distributed_rainfall_station_Mask(T(c.mask), T(np.zeros_like(c.mask)), cuda)
        num.set_boundary_tensor({}, cuda)
        sim = Simulation(num, c.rain_table, np.arange(5), cuda)
        for _ in range(12):
            sim.simulate_one_time_period()
            assert sim.t_list[-1] == num.t.item() == sim.time() and sim.dt_list[-1] == num.dt.item()
        sims.append((sim, sorted(p.name for p in out.iterdir())))
    (a, fa), (b, fb) = sims
    assert a.t_list == b.t_list and a.dt_list == b.dt_list and torch.equal(a.results, b.results)
    assert fa == fb and (len(fa) > 0) == (export_dt < 1e9)
    assert b.numerical.calls == 12
