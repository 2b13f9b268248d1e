"""The compact flux op where its neighbour table runs out: cells without
neighbours, rows and columns one cell wide, holes, every boundary type, lists
that end inside a block; against the oracle (FP64, 1e-10)."""
import numpy as np
import pytest
import torch

from helpers import random_state, rel_err
from hipims_amd.compact_driver import CompactGodunov

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("code", [30, 40, 50, 61, 70, 81, 90])
@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("ny,nx", [(1, 1), (1, 300), (257, 1), (2, 129), (17, 31)])
def test_flux_at_the_ends_of_the_table(oracle_lib, cuda, ny, nx, order, code):
    z, h, qx, qy = random_state(ny, nx, seed=10 * ny + nx, rough=0.1)
    mask = np.ones((ny, nx), dtype=np.int64)
    mask[0, :] = mask[-1, :] = mask[:, 0] = mask[:, -1] = code
    if ny > 2:
        mask[ny // 2, nx // 2] = -9999
        mask[ny // 2, : nx // 2] = code
    pad = lambda a, v: np.pad(a, 1, constant_values=v)  # noqa: E731
    m = pad(mask, -9999)
    f = [pad(a, 0.0) for a in (h, qx, qy, z)]
    series = dict(gd=np.array([[0.0, 0.4, 0.6], [0.5, 0.5, 0.7], [9.0, 0.6, 0.8]]),
                  wl=np.array([[0.0, 0.9, 1.1], [0.5, 1.0, 1.2], [9.0, 1.1, 1.3]]),
                  q=np.array([[0.0, 0.1, 0.2, 0.3, 0.1], [0.5, 0.2, 0.1, 0.1, 0.2], [9.0, 0.1, 0.1, 0.2, 0.2]]))
    man = np.array([0.03])
    num = CompactGodunov(cuda, 1.0, 0.5, 1.0e9, t=1.0, firstTimeStep=0.01, secondOrder=order == 2)
    num.init__fluidField_tensor(m, f[0], f[1], f[2], f[0] + f[3], f[3], cuda)
    num.set__frictionField_tensor(man, cuda)
    num.set_boundary_tensor({"H_GIVEN": series["gd"], "WL_GIVEN": series["wl"], "Q_GIVEN": series["q"]}, cuda)
    o = oracle_lib.OracleSim(m, *f, 1.0, cfl=0.5, order=order, first_dt=0.01, t=1.0, manning=man,
                             given_depth=series["gd"], given_wl=series["wl"], given_q=series["q"])
    for _ in range(2):
        num.addFlux()
        num.time_friction_euler_update_cuda(cuda)
    o.run(2)
    for got, ref in ((num._h_internal, o.h_c), (num._qx_internal, o.qx_c), (num._qy_internal, o.qy_c)):
        assert torch.isfinite(got).all()
        assert rel_err(got.cpu().numpy(), ref) <= 1e-10
