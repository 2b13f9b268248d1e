"""The class columns of the gradient rows: written in every row, whatever the
rows held, and summing to the per-cell values of each class."""
import ctypes

import pytest
import torch

from hipims_amd import _lib
from hipims_amd.adjoint import Calibration
from test_gpu_fold import solver

pytestmark = pytest.mark.gpu


# planes of fewer elements than a block folds, of no multiple of it, of many
@pytest.mark.parametrize("ny,nx", [(1, 1), (9, 60), (37, 100), (300, 257)])
def test_every_row_is_written(cuda, ny, nx):
    s = solver(ny, nx, torch.float64, False)
    cal = Calibration(s, [[1, 1]], 2, 1)
    gen = torch.Generator(cuda).manual_seed(ny)
    cal.gn.copy_(torch.rand(cal.gn.shape, dtype=torch.float64, device=cuda, generator=gen))
    cal.grads.fill_(float("nan"))
    _lib.check(_lib.lib().hp_adjoint_finish(ctypes.byref(s.desc), ctypes.byref(cal.adesc), _lib.stream_ptr(cuda)),
               "hp_adjoint_finish")
    torch.cuda.synchronize()
    want = cal.gn[s.landuse == 0].sum()
    got = cal.grads[:, :15].sum(dim=0)
    # at most 8e4 positive terms in another order: n eps/2 of their sum
    assert abs(got[0] - want) <= 8e4 * 1.2e-16 * want and (got[1:] == 0).all()
    assert cal.grads[:, 15].isnan().all()
