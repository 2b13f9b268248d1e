"""The update pass takes one to eight elements per thread by the size of the
domain: at each of these sizes the two-pass step must leave the bits of the
single-pass one, whose update runs inside the stencil."""
import numpy as np
import pytest
import torch

from helpers import random_state
from hipims_amd.grid import GridSolver

pytestmark = pytest.mark.gpu


def solver(ny, nx, dtype, rain):
    z, h, qx, qy = random_state(ny, nx, seed=ny, rough=0.1)
    h[ny // 3: 2 * ny // 3, nx // 4: 3 * nx // 4] = 0.0
    qx[h == 0], qy[h == 0] = 0.0, 0.0
    mask = np.full((ny, nx), 40)
    mask[ny // 2, nx // 2] = -9999
    pad = lambda a, v: np.pad(a, 1, constant_values=v)  # noqa: E731
    s = GridSolver(pad(mask, -9999), pad(h, 0.0), pad(qx, 0.0), pad(qy, 0.0), pad(z, 0.0), 1.0, order=2, dtype=dtype,
                   first_dt=0.02, t=1.0, manning=[0.03])
    shape = (ny + 2, nx + 2)
    if rain == "stations":
        s.set_station_rain(np.array([[0.0, 1e-5, 2e-5], [1e6, 1e-5, 2e-5]]), np.arange(shape[0] * shape[1]).reshape(shape) % 2)
    elif rain == "field":
        s.set_rain_field(np.linspace(0.0, 1e-5, shape[0] * shape[1]).reshape(shape))
    return s


# loops of 1, 1 (to the last element of 1024 blocks), 2, 4, 8 elements a thread
SIZES = [(1, 1), (9, 254), (510, 510), (511, 510), (730, 727), (1450, 1500)]


@pytest.mark.parametrize("rain", ["none", "stations", "field"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("ny,nx", SIZES)
def test_two_pass_matches_single_pass(cuda, ny, nx, dtype, rain):
    a, b = solver(ny, nx, dtype, rain), solver(ny, nx, dtype, rain)
    a.step(3)
    b.step_fused(3)
    for k in ("h", "qx", "qy", "h_max"):
        assert torch.equal(getattr(a, k), getattr(b, k)), k
    assert torch.equal(a.ctrl[:2], b.ctrl[:2])
    # FP64 sums of up to 2.2e6 terms in another order: n eps/2 of the sum of magnitudes at most
    assert torch.allclose(a.ctrl[5:8], b.ctrl[5:8], rtol=1e-9, atol=1e-12)
