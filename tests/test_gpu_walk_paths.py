"""The column walk's paths through a row (every lane valid, or the general one;
rows with no wet lane) give the same bits: a domain shifted inside its raster
meets other unit boundaries, and so other paths, cell by cell, but must end
with the same state.  One row of units is checked against the CPU oracle."""
import numpy as np
import pytest
import torch

from helpers import compact, random_state, rel_err
from hipims_amd.grid import GridSolver

pytestmark = pytest.mark.gpu


def domain(ny, nx, left, top, right=1):
    """(ny, nx) valid cells (slip walls, a few nodata holes, a dry block) with
    `left` / `top` nodata columns / rows before them."""
    z, h, qx, qy = random_state(ny, nx, seed=100 * ny + nx, rough=0.1)
    h[ny // 3: 2 * ny // 3, nx // 4: 3 * nx // 4] = 0.0
    qx[h == 0], qy[h == 0] = 0.0, 0.0
    mask = np.full((ny, nx), 40)
    rng = np.random.Generator(np.random.PCG64(nx))
    mask[rng.integers(0, ny, 3), rng.integers(0, nx, 3)] = -9999
    pad = lambda a, v: np.pad(a, ((top, 1), (left, right)), constant_values=v)  # noqa: E731
    return pad(mask, -9999), pad(h, 0.0), pad(qx, 0.0), pad(qy, 0.0), pad(z, 0.0)


def run(ny, nx, left, top, dtype, order, fused, steps=4):
    s = GridSolver(*domain(ny, nx, left, top), 1.0, order=order, dtype=dtype, first_dt=0.02, t=1.0, manning=[0.03])
    s.set_station_rain(np.array([[0.0, 1e-5], [1e6, 1e-5]]))
    s.step_fused(steps) if fused else s.step(steps)
    torch.cuda.synchronize()
    return [getattr(s, k)[top: top + ny, left: left + nx].cpu() for k in ("h", "qx", "qy", "h_max")] + [s.ctrl[:2].cpu()]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("ny,nx", [(1, 1), (3, 58), (9, 59), (8, 60), (17, 61), (16, 121), (33, 190)])
def test_same_bits_wherever_the_units_fall(cuda, ny, nx, order, dtype):
    ref = run(ny, nx, 1, 1, dtype, order, True)
    for left, top in ((2, 1), (30, 3), (59, 8), (62, 5)):
        for fused in (True, False):
            for a, b in zip(ref, run(ny, nx, left, top, dtype, order, fused)):
                assert torch.equal(a, b), f"offset ({left}, {top}), fused {fused}"


@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("ny,nx", [(1, 1), (9, 59), (16, 121)])
def test_double_walk_matches_oracle(oracle_lib, cuda, ny, nx, order):
    m, h, qx, qy, z = domain(ny, nx, 1, 1)
    kw = dict(order=order, first_dt=0.02, t=1.0, manning=np.array([0.03]))
    s = GridSolver(m, h, qx, qy, z, 1.0, dtype=torch.float64, **kw)
    o = oracle_lib.OracleSim(m, h, qx, qy, z, 1.0, **kw)
    s.step_fused(1)
    o.run(1)
    for k, ref in (("h", o.h_c), ("qx", o.qx_c), ("qy", o.qy_c)):
        assert rel_err(compact(m, s.raster(getattr(s, k))), ref) <= 1e-10, k
    assert abs(s.dt - o.dt) <= 1e-12 * o.dt
