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


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("ny,nx", [(6, 400), (520, 530), (1030, 1000)])
def test_chosen_unit_height_changes_no_bits(cuda, ny, nx, dtype):
    """The chosen height against one asked for."""
    res = []
    for rows in (0, 8):
        s = GridSolver(*domain(ny, nx, 1, 1), 1.0, order=2, dtype=dtype, first_dt=0.02, t=1.0, manning=[0.03],
                       tile_rows=rows)
        s.step_fused(3)
        res.append([getattr(s, k).clone() for k in ("h", "qx", "qy", "h_max")] + [s.ctrl[:2].clone()])
    for a, b in zip(*res):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype,ny,nx", [
    (torch.float32, 500, 499), (torch.float32, 766, 760), (torch.float32, 2050, 2039),  # one round of 3, 5, 15 rows
    (torch.float32, 2702, 3100), (torch.float64, 1030, 1024), (torch.float64, 2050, 2039)])  # one and several
def test_rounds_of_units_change_no_bits(cuda, dtype, ny, nx):
    """Heights that fit a launch into whole rounds, the last unit of each strip
    a short one: waves step aside for each other, the state must not notice."""
    res = []
    for rows in (0, 8):
        s = GridSolver(*domain(ny, nx, 1, 1), 1.0, order=2, dtype=dtype, first_dt=0.02, t=1.0, manning=[0.03],
                       tile_rows=rows)
        s.step_fused(4)
        s.step(1)
        res.append([getattr(s, k).clone() for k in ("h", "qx", "qy", "h_max")] + [s.ctrl[:2].clone()])
        del s
    for a, b in zip(*res):
        assert torch.equal(a, b)


@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("rows", [1, 2, 3, 63, 64, 65, 129, 289])
def test_rain_table_rows(cuda, rows, fused):
    """The bracketing rows of a rain table, at, between and beyond them: a dry
    flat box holds rate * dt after one step."""
    rng = np.random.Generator(np.random.PCG64(rows))
    tab = np.column_stack([300.0 * np.arange(rows), rng.uniform(1e-5, 2e-5, (rows, 3))])
    mask = np.full((7, 72), -9999)
    mask[1:-1, 1:-1] = 40
    st = np.arange(mask.size).reshape(mask.shape) % 3
    zero = np.zeros(mask.shape)
    for t in sorted({0.0, 10.0, 300.0 * (rows // 2), 300.0 * (rows // 2) + 77.0, 300.0 * (rows - 2) + 299.0,
                     300.0 * (rows - 1), 300.0 * rows}):
        if t < 0:
            continue
        s = GridSolver(mask, zero, zero, zero, zero, 1.0, order=1, dtype=torch.float64, first_dt=1.0, t=t)
        s.set_station_rain(tab, st)
        s.step_fused(1) if fused else s.step(1)
        want = np.zeros(3)
        if t < tab[-1, 0]:
            want = np.array([np.interp(t, tab[:, 0], tab[:, 1 + k]) for k in range(3)])
        got = s.raster(s.h)[mask > 0]
        assert np.abs(got - want[st[mask > 0]]).max() <= 1e-15, (rows, t)


@pytest.mark.parametrize("rows", [1, 2, 64, 65, 130])
def test_boundary_series_rows(oracle_lib, cuda, rows):
    """The row of a boundary series in force (the first whose time is not
    before t), against the oracle."""
    m, h, qx, qy, z = domain(12, 70, 1, 1)
    m[2:8, 1] = 70
    rng = np.random.Generator(np.random.PCG64(rows))
    q = np.column_stack([100.0 * np.arange(rows), rng.uniform(0.1, 0.5, (rows, 2))])
    for t in (1.0, 100.0 * (rows // 2), 100.0 * (rows // 2) + 1.0, 100.0 * rows + 5.0):
        kw = dict(order=2, first_dt=0.02, t=t, manning=np.array([0.03]), given_q=q)
        s = GridSolver(m, h, qx, qy, z, 1.0, dtype=torch.float64, **kw)
        o = oracle_lib.OracleSim(m, h, qx, qy, z, 1.0, **kw)
        s.step_fused(1)
        o.run(1)
        for k, ref in (("h", o.h_c), ("qx", o.qx_c), ("qy", o.qy_c)):
            assert rel_err(compact(m, s.raster(getattr(s, k))), ref) <= 1e-10, (k, rows, t)
