"""The allocation-free step on a domain whose records fit it at the asked unit
height counted in 64 columns, but whose 60-column units of that height would
not: it takes another height, and is not refused.  One strip of 64 columns has
two of 60, so a narrow, long domain lies well between the two counts."""
import ctypes

import pytest
import torch

from hipims_amd import _lib
from hipims_amd._lib import HpGridDesc, lib
from test_zz_no_alloc import solver

pytestmark = pytest.mark.gpu

RECORD = 8 + 32  # bytes of a unit's partial record: CFL minimum, FP64 sums


@pytest.mark.parametrize("asked", [8, 4])
def test_asked_height_beyond_the_records_gives_way(cuda, asked):
    small = solver(40, torch.float64, 2)  # its tables serve the long domain
    fit = lib().hp_grid_noalloc_max_bytes() // RECORD
    nx, pitch = 64, 64
    ny = asked * (fit // 2 + 64)  # two 60-column strips of this do not fit, one of 64 does
    d = HpGridDesc.from_buffer_copy(small.desc)
    d.nx, d.ny, d.pitch, d.tile_rows, d.mass_sums = nx, ny, pitch, asked, 0
    d.cell0_x, d.cell0_y, d.rain_mode, d.cfl = 1, 1, _lib.HP_RAIN_NONE, 0.5
    d.work, d.work_bytes = None, 0
    keep = [torch.zeros(ny, pitch, dtype=torch.uint8, device=cuda), torch.full((ny, pitch), 255, dtype=torch.uint8, device=cuda)]
    keep[0][1:-1, 1:-1] = 1
    keep[1][1:-1, 1:-1] = 0
    code = torch.zeros(256, dtype=torch.int32, device=cuda)
    code[1] = 40
    d.type_slot, d.landuse, d.slot_code = keep[0].data_ptr(), keep[1].data_ptr(), code.data_ptr()
    ctrl = torch.zeros(_lib.CTRL_DOUBLES, dtype=torch.float64, device=cuda)
    d.ctrl = ctrl.data_ptr()

    def plane():
        return torch.zeros(ny, pitch, dtype=torch.float64, device=cuda)

    z, unread = plane(), plane()
    d.z, d.dh, d.dqx, d.dqy = z.data_ptr(), unread.data_ptr(), unread.data_ptr(), unread.data_ptr()
    wet = torch.rand(ny, pitch, dtype=torch.float64, device=cuda, generator=torch.Generator(cuda).manual_seed(5))
    wet[:, 0] = wet[:, -1] = 0.0
    wet[0] = wet[-1] = 0.0
    wet[64:-64] = 0.0  # water at both ends
    ends = []
    work = None
    for noalloc in (True, False):
        ctrl.zero_()
        ctrl[0], ctrl[1], ctrl[2] = 1.0, 0.01, 1e9
        p = {k: plane() for k in ("h", "qx", "qy", "h_max", "h_out", "qx_out", "qy_out")}
        p["h"].copy_(wet)
        for k, v in p.items():
            setattr(d, k, v.data_ptr())
        if noalloc:
            _lib.check(lib().hp_grid_step_fused_noalloc(ctypes.byref(d), 4, _lib.stream_ptr(cuda)), "noalloc")
        else:
            d.tile_rows = 0
            work = torch.empty(lib().hp_grid_workspace_bytes(ctypes.byref(d)), dtype=torch.uint8, device=cuda)
            d.work, d.work_bytes = work.data_ptr(), work.numel()
            _lib.check(lib().hp_grid_step_fused(ctypes.byref(d), 4, _lib.stream_ptr(cuda)), "step_fused")
        torch.cuda.synchronize()
        ends.append([p[k][rows].clone() for k in ("h", "qx", "qy", "h_max") for rows in (slice(0, 128), slice(-128, None))]
                    + [ctrl[:6].clone()])
        del p
    for a, b in zip(*ends):
        assert torch.equal(a, b)
    assert not torch.equal(ends[0][0], wet[:128])
