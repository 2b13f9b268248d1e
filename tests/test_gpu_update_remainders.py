"""The update pass with two, four and eight elements per thread, at planes that
are no multiple of a block's elements: the last block's threads past the end,
and within it a last access that is partly there.  The two-pass step must leave
the bits of the single-pass one, whose update runs inside the stencil."""
import pytest
import torch

from test_gpu_update_sizes import solver

pytestmark = pytest.mark.gpu

# (ny, nx): elements per thread, elements of a block, elements left for the last one
SIZES = [(601, 433), (900, 700), (1101, 1000), (1151, 958), (2702, 3100)]


def plane(ny, nx):
    return (ny + 2) * ((nx + 2 + 63) // 64 * 64)


def test_sizes_leave_remainders():
    got = []
    for ny, nx in SIZES:
        n, loops = plane(ny, nx), 1
        while loops < 8 and n > loops * 256 * 1024:
            loops *= 2
        got.append((loops, n % (256 * loops)))
    assert got == [(2, 320), (4, 128), (8, 1024), (8, 960), (8, 1024)]


@pytest.mark.parametrize("rain", ["none", "stations", "field"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("ny,nx", SIZES)
def test_two_pass_matches_single_pass(cuda, ny, nx, dtype, rain):
    a, b = solver(ny, nx, dtype, rain), solver(ny, nx, dtype, rain)
    a.step(2)
    b.step_fused(2)
    for k in ("h", "qx", "qy", "h_max"):
        assert torch.equal(getattr(a, k), getattr(b, k)), k
    assert torch.equal(a.ctrl[:2], b.ctrl[:2])
    # FP64 sums of up to 8.5e6 terms in another order: n eps/2 of the sum of magnitudes at most
    assert torch.allclose(a.ctrl[5:8], b.ctrl[5:8], rtol=1e-9, atol=1e-12)
