"""Where no unit height is asked for, a domain takes one height alone and
another in an ensemble, whose units share a launch.  State, h_max and time
control do not depend on it and keep their bits; the FP64 mass sums add the
same terms in another order, and keep theirs where one height is asked for."""
import pytest
import torch

from hipims_amd import _lib
from hipims_amd.ensemble import Ensemble
from test_gpu_fold import solver, state

pytestmark = pytest.mark.gpu

SIZES = [(700, 640), (512, 512), (900, 333), (640, 700)]  # alone 3 or 4 rows a unit, together 7 or 9


def pair(dtype, rows, single_pass, steps):
    a, b = ([solver(ny, nx, dtype, True, t=1.0, tile_rows=rows) for ny, nx in SIZES] for _ in range(2))
    e = Ensemble(a, single_pass=single_pass)
    e.step(steps)
    alone = Ensemble(b[:1], single_pass=single_pass).handle.tile_rows
    for s in b:
        s.step_fused(steps) if single_pass else s.step(steps)
    return a, b, e.handle.tile_rows, alone


@pytest.mark.parametrize("single_pass", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_state_and_clock_keep_their_bits(cuda, dtype, single_pass):
    a, b, together, alone = pair(dtype, 0, single_pass, 6)
    assert together > alone
    for s, t in zip(a, b):
        (*x, c), (*y, d) = state(s), state(t)
        for u, v in zip(x, y):
            assert torch.equal(u, v)
        sums = slice(_lib.CTRL_FIELDS.index("volume"), _lib.CTRL_FIELDS.index("volume") + 3)
        # up to 4.5e5 terms of one sign (or a flux sum near zero beside them) in another order: n eps/2 of the sum
        # of magnitudes at most, which the volume is for all three
        assert (c[sums] - d[sums]).abs().max() <= 4.5e5 * 1.2e-16 * 6 * d[sums][0].abs()
        c[sums] = d[sums] = 0.0
        assert torch.equal(c, d)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_an_asked_height_keeps_the_sums(cuda, dtype):
    a, b, together, alone = pair(dtype, 8, True, 6)
    assert together == alone == 8
    for s, t in zip(a, b):
        for u, v in zip(state(s), state(t)):
            assert torch.equal(u, v)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_two_pass_sums_keep_their_bits(cuda, dtype):
    """The two-pass step's sums come from its update pass, whose blocks are a
    domain's own: one to eight elements a thread."""
    sizes = [(70, 61), (601, 433), (900, 700), (1101, 1000)]
    a, b = ([solver(ny, nx, dtype, True, t=1.0) for ny, nx in sizes] for _ in range(2))
    Ensemble(a, single_pass=False).step(3)
    for s in b:
        s.step(3)
    for s, t in zip(a, b):
        for u, v in zip(state(s), state(t)):
            assert torch.equal(u, v)
