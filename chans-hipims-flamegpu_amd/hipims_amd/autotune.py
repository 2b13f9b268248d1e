"""Flux unit-height autotuner.

The flux pass and the single-pass step run as column walks: one wave per unit
of 60 columns x R rows.  A taller unit re-loads fewer halo rows and solves
fewer duplicate y-edges (four prologue rows and one edge per unit), a shorter
one gives more waves.  Height 0 leaves the choice to the library, which takes
any height up to 32 by the domain's size so that the units fill whole rounds
of the GPU's wave slots (2048^2 in float: 59 us a step, against 62 at the best
fixed height); the other choices are fixed heights, R in {2, 4, 6, 8, 10, 12,
16} in float and {4, 8} in double.  Which wins depends on dtype, order, domain
and on the step path.  tune() times each on the caller's own domain with HIP
events - the flux pass alone, or single-pass steps - restores the
domain's state afterwards and keeps the fastest; results are memoised per
(dtype, order, size class, path) for the process.
"""
from __future__ import annotations

import torch

from .grid import GridSolver

CHOICES = {torch.float32: (2, 4, 6, 8, 10, 12, 16, 0), torch.float64: (4, 8, 0)}
_cache: dict = {}


def _key(s: GridSolver, path: str):
    cells = s.layout.ny * s.layout.pitch
    return (s.dtype, s.order, max(0, cells.bit_length() - 18), path)


# The clocks rise over the first tens of milliseconds of work, by more than the
# heights differ: so long the tuner warms up, or for as many calls as it times.
WARM_MS = 30.0


def _time(s: GridSolver, path: str, reps: int) -> float:
    """ms per flux pass, or per call of four single-pass steps (as in a run,
    such a call folds the time control in)."""
    run = (lambda: s.step_fused(4)) if path == "fused" else s.flux
    run()  # untimed: the fused path's second buffers
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    a.record()
    for _ in range(reps):
        run()
    b.record()
    torch.cuda.synchronize(s.device)
    return a.elapsed_time(b) / reps


def tune(s: GridSolver, reps: int = 20, apply: bool = True, path: str = "flux") -> int:
    """Best unit height for `path` ("flux": the two-pass flux pass,
    "fused": the single-pass step) on this domain, 0 for the library's own
    choice: each is timed over `reps` flux passes, or 2 * reps single-pass
    steps in calls of four.  s.tune_timings holds the ms per pass or call."""
    if path not in ("flux", "fused"):
        raise ValueError("path must be 'flux' or 'fused'")
    key = _key(s, path)
    if key in _cache:
        best = _cache[key]
    else:
        saved = [s.U.clone(), s.D.clone(), s.h_max.clone(), s.ctrl.clone(), None if s.F is None else s.F.clone()]
        saved_rows = s.tile_rows
        timings = {}
        calls = max(1, reps // 2) if path == "fused" else reps

        def timed():
            ms = _time(s, path, calls)
            s.U.copy_(saved[0])
            s.D.copy_(saved[1])
            s.h_max.copy_(saved[2])
            s.ctrl.copy_(saved[3])
            if saved[4] is not None:
                s.F.copy_(saved[4])
            return ms

        warm = 0.0
        for _ in CHOICES[s.dtype]:
            warm += timed() * calls
            if warm >= WARM_MS:
                break
        for ty in CHOICES[s.dtype]:
            s.set_tile_rows(ty)
            timings[ty] = timed()
        s.set_tile_rows(saved_rows)
        best = min(timings, key=timings.get)
        _cache[key] = best
        s.tune_timings = timings
    if apply:
        s.set_tile_rows(best)
    return best


def tune_ensemble(solvers: list[GridSolver], single_pass: bool = True, steps: int = 10,
                  max_rows: int | None = None, restore: bool = True) -> int:
    """Best unit height for one ensemble launch over `solvers` (all must share
    dtype and order): each legal height (up to `max_rows` when given) and the
    library's own choice (0, of any height) is timed over `steps` ensemble
    steps (after two untimed ones).  With
    `restore` every domain's state is put back afterwards; without it the
    steps stand as the run's own (the states do not depend on the height),
    so a run that retunes on the way loses no work to it.  Sets the winner
    on every solver and returns it."""
    from .ensemble import Ensemble

    if not solvers:
        raise ValueError("no domains")
    dt = solvers[0].dtype
    steps += steps & 1  # the single-pass ensemble steps in pairs
    saved = [(s.U.clone(), s.h_max.clone(), s.ctrl.clone()) for s in solvers] if restore else []
    timings = {}
    for ty in CHOICES[dt]:
        if max_rows is not None and ty > max_rows:
            continue
        for s in solvers:
            s.set_tile_rows(ty)
        e = Ensemble(solvers, single_pass=single_pass)
        e.step(2)
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        e.step(steps)
        b.record()
        torch.cuda.synchronize(solvers[0].device)
        timings[ty] = a.elapsed_time(b) / steps
        del e
        for s, (u, hm, c) in zip(solvers, saved):
            s.U.copy_(u)
            s.h_max.copy_(hm)
            s.ctrl.copy_(c)
            s.state_written()
    best = min(timings, key=timings.get)
    for s in solvers:
        s.set_tile_rows(best)
    solvers[0].tune_timings = timings
    return best
