"""Workloads of the shallow-water step, through the package's public entry points.

Each case is one of five kinds of program:

  step       a simulation loop on ``GridSolver.step_fused`` (several steps per call)
  server     the flood server's step: ``Simulation.simulate_one_time_period`` on
             a ``Godunov`` (flux, station rain, update, host reads of t and dt,
             depths at the agent model's cells); with infiltration, the
             catchment script's call sequence on the same class
  ensemble   uneven scenarios advanced by one replayed graph (``Ensemble``)
  calib      one calibration iteration: forward run and gradient (``Calibration``)
  ops        the reference driver's own op sequence on the compact layout
             (``CompactGodunov`` over ``hipims_amd.ops``)

The states are those of a run under way: a rain film of millimetres with water
in the hollows, momentum near the Manning equilibrium of the surface slope, the
time step of its CFL condition; flood cases are mostly dry with a wet channel.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

_PKG = os.path.join(os.getcwd(), "chans-hipims-flamegpu_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

G, HS = 9.81, 1.0e-6
MANNING = (0.02, 0.03, 0.035, 0.05, 0.06, 0.08)
# Green-Ampt parameters per landuse class (m/s, m, -)
INFIL = ((1.0e-6, 2.0e-6, 5.0e-7, 1.5e-6, 3.0e-6, 8.0e-7), (0.11, 0.09, 0.2, 0.06, 0.16, 0.12),
         (0.3, 0.25, 0.2, 0.32, 0.28, 0.22))
GAUGE_S = 300.0     # interval of rain gauge rows
SERIES_S = 900.0    # interval of boundary series rows
T_NOW = 3.0 * 3600  # a storm three hours in (t = 0 for a dam break)

DEFAULTS = dict(kind="step", ny=256, nx=256, dx=5.0, dtype="float32", order=2, steps=10, state="rain", rain="uniform",
                stations=1, domain="box", infil=False, sums=True, gauges=0, checkpoint=0, scenarios=0)


def _case(name=None, **kw):
    c = dict(DEFAULTS, **kw)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: the server's default scheme on a 75 x 75 block around an agent model's town
        _case("server_75_fp64_o1", kind="server", ny=75, nx=75, dx=10.0, dtype="float64", order=1, rain="gauges",
              steps=1),
        # a catchment script: irregular basin, five rain gauges, infiltration, second order
        _case("catchment_601x433_fp64_o2", kind="server", ny=601, nx=433, dx=10.0, dtype="float64", domain="basin",
              rain="gauges", stations=5, infil=True, steps=1),
        # the small plain run: a closed 256 x 256 dam break in double
        _case("dam_break_256_fp64_o2", ny=256, nx=256, dx=1.0, dtype="float64", state="dam", rain="none", steps=20),
        # the headline run: rainfall-runoff at 2048 x 2048, no accounting
        _case("runoff_2048_fp32_o2", ny=2048, nx=2048, sums=False),
        # the same in double
        _case("runoff_2048_fp64_o2", ny=2048, nx=2048, dtype="float64", sums=False, steps=4),
        # the largest domain: per-cell rain field and FP64 mass accounting
        _case("rainfield_8192_fp32_o2", ny=8192, nx=8192, dx=2.0, rain="field", steps=2),
        # river flood on a mostly dry plain: inflow hydrographs, a given water level, first order, ragged sizes
        _case("flood_1021x1537_fp32_o1", ny=1021, nx=1537, order=1, state="flood", rain="none"),
        # uncertainty study: uneven scenarios, one graph replay of ten steps
        _case("ensemble_8_fp32_o2", kind="ensemble", ny=1024, nx=1024, scenarios=8),
        # long-horizon calibration scheme (first order), one iteration over 40 steps and 32 gauges
        _case("calib_1024_fp32_o1", kind="calib", ny=1024, nx=1024, order=1, steps=40, checkpoint=10, gauges=32),
        # short-horizon second-order calibration in double, every state kept
        _case("calib_193x161_fp64_o2", kind="calib", ny=193, nx=161, dtype="float64", steps=10, checkpoint=1,
              gauges=8),
        # the reference driver on the drop-in ops: its defaults (double, first order) and single precision, second order
        _case("ops_701x503_fp64_o1", kind="ops", ny=701, nx=503, dtype="float64", order=1, domain="basin",
              rain="gauges", stations=3, steps=1),
        _case("ops_1500x1301_fp32_o2", kind="ops", ny=1500, nx=1301, rain="gauges", stations=3, steps=1),
    ]


def draw(rng):
    def size(lo, hi):
        n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        return n | 1 if rng.random() < 0.5 else n

    kind = rng.choice(["step", "step", "step", "server", "server", "ensemble", "calib", "ops"])
    dtype = rng.choice(["float32", "float64"])
    order = rng.choice([1, 2])
    if kind == "step":
        n, m = size(72, 3000), rng.uniform(0.6, 1.6)
        state = rng.choice(["rain", "rain", "flood", "dam"])
        rain = rng.choice(["uniform", "gauges", "field"]) if state == "rain" else "none"
        return _case(ny=n, nx=max(64, int(n * m)), dtype=dtype, order=order, state=state, rain=rain,
                     dx=1.0 if state == "dam" else rng.choice([2.0, 5.0, 10.0]),
                     stations=rng.choice([1, 4, 12]) if rain == "gauges" else 1,
                     domain=rng.choice(["box", "basin"]) if state == "rain" else "box",
                     infil=state == "rain" and rng.random() < 0.25, sums=rng.random() < 0.5,
                     steps=rng.choice([2, 3, 4, 6, 10]))
    if kind == "server":
        n = size(64, 1100)
        return _case(kind=kind, ny=n, nx=max(64, int(n * rng.uniform(0.6, 1.6))), dx=10.0, dtype=dtype, order=order,
                     rain="gauges", stations=rng.choice([1, 3, 8]), domain=rng.choice(["box", "basin"]),
                     infil=rng.random() < 0.3, steps=1)
    if kind == "ensemble":
        n = size(128, 900)
        return _case(kind=kind, ny=n, nx=n, dtype=dtype, order=order, scenarios=rng.randint(2, 8),
                     steps=rng.choice([2, 4, 10]))
    if kind == "calib":
        n = size(96, 900 if order == 1 else 300)
        k = rng.randint(6, 30) if order == 1 else rng.randint(3, 10)
        return _case(kind=kind, ny=n, nx=max(64, int(n * rng.uniform(0.6, 1.6))), dtype=dtype, order=order, steps=k,
                     checkpoint=rng.choice([1, 3, 5, k]), gauges=rng.choice([4, 16, 32]))
    n = size(72, 1800)
    return _case(kind=kind, ny=n, nx=max(64, int(n * rng.uniform(0.6, 1.6))), dtype=dtype, order=order, rain="gauges",
                 stations=rng.choice([1, 3, 8]), domain=rng.choice(["box", "basin"]), steps=1)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _noise(ny, nx, gen, top=4, bottom=2, gain=0.6):
    """Fractal value noise: octaves of bilinearly refined lattices, from a
    quarter of the domain down to `bottom` cells."""
    dev = gen.device
    out = torch.zeros(ny, nx, device=dev)
    cell, amp = max(bottom, 2 ** int(math.ceil(math.log2(max(ny, nx)))) // top), 1.0
    while cell >= bottom:
        ly, lx = ny // cell + 2, nx // cell + 2
        lat = torch.randn(1, 1, ly, lx, generator=gen, device=dev)
        out += amp * F.interpolate(lat, size=(ly * cell, lx * cell), mode="bilinear")[0, 0, :ny, :nx]
        cell, amp = cell // 2, amp * gain
    return out


def _unit(a):
    a = a - a.min()
    return a / a.max()


def _sh(a, k, axis):
    """a at the cell k steps further along `axis` (1: east, 0: south)."""
    return torch.roll(a, -k, axis)


def _pad(a, fill=0):
    return F.pad(a, (1, 1, 1, 1), value=fill)


def _gauge_table(gen, rows, cols, peak_mmh):
    r = torch.rand(rows, cols, generator=gen, device=gen.device, dtype=torch.float64) * peak_mmh / 3.6e6
    t = torch.arange(rows, device=gen.device, dtype=torch.float64) * GAUGE_S
    return torch.cat([t[:, None], r], 1).cpu().numpy()


def _round(a, dtype):
    """A 64-bit array of the values the run itself holds in `dtype`."""
    return a.to(dtype).double() if torch.is_tensor(a) else np.asarray(a).astype(
        np.float32 if dtype == torch.float32 else np.float64).astype(np.float64)


def _inputs(case, seed):
    """Rasters with their ring of nodata, on the device (64-bit values that
    are exact in the run's type), tables as numpy arrays."""
    c, dtype = case, getattr(torch, case["dtype"])
    gen = torch.Generator(device=_device())
    gen.manual_seed(int(seed))
    ny, nx, dx = c["ny"], c["nx"], c["dx"]
    n = max(ny, nx)
    dev = gen.device
    valid = torch.ones(ny, nx, dtype=torch.bool, device=dev)
    t0 = T_NOW
    if c["state"] == "dam":
        t0 = 0.0
        z = torch.zeros(ny, nx, device=dev)
        left = torch.arange(nx, device=dev)[None, :] < nx // 2
        lvl = torch.rand(2, generator=gen, device=dev)
        h = torch.where(left, 1.75 + 0.5 * lvl[0], 0.4 + 0.2 * lvl[1]).expand(ny, nx).clone()
        h += 0.05 * _noise(ny, nx, gen, bottom=8)
        cls = torch.full((ny, nx), 1, device=dev)
    else:
        z = _unit(_noise(ny, nx, gen)) * 50.0 * math.sqrt(n / 2048.0)
        w = max(1, int(round(10.0 / dx)))
        z[ny // 2 - w // 2: ny // 2 - w // 2 + w, :] -= 2.0
        k = 17
        smooth = F.avg_pool2d(z[None, None], k, 1, k // 2, count_include_pad=False)[0, 0]
        hollow = (smooth - z).clamp(min=0.0)
        u = _unit(_noise(ny, nx, gen, bottom=8))
        h = 1.0e-3 * (0.5 + 4.0 * u) + hollow
        if c["state"] == "flood":
            low = z < torch.quantile(z[:: max(1, ny // 256), :: max(1, nx // 256)].flatten(), 0.3)
            h = torch.where(low, h + 0.3, torch.zeros_like(h))
        cls = (_unit(_noise(ny, nx, gen, bottom=16)) * 5.999).long()
    if c["domain"] == "basin":
        yy = torch.linspace(-1, 1, ny, device=dev)[:, None]
        xx = torch.linspace(-1, 1, nx, device=dev)[None, :]
        outline = torch.Generator(device=dev)  # a catchment's outline is its own, whatever the storm
        outline.manual_seed(1000003 * ny + nx)
        valid = (xx ** 2 + yy ** 2 + 0.12 * _noise(ny, nx, outline, bottom=4)) < 0.9
    # surface slope -> Manning momentum below the critical Froude number
    eta = (z + h)[None, None]
    eta = F.pad(eta, (1, 1, 1, 1), mode="replicate")[0, 0]
    sx, sr = (eta[1:-1, 2:] - eta[1:-1, :-2]) / (2 * dx), (eta[2:, 1:-1] - eta[:-2, 1:-1]) / (2 * dx)
    s = torch.sqrt(sx ** 2 + sr ** 2) + 1e-9
    man = torch.tensor(MANNING, device=dev)[cls]
    vel = torch.minimum(h ** (2 / 3) * torch.sqrt(s) / man, 0.5 * torch.sqrt(G * h))
    if c["state"] == "dam":
        vel = torch.zeros_like(vel)
    qx, qy = -h * vel * sx / s, h * vel * sr / s  # y grows towards row 0
    # mask codes: 1 inside, 40 slip wall, 50 open, 30 rigid, 70/71 given discharge, 80 given level
    valid = _pad(valid)
    rim = valid & ~(_sh(valid, 1, 0) & _sh(valid, -1, 0) & _sh(valid, 1, 1) & _sh(valid, -1, 1))
    col = torch.arange(nx + 2, device=dev)[None, :].expand(ny + 2, nx + 2)
    row = torch.arange(ny + 2, device=dev)[:, None].expand(ny + 2, nx + 2)
    mask = torch.where(rim, 30 if c["state"] == "dam" else 40, 1)
    if c["state"] == "flood":
        mask = torch.where(rim & (col == 1) & (row > ny // 4) & (row < ny // 2), 70, mask)
        mask = torch.where(rim & (col == 1) & (row >= ny // 2) & (row < 3 * ny // 4), 71, mask)
        mask = torch.where(rim & (col == nx), 80, mask)
    elif c["state"] == "rain":
        mask = torch.where(rim & (col >= nx - (0 if c["domain"] == "box" else nx // 10)), 50, mask)
    mask = torch.where(valid, mask, -9999).int()
    off = lambda a: torch.where(valid, _pad(a).to(dtype), 0.0).double()  # noqa: E731
    d = dict(valid=valid, mask=mask, z=off(z), h=off(h), qx=off(qx), qy=off(qy), t=t0, dx=dx,
             cls=torch.where(valid, _pad(cls), 0), manning=_round(MANNING, dtype))
    cel = torch.sqrt(G * d["h"]) + torch.maximum(d["qx"].abs(), d["qy"].abs()) / d["h"].clamp(min=1e-5)
    d["dt"] = float(0.5 * dx / float(cel.max()))
    # rain
    d["table"] = d["field"] = d["station"] = None
    if c["rain"] == "uniform":
        r = (30.0 + 40.0 * float(torch.rand(1, generator=gen, device=dev))) / 3.6e6
        d["table"] = np.array([[0.0, r], [1.0e6, r], [1.1e6, 0.0]])
    elif c["rain"] == "gauges":
        d["table"] = _gauge_table(gen, 289, c["stations"], 80.0)
        st = (_unit(_noise(ny, nx, gen, bottom=32)) * (c["stations"] - 1e-3)).long()
        d["station"] = torch.where(valid, _pad(st), 0)
    elif c["rain"] == "field":
        f = (30.0 + 10.0 * _noise(ny, nx, gen, bottom=64)).clamp(min=0.0) / 3.6e6
        d["field"] = torch.where(valid, _pad(f).float(), 0.0).double()
    # boundary series (discharge per unit width into the domain; water level)
    d["wl"], d["q"] = np.array([[0.0, 0.0]]), np.array([[0.0, 0.0, 0.0]])
    if c["state"] == "flood":
        rows = 97
        t = np.arange(rows) * SERIES_S
        amp = torch.rand(rows, 2, generator=gen, device=dev).double().cpu().numpy()
        d["q"] = _round(np.stack([t, 0.5 + 1.5 * amp[:, 0], 0 * t, 0.2 + amp[:, 1], 0 * t], 1), dtype)
        lvl = float(d["z"][valid].quantile(0.1)) if valid.sum() < 1e6 else float(d["z"][::8, ::8][valid[::8, ::8]].quantile(0.1))
        d["wl"] = _round(np.stack([t, lvl + 0.5 * amp[:, 0]], 1), dtype)
    if c["gauges"]:
        g = torch.randperm((ny - 4) * (nx - 4), generator=gen, device=dev)[: c["gauges"]].cpu().numpy()
        d["gauges"] = np.stack([3 + g // (nx - 4), 3 + g % (nx - 4)], 1)
        h0 = d["h"].cpu().numpy()[d["gauges"][:, 0], d["gauges"][:, 1]]
        rnd = torch.rand(c["steps"] + 1, c["gauges"], generator=gen, device=dev).double().cpu().numpy()
        d["obs"] = h0[None, :] * (0.7 + 0.6 * rnd)
        th = torch.rand(len(MANNING) + 1, generator=gen, device=dev).double().cpu().numpy()
        d["theta"] = np.array(MANNING + (1.0,)) * (0.8 + 0.4 * th)
    return d


def _members(case, seed):
    """The scenarios of an ensemble: sizes from half to three halves of the case's."""
    r = np.random.Generator(np.random.PCG64(int(seed)))
    for k in range(case["scenarios"]):
        n = int(round(case["ny"] * (0.5, 0.75, 1.0, 1.5, 1.25)[k % 5]))
        yield dict(case, ny=n, nx=n), int(r.integers(1 << 40))


def _np(t):
    return t.cpu().numpy()


# ---------------------------------------------------------------------------
# what a program holds before the call, and one pass
# ---------------------------------------------------------------------------
def _solver(case, d, dev):
    from hipims_amd.grid import GridSolver

    s = GridSolver(_np(d["mask"]), _np(d["h"]), _np(d["qx"]), _np(d["qy"]), _np(d["z"]), d["dx"], order=case["order"],
                   dtype=getattr(torch, case["dtype"]), device=dev, first_dt=d["dt"], t=d["t"], manning=d["manning"],
                   landuse=_np(d["cls"]), given_wl=d["wl"], given_q=d["q"], mass_sums=case["sums"])
    if d["table"] is not None:
        s.set_station_rain(d["table"], _np(d["station"]) if d["station"] is not None and case["stations"] > 1 else None)
    elif d["field"] is not None:
        s.set_rain_field(_np(d["field"]))
    if case["infil"]:
        s.set_infiltration(*INFIL)
    return s


def prepare(case, seed):
    dev, dtype = torch.device("cuda", 0), getattr(torch, case["dtype"])
    st = {"case": case}
    if case["kind"] == "ensemble":
        from hipims_amd.ensemble import Ensemble

        st["solvers"] = [_solver(c, _inputs(c, s), dev) for c, s in _members(case, seed)]
        st["run"] = Ensemble(st["solvers"])
        st["run"].capture(case["steps"])
        return st
    d = _inputs(case, seed)
    if case["kind"] == "step":
        st["run"] = _solver(case, d, dev)
    elif case["kind"] == "calib":
        from hipims_amd.adjoint import Calibration

        st["run"] = Calibration(_solver(case, d, dev), d["gauges"], case["steps"], checkpoint=case["checkpoint"],
                                obs=d["obs"])
        st["theta"] = torch.from_numpy(d["theta"])
    else:
        from hipims_amd.SWE_CUDA import Godunov
        from hipims_amd.compact_driver import CompactGodunov
        from hipims_amd.server import Simulation

        cls = Godunov if case["kind"] == "server" else CompactGodunov
        g = cls(dev, d["dx"], 0.5, 1.0e9, t=d["t"], secondOrder=case["order"] == 2, firstTimeStep=d["dt"],
                tensorType=dtype)
        m = _np(d["mask"])
        g.set__frictionField_tensor(d["manning"], dev)
        z, h = _np(d["z"]), _np(d["h"])
        g.init__fluidField_tensor(m, h, _np(d["qx"]), _np(d["qy"]), z + h, z, dev)
        g.set_landuse(m, _np(d["cls"]), dev)
        g.set_distributed_rainfall_station_Mask(m, _np(d["station"]), dev)
        if case["infil"]:
            g.set__infiltrationField_tensor(*[np.array(v) for v in INFIL], dev)
        st["run"], st["table"], st["device"] = g, d["table"], dev
        if case["kind"] == "server" and not case["infil"]:
            st["sim"] = Simulation(g, d["table"], _watched(d), dev)
    return st


def _watched(d):
    """Compact ids of the cells the agent model covers: the middle of the domain."""
    v = _np(d["valid"])
    box = np.zeros_like(v)
    box[v.shape[0] // 4: -(v.shape[0] // 4), v.shape[1] // 4: -(v.shape[1] // 4)] = True
    return np.flatnonzero(box[v])


def _fields(s):
    return {"h": s.h, "qx": s.qx, "qy": s.qy, "h_max": s.h_max}


def run(state):
    c, r = state["case"], state["run"]
    if c["kind"] == "step":
        r.step_fused(c["steps"])
        out = _fields(r)
        out["clock"] = r.ctrl[:2].to(r.dtype)
        if c["sums"]:
            out["volume"] = r.ctrl[5:8].to(r.dtype)
        if c["infil"]:
            out["F"] = r.F
        return out
    if c["kind"] == "server":
        if "sim" in state:
            state["sim"].simulate_one_time_period()
            extra = {"depths": state["sim"].results}
        else:
            r.addFlux()
            r.addStation_PrecipitationSource(state["table"], state["device"])
            r.addInfiltrationSource()
            r.time_friction_euler_update_cuda(state["device"])
            extra = {"F": r.solver.F, "depths": r.get_h()}
        return {**_fields(r.solver), **extra, "t": r.t.to(r.solver.dtype), "dt": r.dt.to(r.solver.dtype)}
    if c["kind"] == "ensemble":
        r.replay()
        return {"scenarios": [_fields(s) for s in state["solvers"]], "t": r.times().to(state["solvers"][0].dtype)}
    if c["kind"] == "calib":
        loss = r.run(state["theta"])
        grad = r.gradient()
        return {"loss": loss.to(r.s.dtype), "grad": grad.to(r.s.dtype), "depths": r.hist}
    r.addFlux()
    r.addStation_PrecipitationSource(state["table"], state["device"])
    r.time_friction_euler_update_cuda(state["device"])
    return {"h": r._h_internal, "qx": r._qx_internal, "qy": r._qy_internal, "wl": r._wl_internal, "h_max": r._h_max,
            "t": r.t, "dt": r.dt}


def work(case):
    """Per cell and step: h, qx, qy, z, h_max read once, h, qx, qy, h_max
    written once, plus the class planes and the rain; about 150 (first order
    110) operations per edge, two edges per cell, and 60 for the update.  A
    gradient step costs about two forward ones in operations and reads the
    saved state and flux beside the cotangents."""
    b = 8 if case["dtype"] == "float64" else 4
    rain = {"field": 4, "gauges": 2 if case["stations"] > 1 else 0}.get(case["rain"], 0)
    per_cell = 9 * b + 2 + rain + (2 * b if case["infil"] else 0)
    flops = 2 * (150 if case["order"] == 2 else 110) + 60
    cells = case["ny"] * case["nx"]
    if case["kind"] == "ensemble":
        cells = sum(c["ny"] * c["nx"] for c, _ in _members(case, 0))
    if case["kind"] == "ops":
        per_cell += 20 + 2 * b  # the neighbour table, wl read and written
    if case["kind"] == "calib":
        per_cell, flops = per_cell + 12 * b + 2, 3 * flops
    return {"bytes": float(cells * case["steps"] * per_cell), "flops": float(cells * case["steps"] * flops)}


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _minmod(a, b):
    return torch.where(a * b <= 0, torch.zeros_like(a), torch.where(a.abs() < b.abs(), a, b))


def _safe_sqrt(x):
    return torch.where(x > 0, torch.sqrt(torch.where(x > 0, x, torch.ones_like(x))), torch.zeros_like(x))


def _hllc(order, L, R, etaC, etaR):
    """Fluxes between the faces L and R = (h, qn, qt, z) after the hydrostatic
    reconstruction, and the reconstructed (h, z) of both sides."""
    (hL, nL, tL, zL), (hR, nR, tR, zR) = L, R
    zero, one = torch.zeros_like(hL), torch.ones_like(hL)
    vel = lambda q, h: torch.where(h < HS, zero, q / torch.where(h < HS, one, h))  # noqa: E731
    uL, vL, uR, vR = vel(nL, hL), vel(tL, hL), vel(nR, hR), vel(tR, hR)
    lo, hi = torch.minimum(etaC, etaR), torch.maximum(etaC, etaR)
    wL = torch.maximum(torch.minimum(hL + zL, hi), lo)
    wR = torch.maximum(torch.minimum(hR + zR, hi), lo)
    if order == 1:
        m, avg = (wL + wR) / 2, (etaC - etaR) * (wL - wR) < 0
        wL, wR = torch.where(avg, m, wL), torch.where(avg, m, wR)
    else:
        w, left = torch.maximum(wL, wR), etaC > etaR
        wL, wR = torch.where(left, w, wL), torch.where(left, wR, w)
    zb = torch.maximum(wL - hL, wR - hR)
    hL, hR = (wL - zb).clamp(min=0), (wR - zb).clamp(min=0)
    zL, zR = wL - hL, wR - hR
    qL, qR, pL, pR = uL * hL, uR * hR, vL * hL, vR * hR
    aL, aR = _safe_sqrt(G * hL), _safe_sqrt(G * hR)
    a_s, u_s = ((aL + aR) / 2 + (uL - uR) / 4).abs(), (uL + uR) / 2 + aL - aR
    sL = torch.where(hL <= HS, uR - 2 * aR, torch.minimum(uL - aL, u_s - a_s))
    sR = torch.where(hR <= HS, uL + 2 * aL, torch.maximum(uR + aR, u_s + a_s))
    den = hR * (uR - sR) - hL * (uL - sL)
    sM = (sL * hR * (uR - sR) - sR * hL * (uL - sL)) / den
    fL, fR = uL * qL + 0.5 * G * hL * hL, uR * qR + 0.5 * G * hR * hR
    span = sR - sL
    rS = 1 / torch.where(span == 0, one, span)
    fh = (sR * qL - sL * qR + sL * sR * (hR - hL)) * rS
    fn = (sR * fL - sL * fR + sL * sR * (qR - qL)) * rS
    star_l = (sL < 0) & (sM >= 0)
    ft = fh * torch.where(star_l, vL, vR)
    left, star = sL >= 0, star_l | ((sM < 0) & (sR >= 0))
    dry = (hL < HS) & (hR < HS)
    pick = lambda l, s, r: torch.where(dry, zero, torch.where(left, l, torch.where(star, s, r)))  # noqa: E731
    return pick(qL, fh, qR), pick(fL, fn, fR), pick(uL * pL, ft, uR * pR), (hL, zL), (hR, zR)


def _series(tab, t):
    r = 0
    while r < len(tab) - 1 and t > tab[r, 0]:
        r += 1
    return tab[r]


def _flux(order, d, h, qx, qy, t, dt):
    """Flux increments (dh, dqx, dqy) of the listed cells, and the list."""
    V, z, dx = d["valid"], d["z"], d["dx"]
    k = dt / dx
    acc = [torch.zeros_like(h), torch.zeros_like(h), torch.zeros_like(h)]
    for axis in (1, 0):  # edges to the east, edges to the south
        n_, t_ = (qx, qy) if axis == 1 else (-qy, qx)
        vB, vl, vr = _sh(V, 1, axis), _sh(V, -1, axis), _sh(V, 2, axis)
        A, Bc = (h, n_, t_, z), tuple(_sh(a, 1, axis) for a in (h, n_, t_, z))
        both = V & vB & ~((A[0] < HS) & (Bc[0] < HS))
        lo = tuple(torch.where(vl, _sh(a, -1, axis), a) for a in A)
        up = tuple(torch.where(vr, _sh(a, 2, axis), b) for a, b in zip(A, Bc))
        half = lambda i: (0.5 * _minmod(A[i] - lo[i], Bc[i] - A[i]), 0.5 * _minmod(Bc[i] - up[i], A[i] - Bc[i]))  # noqa: E731,B023
        sz = half(3)
        if order == 1:
            L = (A[0], A[1], A[2], torch.where(Bc[0] > HS, z + sz[0], z))
            R = (Bc[0], Bc[1], Bc[2], torch.where(A[0] > HS, Bc[3] + sz[1], Bc[3]))
        else:
            s = [half(i) for i in range(3)]
            dryA, dryB, zero = A[0] < HS, Bc[0] < HS, torch.zeros_like(h)
            L = (A[0] + s[0][0], torch.where(dryA, zero, A[1] + s[1][0]), torch.where(dryA, zero, A[2] + s[2][0]),
                 z + sz[0])
            R = (Bc[0] + s[0][1], torch.where(dryB, zero, Bc[1] + s[1][1]),
                 torch.where(dryB, zero, Bc[2] + s[2][1]), Bc[3] + sz[1])
        fh, fn, ft, rL, rR = _hllc(order, L, R, A[0] + z, Bc[0] + Bc[3])
        bA = 0.5 * G * (rL[0] + A[0]) * (rL[1] - z)
        bB = 0.5 * G * (rR[0] + Bc[0]) * (rR[1] - Bc[3])
        zero = torch.zeros_like(h)
        fh, fn, ft, bA, bB = (torch.where(both, v, zero) * k for v in (fh, fn, ft, bA, bB))
        nA = 1.0 if axis == 1 else -1.0
        gx, gy = (fn, ft) if axis == 1 else (ft, -fn)
        own, far = [-fh, -gx, -gy], [fh, gx, gy]
        i = 1 if axis == 1 else 2
        own[i] = own[i] - bA * nA
        far[i] = far[i] + bB * nA
        acc = [a + o + _sh(f, -1, axis) for a, o, f in zip(acc, own, far)]
    # boundary edges, from the valid side with its outward normal
    wl, q = _series(d["wl"], t), _series(d["q"], t)
    for dr, (axis, step) in enumerate(((1, 1), (0, -1), (1, -1), (0, 1))):  # E, N, W, S
        at = (V & ~_sh(V, step, axis)).nonzero(as_tuple=True)
        if at[0].numel() == 0:
            continue
        hc, x, y, zc, code = h[at], qx[at], qy[at], z[at], d["mask"][at].long()
        ty, ids = torch.where(code >= 10, code // 10, code), torch.where(code >= 10, code % 10, 0)
        cn, ct = ((x, y), (y, -x), (-x, -y), (-y, x))[dr]
        gh, gn, gt = hc.clone(), cn.clone(), ct.clone()
        if dr in (0, 2):
            gn, gt = torch.where(ty == 3, -gn, gn), torch.where(ty == 3, -gt, gt)
        gn = torch.where(ty == 4, -gn, gn)
        val = lambda row, j: torch.as_tensor(row, device=h.device)[j.clamp(max=len(row) - 1)]  # noqa: E731
        bx, by = val(q, 1 + 2 * ids), val(q, 2 + 2 * ids)
        bn, bt = ((bx, by), (by, -bx), (-bx, -by), (-by, bx))[dr]
        gn, gt = torch.where(ty == 7, bn, gn), torch.where(ty == 7, bt, gt)
        gh = torch.where(ty == 8, (val(wl, 1 + ids) - zc).clamp(min=0), gh)
        etaG = zc + gh if order == 1 else torch.where((ty == 7) | (ty == 8), zc + gh, zc + hc)
        fh, fn, ft, rL, _ = _hllc(order, (hc, cn, ct, zc), (gh, gn, gt, zc), hc + zc, etaG)
        live = ~((hc < HS) & (gh < HS))
        bed = 0.5 * G * (rL[0] + hc) * (rL[1] - zc)
        fh, fn, ft, bed = (torch.where(live, v, torch.zeros_like(v)) * k for v in (fh, fn, ft, bed))
        gx, gy = ((fn, ft), (-ft, fn), (-fn, -ft), (ft, -fn))[dr]
        if axis == 1:
            gx = gx + bed * (1.0 if dr == 0 else -1.0)
        else:
            gy = gy + bed * (1.0 if dr == 1 else -1.0)
        acc = [a.index_put(at, -v, accumulate=True) for a, v in zip(acc, (fh, gx, gy))]
    wet = V & (h > HS)
    first = int(V.flatten().int().argmax())  # the first cell never counts as a wet neighbour
    seen = wet.clone()
    seen.view(-1)[first] = False
    on = V if t == 0.0 else V & (wet | _sh(seen, 1, 1) | _sh(seen, -1, 1) | _sh(seen, 1, 0) | _sh(seen, -1, 0))
    return [torch.where(on, a, torch.zeros_like(a)) for a in acc], on


def _rain(d, t, h):
    if d["field"] is not None:
        return d["field"]
    tab = d["table"]
    if tab is None or t >= tab[-1, 0]:
        return torch.zeros_like(h)
    i = 0
    while i + 1 < len(tab) - 1 and t >= tab[i + 1, 0]:
        i += 1
    w = (t - tab[i, 0]) / (tab[i + 1, 0] - tab[i, 0])
    r = torch.as_tensor(tab[i, 1:] + w * (tab[i + 1, 1:] - tab[i, 1:]), device=h.device)
    return torch.where(d["valid"], r[d["station"]] if d["station"] is not None else r[0], torch.zeros_like(h))


def _friction(h, n, dt, qx, qy):
    cf = G * n * n * h ** (-1 / 3)
    qn = _safe_sqrt(qx * qx + qy * qy)
    k = 2 / (1 + torch.sqrt(1 + 4 * dt * cf / (h * h) * qn))
    lim = 5 * h * torch.sqrt(G * h)
    out = []
    for q in (qx, qy):
        tq = k * q
        refl = 2 * tq - q
        o = torch.where(tq.abs() > lim, torch.where(refl * tq <= 0, torch.zeros_like(q), refl), tq)
        out.append(torch.where(q.abs() > 1e-10, o, q))
    return out


def _steps(case, d, steps, manning=None, rain_scale=1.0, watch=None):
    """`steps` steps in 64 bits; the state, clock, sums and watched depths."""
    V, dx = d["valid"], d["dx"]
    h, qx, qy = d["h"], d["qx"], d["qy"]
    hm = h
    man = torch.as_tensor(d["manning"], device=h.device) if manning is None else manning
    n = man[d["cls"]]
    t, dt = d["t"], d["dt"]
    if case["dtype"] == "float32":
        dt = float(np.float32(dt)) if case["kind"] == "ops" else dt
    infil = [torch.as_tensor(_round(v, getattr(torch, case["dtype"])), device=h.device)[d["cls"]] for v in INFIL] \
        if case["infil"] else None
    Fc = torch.zeros_like(h)
    vol = rain_v = flux_v = 0.0
    seen = [h[watch]] if watch is not None else []
    zero, one = torch.zeros_like(h), torch.ones_like(h)
    for _ in range(steps):
        (dh, dqx, dqy), on = _flux(case["order"], d, h, qx, qy, t, dt)
        rdt = _rain(d, t, h) * rain_scale * dt
        dF = zero
        if infil:
            ks, phi, dth = infil
            a = Fc + dt * ks
            dF = torch.where(on, torch.minimum(h, 0.5 * (a + torch.sqrt(a * a + 4 * dt * ks * (phi + h) * dth)) - Fc), zero)
            Fc = Fc + dF
        dht = dh + rdt - dF
        upd = V & ((dht.abs() > 0) | (h >= 0))
        h1 = torch.where(upd, h + dht, h)
        wet = upd & (h1 >= HS)
        hw = torch.where(wet, h1, one)
        fx, fy = _friction(hw, n, dt, torch.where(wet, qx + dqx, one), torch.where(wet, qy + dqy, one))
        qx = torch.where(wet, fx, torch.where(upd, zero, qx))
        qy = torch.where(wet, fy, torch.where(upd, zero, qy))
        h = h1
        with torch.no_grad():
            hm = torch.where(upd, torch.maximum(hm, h), hm)
            live = upd & (h > HS)
            hd = torch.where(live, h, one)
            c = torch.sqrt((G * hd).float()).double()  # the celerity is single precision in every build
            cand = torch.where(live, 0.5 * dx / (c + torch.maximum(qx.abs(), qy.abs()) / hd), 60.0)
            new = min(float(cand[upd].min()) if bool(upd.any()) else dt, 10 * dt)
            vol = float(torch.where(V, h, zero).sum()) * dx * dx
            flux_v += float(torch.where(upd, dh, zero).sum()) * dx * dx
            rain_v += float(torch.where(upd, rdt, zero).sum()) * dx * dx
        dt, t = new, t + new
        if watch is not None:
            seen.append(h[watch])
    return dict(h=h, qx=qx, qy=qy, h_max=hm, F=Fc, t=t, dt=dt, sums=(vol, rain_v, flux_v), seen=seen)


def _plane(a):
    return F.pad(a, (0, -a.shape[1] % 64))


def _planes(r):
    return {k: _plane(r[k]) for k in ("h", "qx", "qy", "h_max")}


def exact(case, seed):
    one = lambda v: torch.tensor([v], dtype=torch.float64)  # noqa: E731
    if case["kind"] == "ensemble":
        rs = [_steps(c, _inputs(c, s), case["steps"]) for c, s in _members(case, seed)]
        return {"scenarios": [_planes(r) for r in rs], "t": torch.tensor([r["t"] for r in rs], dtype=torch.float64)}
    d = _inputs(case, seed)
    if case["kind"] == "calib":
        dtype = getattr(torch, case["dtype"])
        th = torch.tensor(d["theta"], device=d["h"].device)
        th[:-1] = _round(th[:-1], dtype)
        th.requires_grad_(True)
        at = tuple(torch.as_tensor(v, device=d["h"].device) for v in d["gauges"].T)
        r = _steps(case, d, case["steps"], manning=th[:-1], rain_scale=th[-1], watch=at)
        obs = torch.as_tensor(d["obs"], device=th.device)
        loss = sum(((s - o) ** 2).sum() for s, o in zip(r["seen"][1:], obs[1:]))
        loss.backward()
        return {"loss": loss.detach(), "grad": th.grad, "depths": torch.stack([s.detach() for s in r["seen"]])}
    r = _steps(case, d, case["steps"])
    if case["kind"] == "step":
        out = _planes(r)
        out["clock"] = torch.tensor([r["t"], r["dt"]], dtype=torch.float64)
        if case["sums"]:
            out["volume"] = torch.tensor(r["sums"], dtype=torch.float64)
        if case["infil"]:
            out["F"] = _plane(r["F"])
        return out
    if case["kind"] == "server":
        out = {**_planes(r), "t": one(r["t"]), "dt": one(r["dt"])}
        out["depths"] = r["h"][d["valid"]]
        if case["infil"]:
            out["F"] = _plane(r["F"])
        else:
            out["depths"] = out["depths"][torch.as_tensor(_watched(d), device=r["h"].device)]
        return out
    v = d["valid"]
    return {"h": r["h"][v], "qx": r["qx"][v], "qy": r["qy"][v], "wl": (r["h"] + d["z"])[v], "h_max": r["h_max"][v],
            "t": one(r["t"]), "dt": one(r["dt"])}
