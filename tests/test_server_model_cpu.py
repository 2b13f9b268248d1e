"""A model that replaces the export hook or the clock keeps working in the
server's step: the hook is not asked for a return value, and the lists hold the
model's own clock."""
import torch

from hipims_amd.server import Simulation
from hipims_amd.SWE_CUDA import Godunov


class Model(Godunov):
    """Godunov's step and clock over a control block, without a domain."""

    def __init__(self):
        self._ctrl = torch.zeros(16, dtype=torch.float64)
        self._tensorType, self._device, self.exports = torch.float64, "cpu", 0

    def addFlux(self):
        pass

    def addStation_PrecipitationSource(self, table, device):
        pass

    def _run_update(self, mode):
        self._ctrl[1] = 0.5
        self._ctrl[0] += 0.5
        self._ctrl[4] = 1.0  # an export is due

    def _export(self, tag):
        self.exports += 1

    def get_h(self):
        return torch.arange(4.0)


class OwnExport(Model):
    def _export_if_due(self):
        super()._export_if_due()
        self.exports += 100


class OwnClock(Model):
    @property
    def t(self):
        return 3600.0 + self._ctrl[0:1]


def lists(model):
    sim = Simulation(model, None, torch.arange(2), torch.device("cpu"))
    for _ in range(3):
        sim.simulate_one_time_period()
    return sim.t_list[-3:], sim.dt_list[-3:]


def test_clock_lists_with_the_librarys_export():
    m = Model()
    assert lists(m) == ([0.5, 1.0, 1.5], [0.5, 0.5, 0.5])
    assert m.exports == 3


def test_clock_lists_with_an_own_export_hook():
    m = OwnExport()
    assert lists(m) == ([0.5, 1.0, 1.5], [0.5, 0.5, 0.5])
    assert m.exports == 303


def test_an_instances_own_export_hook():
    m = Model()
    due = []
    m._export_if_due = lambda: due.append(m._ctrl[4].item())
    assert lists(m) == ([0.5, 1.0, 1.5], [0.5, 0.5, 0.5])
    assert due == [1.0, 1.0, 1.0] and m.exports == 0


def test_clock_lists_with_an_own_clock():
    assert lists(OwnClock()) == ([3600.5, 3601.0, 3601.5], [0.5, 0.5, 0.5])
