"""Cells of thousands of simulators, most of which leave their cell past its
neighbours in a step: what is done for them must not grow out of proportion.
The bounds are ratios of times of one run, between those measured with and
without the forms that keep to them."""
import pytest

from unigasfoam_amd import workloads
from unigasfoam_amd.core import Case

pytestmark = pytest.mark.gpu


def phase_us(per_cell, crossings, phase, steps=3, n_cells=1000):
    """Shortest time of a phase over `steps` steps of a channel whose simulators
    cross about `crossings` cells per step."""
    spec, fill = workloads.couette(n_cells=n_cells, per_cell=per_cell, dt=5.0e-9 * crossings, collision_model="none")
    g = Case(spec, precision="fp32", capacity=int(1.3 * n_cells * per_cell) + 70000)
    g.fill(**fill)
    g.step(10)   # past the tuner's steps
    best = float("inf")
    for _ in range(steps):
        g.timing(True)
        g.step(1)
        g.sync()
        best = min(best, 1000.0 * g.phase_times()[0][phase])
    g.close()
    return best


def test_count_of_cells_crossed(require_gpu):
    """Simulators that crossed one cell are counted in LDS, those that crossed
    more by atomics on 1000 counters (1.5 times as long, 2.0 with an atomic per
    simulator)."""
    assert phase_us(10000, 5, "scan") < 1.75 * phase_us(10000, 1, "scan")
