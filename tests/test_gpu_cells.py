"""The form of the cells phase without tiles (k_order, k_gather_all,
k_cell_sums): the tuner runs it on a world's fourth step, so the state after
five steps has been through it and through every tile configuration.
"""
import numpy as np
import pytest

from oracle.orc import OracleCase
from unigasfoam_amd import workloads
from unigasfoam_amd.core import Case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_cells, per_cell, dt", [
    (5, 1, 2.0e-6),        # cells of no, one and two simulators
    (1, 300, 2.0e-6),      # one cell, nothing to merge
    (3, 64, 1.0e-5),       # merges of up to the eight lanes' size
    (3, 128, 1.0e-5),      # about that size: both forms
    (4, 500, 1.0e-5),      # merges by the wave, most of the simulators
    (4, 500, 2.0e-7),      # and with few simulators to merge
])
def test_merges_match_oracle(require_gpu, n_cells, per_cell, dt):
    spec, fill = workloads.heat_bath(n_cells=n_cells, per_cell=per_cell, side=1.0e-3 * n_cells, dt=dt)
    g = Case(spec, precision="fp64", capacity=1 << 16)
    o = OracleCase(spec, capacity=1 << 16)
    for c in (g, o):
        c.fill(**fill)
        c.step(5)
    pg, po = g.particles(), o.particles()
    for k in ("local", "velocity", "erot", "cell", "species"):
        assert np.array_equal(pg[k], po[k]), k
    assert np.array_equal(g.samples(), o.samples())
    g.close()
    o.close()


def test_inflow_merges_match_oracle(require_gpu):
    """Two species, a row of cells with inflow and simulators that cross corners."""
    spec, fill = workloads.cylinder(n_theta=24, n_r=10, target=24 * 10 * 200.0, dt=2.0e-6)
    g = Case(spec, precision="fp64", capacity=1 << 18)
    o = OracleCase(spec, capacity=1 << 18)
    for c in (g, o):
        c.fill(**fill)
        c.step(6)
    pg, po = g.particles(), o.particles()
    for k in ("local", "velocity", "erot", "cell", "species"):
        assert np.array_equal(pg[k], po[k]), k
    assert np.array_equal(g.samples(), o.samples())
    g.close()
    o.close()
