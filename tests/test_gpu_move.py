"""The move's staged wall interactions and its case table at their edges.

A wave stages up to 64 wall interactions before it records them, and a block
stages the cases of worlds of 2 to 256 cases; the results may depend on
neither.
"""
import numpy as np
import pytest

from oracle.orc import OracleCase
from unigasfoam_amd import abi, workloads
from unigasfoam_amd.batch import Batch
from unigasfoam_amd.core import Case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_cells, per_cell, dt", [
    (1, 1, 2.0e-6),       # one simulator
    (2, 9, 2.0e-5),       # 72 simulators: a full chunk and a remainder, several hits each
    (3, 150, 2.0e-5),     # about 5 hits per simulator and step (sum of sigma sqrt(2 / pi) dt / L
                          # over the axes is 4.8): the stage fills many times
    (6, 40, 2.0e-6),      # most simulators meet no wall
])
@pytest.mark.parametrize("diffuse", [False, True])
def test_wall_interactions_match_oracle(require_gpu, n_cells, per_cell, dt, diffuse):
    """Particles, counters and wall sums equal the oracle's, bit for bit: all
    walls specular, and two of them diffuse (stopped tracks and hits mixed in
    one stage)."""
    spec, fill = workloads.heat_bath(n_cells=n_cells, per_cell=per_cell, side=1.0e-3 * n_cells, dt=dt)
    if diffuse:
        for b in spec.boundaries[:2]:
            b.kind, b.temperature = abi.BND_DIFFUSE, 400.0
    g = Case(spec, precision="fp64", capacity=1 << 14)
    o = OracleCase(spec, capacity=1 << 14)
    for c in (g, o):
        c.fill(**fill)
        c.step(4)
    pg, po = g.particles(), o.particles()
    for k in ("local", "velocity", "cell", "species"):
        assert np.array_equal(pg[k], po[k]), k
    assert np.array_equal(g.wall_samples(), o.wall_samples())
    cg, co = g.counters(), o.counters()
    for k in ("wall_hits", "deleted", "track_errors", "collisions"):
        assert cg[k] == co[k], k
    if n_cells == 3:
        assert cg["wall_hits"] > 4 * 4 * n_cells ** 3 * per_cell
    g.close()
    o.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n_cases", [2, 64, 65, 256, 257])
def test_case_of_a_slot(require_gpu, precision, n_cases):
    """Cases of ragged sizes and different steps in one world move as they do
    alone, below, at and above the staged table's size."""
    def case(i):
        return workloads.couette(n_cells=3 + i % 5, per_cell=1 + (7 * i) % 40, dt=(1 + i % 3) * 5.0e-9, seed=50 + i)
    b = Batch(precision=precision)
    slots = []
    for i in range(n_cases):
        spec, fill = case(i)
        slots.append(b.admit(spec, fill, 256))
    b.step(5)
    b.sync()
    for i in sorted({0, 1, n_cases // 2, n_cases - 2, n_cases - 1}):
        spec, fill = case(i)
        a = Case(spec, precision=precision, capacity=1 << 10)
        a.fill(**fill)
        a.step(5)
        pa, pb = a.particles(), b.case(slots[i]).particles()
        for k in ("local", "velocity", "cell"):
            assert np.array_equal(pa[k], pb[k]), (i, k)
        assert np.array_equal(a.samples(), b.case(slots[i]).samples()), i
        a.close()
    b.close()
