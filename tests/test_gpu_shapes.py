"""The step's kernels at the sizes where their work division changes: GPU
(FP64) against the CPU oracle, bit for bit (assert_identical of
test_gpu_parity: particles in slot order, counters, sampler and wall sums)."""
import pytest

from test_gpu_parity import assert_identical, pair
from unigasfoam_amd import workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,per_cell,stretch", [(1, 3, 4.0), (3, 61, 6.0), (5, 17, 3.0), (9, 8, 2.0)])
def test_many_cells_crossed_per_step_identical(require_gpu, n, per_cell, stretch):
    """Simulators that end beyond their cell's neighbours are counted by
    atomics per run of equal cells in a wave: single cells (one run of every
    length), and boxes where most of them are in runs of one."""
    spec, fill = workloads.heat_bath(n_cells=n, per_cell=per_cell, side=1.0e-3 * n, dt=stretch * 2.0e-6)
    g, o = pair(spec, fill)
    g.step(6)
    o.step(6)
    assert_identical(g, o, f"{n}^3 cells, {per_cell} each")
