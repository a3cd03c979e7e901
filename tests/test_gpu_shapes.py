"""The step's kernels at the sizes where their work division changes: GPU
(FP64) against the CPU oracle, bit for bit (assert_identical of
test_gpu_parity: particles in slot order, counters, sampler and wall sums)."""
import numpy as np
import pytest

from test_gpu_parity import assert_identical, pair
from unigasfoam_amd import abi, workloads
from unigasfoam_amd.core import Case
from unigasfoam_amd.mesh import box_mesh
from unigasfoam_amd.spec import Boundary, CaseSpec

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


@pytest.mark.parametrize("cells,per_cell", [((1, 1, 1), 7), ((1, 1, 1), 700), ((5, 3, 2), 150), ((65, 64, 1), 3),
                                            ((65, 64, 1), 90)])
@pytest.mark.parametrize("kind", [abi.BND_SPECULAR, abi.BND_DIFFUSE])
def test_wall_sums_of_few_and_many_hits_identical(require_gpu, cells, per_cell, kind):
    """Two species between measured walls in a flat box: faces with no hit, a
    few, and more than the sort stages at a time, with a wave per face (up to
    8192 faces) and with sixteen lanes (65 x 64 x 1 has 8578)."""
    pt = {k: abi.WALL for k in ("xmin", "xmax", "ymin", "ymax", "zmin", "zmax")}
    size = (1.0e-3 * cells[0], 1.0e-3 * cells[1], 2.0e-4 * cells[2])
    mesh = box_mesh((0.0, 0.0, 0.0), size, cells, pt)
    n = 1.0e20
    spec = CaseSpec(mesh=mesh, species=[workloads.N2, workloads.ARGON], delta_t=4.0e-7,
                    n_equivalent_particles=n * size[0] * size[1] * size[2] / (per_cell * mesh.n_cells),
                    collision_model="dsmc", dsmc_model="LarsenBorgnakkeVariableHardSphere", Tref=273.0, seed=9,
                    boundaries=[Boundary(p, kind, 400.0, (30.0, 0.0, 0.0)) for p in sorted(pt)])
    g, o = pair(spec, dict(number_density={"N2": 0.6 * n, "Ar": 0.4 * n}, T=300.0),
                capacity=1 << 22)   # the event buffers hold an eighth of it
    g.step(2)
    o.step(2)
    assert g.counters()["wall_hits"] > 0
    assert_identical(g, o, f"{cells} cells, {per_cell} each")


@pytest.mark.parametrize("n", [1, 255, 256, 1023, 1024, 1025, 2048])
def test_offsets_at_block_edges_identical(require_gpu, n):
    """Cell counts around the blocks of the offset scan (1024 cells each)."""
    spec, fill = workloads.couette(n_cells=n, per_cell=5)
    g, o = pair(spec, fill)
    g.step(5)
    o.step(5)
    assert_identical(g, o, f"{n} cells")


def test_offsets_of_more_than_4096_blocks(require_gpu):
    """4.3e6 cells: the scan's block sums are scanned first.  Every simulator
    is where the sampler counted it, in cell order, and none is lost."""
    spec, fill = workloads.heat_bath(n_cells=162, per_cell=1, side=0.162)
    g = Case(spec, precision="fp32")
    g.fill(**fill)
    g.step(2)
    cell = g.particles()["cell"]
    assert cell.size == 162 ** 3
    assert np.all(np.diff(cell) >= 0)
    g.reset_samples()
    g.step(1)
    cell = g.particles()["cell"]
    assert np.all(np.diff(cell) >= 0)
    assert np.array_equal(g.samples()[abi.S["N"]] / spec.delta_t, np.bincount(cell, minlength=162 ** 3))
