"""Passes that change form with the size: offsets beside the populations up to
1023 cells, wall offsets inside the bucketing up to 4096 faces, and clone
counts by chunks of 1024 slots; and the occupancy count with one or four tiles
per block, by the length of the tile table.  All equal the oracle, bit for
bit."""
import numpy as np
import pytest

from oracle.orc import OracleCase
from test_gpu_parity import assert_identical
from test_gpu_weighting import graded_box
from unigasfoam_amd import workloads
from unigasfoam_amd.core import Case

pytestmark = pytest.mark.gpu


def compare(spec, fill, steps, capacity):
    g = Case(spec, precision="fp64", capacity=capacity)
    o = OracleCase(spec, capacity=capacity)
    for c in (g, o):
        c.fill(**fill)
        c.step(steps)
    assert_identical(g, o, f"after {steps} steps")
    if g.wall_face_count():
        assert np.array_equal(g.wall_samples(), o.wall_samples())
    g.close()
    o.close()


@pytest.mark.parametrize("n_cells", [1, 2, 1022, 1023, 1024, 1025])
def test_cells_of_one_block(require_gpu, n_cells):
    spec, fill = workloads.couette(n_cells=n_cells, per_cell=7)
    compare(spec, fill, 3, 1 << 14)


@pytest.mark.parametrize("n", [1, 26, 27])   # 6, 4056 and 4374 wall faces
def test_wall_faces_of_one_scan(require_gpu, n):
    spec, fill = workloads.heat_bath(n_cells=n, per_cell=2, side=1.0e-3 * n)
    compare(spec, fill, 3, 1 << 17)


@pytest.mark.parametrize("npps", [3, 32, 33, 1500])   # about 100, 1024 and 48000 slots in 32 cells
def test_clones_by_chunks(require_gpu, npps):
    compare(graded_box(npps=npps), dict(number_density={"Ar": 1.0e20}, T=300.0), 6, 1 << 18)


@pytest.mark.parametrize("capacity", [1 << 14, 1 << 20, 1 << 22])   # tables of about 200, 8300 and 33000 tiles
def test_tiles_of_a_count_block(require_gpu, capacity):
    spec, fill = workloads.heat_bath(n_cells=9, per_cell=12, side=9.0e-3)
    compare(spec, fill, 6, capacity)
