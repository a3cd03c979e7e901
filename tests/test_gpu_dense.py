"""Cells of thousands of simulators, most of which leave their cell past its
neighbours in a step: what is done for them must not grow out of proportion.
The bounds are ratios of times of one run, between those measured with and
without the forms that keep to them."""
import numpy as np
import pytest

from oracle.orc import OracleCase
from unigasfoam_amd import abi, workloads
from unigasfoam_amd.core import Case
from unigasfoam_amd.mesh import box_mesh
from unigasfoam_amd.spec import Boundary, CaseSpec

pytestmark = pytest.mark.gpu


def phase_us(per_cell, crossings, phase, steps=3, n_cells=1000, variant=-1):
    """Shortest time of a phase over `steps` steps of a channel whose simulators
    cross about `crossings` cells per step."""
    spec, fill = workloads.couette(n_cells=n_cells, per_cell=per_cell, dt=5.0e-9 * crossings, collision_model="none")
    g = Case(spec, precision="fp32", capacity=int(1.3 * n_cells * per_cell) + 70000)
    g.fill(**fill)
    if variant >= 0:
        g.tile_select(variant)
    g.step(2 if variant >= 0 else 10)   # past the tuner's steps
    best = float("inf")
    for _ in range(steps):
        g.timing(True)
        g.step(1)
        g.sync()
        best = min(best, 1000.0 * g.phase_times()[0][phase])
    g.close()
    return best


def test_count_of_cells_crossed(require_gpu):
    """Simulators that crossed several cells are counted by atomics on 1000 counters,
    those that crossed none or one in LDS: two crossings per step take 1.1 times as
    long as next to none (2.9 with an atomic per simulator)."""
    assert phase_us(10000, 2, "scan", variant=1) < 1.7 * phase_us(10000, 0.02, "scan", variant=1)


def test_sums_of_many_hits_per_face(require_gpu):
    """Ten times the hits on the two faces of a channel (570 and 5700 each)."""
    assert phase_us(1000, 10, "wall") < 20.0 * phase_us(1000, 1, "wall")


def same_wall_sums(spec, fill, steps, capacity):
    """The wall sums after `steps` steps, equal to the oracle's; hits per face."""
    g = Case(spec, precision="fp64", capacity=capacity)
    o = OracleCase(spec, capacity=1 << 19)
    for c in (g, o):
        c.fill(**fill)
        c.step(steps)
    assert np.array_equal(g.wall_samples(), o.wall_samples())
    hits = g.counters()["wall_hits"] / steps / g.wall_face_count()
    g.close()
    o.close()
    return hits


@pytest.mark.parametrize("per_cell, least, most", [(420, 180, 250), (480, 230, 290), (1060, 470, 560),
                                                   (2100, 950, 1100), (10000, 4500, 5200)])
def test_order_of_many_hits(require_gpu, per_cell, least, most):
    """Faces of less and more hits than a wave orders at a time (256), odd and even
    numbers of stretches, one, two and several merges."""
    spec, fill = workloads.couette(n_cells=10, per_cell=per_cell, dt=5.0e-7, gas="Ar")
    spec.boundaries[1].kind = abi.BND_SPECULAR
    hits = same_wall_sums(spec, fill, 3, 1 << 20)
    assert least < hits < most, hits


def test_order_of_many_hits_on_many_faces(require_gpu):
    """More than 8192 faces, 16 lanes each, that order 64 hits at a time."""
    pt = {k: abi.WALL for k in ("xmin", "xmax", "ymin", "ymax", "zmin", "zmax")}
    mesh = box_mesh((0.0, 0.0, 0.0), (2.1, 1.0e-3, 1.0e-3), (2100, 1, 1), pt)
    spec = CaseSpec(mesh=mesh, species=[workloads.ARGON, workloads.N2], delta_t=2.0e-5, n_equivalent_particles=1.0e9,
                    collision_model="none", boundaries=[Boundary(p, abi.BND_SPECULAR) for p in pt])
    hits = same_wall_sums(spec, dict(number_density={"Ar": 2.0e19, "N2": 2.0e19}, T=300.0), 2, 1 << 23)
    assert 64 < hits < 256, hits


@pytest.mark.parametrize("per_cell", [70, 140, 270, 1100, 6000])
def test_merge_lists_match_oracle(require_gpu, per_cell):
    """Merge lists of some 60 to 6000 slots, sorted 64 at a time: one stretch, an odd
    and an even number of them."""
    spec, fill = workloads.heat_bath(n_cells=2, per_cell=per_cell, side=2.0e-3, dt=1.0e-5)
    g = Case(spec, precision="fp64", capacity=1 << 19)
    o = OracleCase(spec, capacity=1 << 19)
    for c in (g, o):
        c.fill(**fill)
    g.tile_select(3)
    for c in (g, o):
        c.step(3)
    pg, po = g.particles(), o.particles()
    for k in ("local", "velocity", "erot", "cell", "species"):
        assert np.array_equal(pg[k], po[k]), k
    g.close()
    o.close()


def test_merges_of_thousands_per_cell(require_gpu):
    """Cells of 10,000 simulators of which most are merged by slot: the form
    without tiles, whose merge lists have a wave, against tiles of 256 threads."""
    assert phase_us(10000, 5, "cells", variant=3) < phase_us(10000, 5, "cells", variant=1)


def test_slow_configurations_are_timed_once(require_gpu):
    """A dense world, where some configurations take milliseconds and more than twice
    the fastest, has its choice after fewer steps than two timings of all four would
    take; a small one, where a kernel's first launch may look as slow, times all twice."""
    spec, fill = workloads.couette(n_cells=20, per_cell=20, collision_model="none")
    g = Case(spec, precision="fp32", capacity=1000)
    g.fill(**fill)
    g.step(7)
    assert not g.tile_config()["tuned"]
    g.step(1)
    assert g.tile_config()["tuned"]
    g.close()
    spec, fill = workloads.couette(n_cells=1000, per_cell=10000, collision_model="none")
    g = Case(spec, precision="fp32", capacity=14000000)
    g.fill(**fill)
    g.step(7)
    assert g.tile_config()["tuned"]
    g.close()
