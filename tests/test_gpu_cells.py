"""The form of the cells phase without tiles (k_order, k_gather_all,
k_cell_sums): the tuner runs it on a world's fourth step, so the state after
five steps has been through it and through every tile configuration.
"""
import numpy as np
import pytest

from oracle.orc import OracleCase
from unigasfoam_amd import workloads
from unigasfoam_amd.core import Case, UgxError

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


def world(kind, precision, graphs=False):
    if kind == "cylinder":     # two species, inflow, cells of no to 400 simulators
        spec, fill = workloads.cylinder(n_theta=24, n_r=10, target=24 * 10 * 200.0, dt=2.0e-6)
    elif kind == "channel":    # second and third moments, BGK moments
        spec, fill = workloads.couette(n_cells=30, per_cell=90, dt=2.0e-8, collision_model="bgk",
                                       bgk_model="unifiedStochasticParticleSBGK")
        spec.sampler_full = True
    else:                      # most simulators cross several cells
        spec, fill = workloads.heat_bath(n_cells=4, per_cell=500, side=4.0e-3, dt=1.0e-5)
    g = Case(spec, precision=precision, capacity=1 << 18, use_graphs=graphs)
    g.fill(**fill)
    return g, spec, fill


def state(g):
    p = g.particles()
    return [p[k] for k in ("local", "velocity", "erot", "cell", "species")] + [g.samples(), g.sigma_max()]


@pytest.mark.parametrize("kind", ["cylinder", "channel", "bath"])
@pytest.mark.parametrize("variant", [0, 1, 2, 3])
def test_configuration_matches_oracle(require_gpu, kind, variant):
    """Every step in one configuration."""
    g, spec, fill = world(kind, "fp64")
    g.tile_select(variant)
    assert g.tile_config()["variant"] == variant and g.tile_config()["tuned"]
    g.step(6)
    o = OracleCase(spec, capacity=1 << 18)
    o.fill(**fill)
    o.step(6)
    po = o.particles()
    want = [po[k] for k in ("local", "velocity", "erot", "cell", "species")] + [o.samples(), o.sigma_max()]
    for a, b in zip(state(g), want):
        assert np.array_equal(a, b)
    assert g.tile_config()["variant"] == variant
    g.close()
    o.close()


@pytest.mark.parametrize("kind", ["cylinder", "channel", "bath"])
def test_configurations_agree_in_fp32(require_gpu, kind):
    """The same bits from every configuration, launched and replayed."""
    want = None
    for variant in (0, 1, 2, 3):
        for graphs in (False, True):
            g, _, _ = world(kind, "fp32", graphs)
            g.tile_select(variant)
            g.step(9)
            got = state(g)
            want = want or got
            for a, b in zip(got, want):
                assert np.array_equal(a, b), (variant, graphs)
            g.close()


def test_unknown_configuration_is_refused(require_gpu):
    g, _, _ = world("bath", "fp64")
    for variant in (-2, 4):
        with pytest.raises(UgxError):
            g.tile_select(variant)
    g.tile_select(-1)
    assert not g.tile_config()["tuned"]
    g.close()
