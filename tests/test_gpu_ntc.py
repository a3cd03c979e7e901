"""The single-precision decision of an NTC candidate over relative speeds from
nothing to far above thermal, and over the VHS exponents (omega = 0.5 hard
spheres, 1 Maxwell molecules, whose sigma c_r is a constant that ties with the
maximum): particles, maxima and counts equal the oracle's, bit for bit."""
import dataclasses

import numpy as np
import pytest

from oracle.orc import OracleCase
from unigasfoam_amd import workloads
from unigasfoam_amd.core import Case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("omega", [0.5, 0.81, 1.0])
@pytest.mark.parametrize("T, dt", [(1.0e-40, 1.0), (1.0e-4, 3.0e-3), (300.0, 2.0e-6), (3.0e8, 2.0e-9)])
def test_candidates_match_oracle(require_gpu, omega, T, dt):
    spec, fill = workloads.heat_bath(n_cells=3, per_cell=40, side=3.0e-3, n_density=4.0e21, dt=dt)
    spec.species = [dataclasses.replace(spec.species[0], omega=omega)]
    fill["T"] = T
    g = Case(spec, precision="fp64", capacity=1 << 14)
    o = OracleCase(spec, capacity=1 << 14)
    for c in (g, o):
        c.fill(**fill)
        c.step(6)
    pg, po = g.particles(), o.particles()
    for k in ("local", "velocity", "cell"):
        assert np.array_equal(pg[k], po[k]), k
    assert np.array_equal(g.sigma_max(), o.sigma_max())
    cg, co = g.counters(), o.counters()
    assert cg["candidates"] == co["candidates"] and cg["collisions"] == co["collisions"]
    if T >= 300.0:   # (Maxwell molecules collide a thousandth as often in the thousandth of the step)
        assert cg["collisions"] > (100 if T == 300.0 else 0)
    g.close()
    o.close()
