"""Sampler downloads (rows over cells) equal the restart state's sums (cells
over rows, copied as they lie): one copy, several threads' ranges, more ranges
than the staging memory holds, and two threads at once."""
import threading

import numpy as np
import pytest

from unigasfoam_amd import workloads
from unigasfoam_amd.batch import Batch
from unigasfoam_amd.core import Case

pytestmark = pytest.mark.gpu


def bath(shape_n, per_cell, seed=1):
    return workloads.heat_bath(n_cells=shape_n, per_cell=per_cell, side=1.0e-3 * shape_n, seed=seed)


@pytest.mark.parametrize("n", [1, 3, 4, 15, 16, 39])   # 1, 27, 64, 3375, 4096, 59319 cells (288 bytes each)
def test_download_equals_state(require_gpu, n):
    spec, fill = bath(n, 3)
    g = Case(spec)
    g.fill(**fill)
    g.step(3)
    s = g.state()["samples"].reshape(n ** 3, -1)
    d = g.samples()
    assert d[0].sum() > 0.0 and np.array_equal(d, s.T)
    g.step(2)
    assert np.array_equal(g.samples(), g.state()["samples"].reshape(n ** 3, -1).T)
    g.close()


@pytest.mark.parametrize("n", [6, 17])
def test_two_threads_on_one_world(require_gpu, n):
    b = Batch(precision="fp64")
    slots = [b.admit(*bath(n - k, 4, seed=5 + k), 5 * n ** 3) for k in range(2)]
    b.step(4)
    b.sync()
    want = [b.case(s).samples() for s in slots]
    got = [[], []]

    def read(k):
        for _ in range(10):
            got[k].append(b.case(slots[k]).samples())
    th = [threading.Thread(target=read, args=(k,)) for k in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for k in range(2):
        assert len(got[k]) == 10 and all(np.array_equal(x, want[k]) for x in got[k])
    b.close()
