"""The move in FP32, bit for bit.  The oracle works in FP64, so the tracks are
restated here in numpy's float32, face by face and without the frame shift that
k_move holds back until the next cell's faces are requested."""
import dataclasses

import numpy as np
import pytest

from unigasfoam_amd import abi, core, workloads
from unigasfoam_amd.core import Case
from unigasfoam_amd.spec import Boundary, CaseSpec

pytestmark = pytest.mark.gpu
F = np.float32
MAX_CROSSINGS = 1000
EMPTY = -2 ** 31


def track(spec, x, v, cell, moves):
    """One step of the given simulators: (x, v, cell, crossings into another cell,
    mirror reflections, met a diffuse wall, ran out of crossings, sum of the change
    of speed along each axis at the mirror reflections)."""
    g = core.geometry(spec)
    planes, nbr, delta = g["planes"].astype(F), g["nbr"], g["delta"].astype(F)
    by_patch = {b.patch: b.kind for b in spec.boundaries}
    kinds = np.array([by_patch.get(p.name, -1) for p in spec.mesh.patches])
    x, v, cell = x.astype(F), v.astype(F), cell.copy()
    n = len(cell)
    tau = np.full(n, F(spec.delta_t), dtype=F)
    mask = np.array(moves, dtype=F)
    live = np.arange(n)
    crossed, hits = np.zeros(n, dtype=int), np.zeros(n, dtype=int)
    stopped, push = np.zeros(n, dtype=bool), np.zeros(3)
    with np.errstate(divide="ignore", invalid="ignore"):
        for _ in range(MAX_CROSSINGS):
            c = cell[live]
            vt = v[live] * mask
            tmin, face = tau[live].copy(), np.full(len(live), -1)
            for f in range(6):
                q = planes[c, f]
                dn = q[:, 0] * vt[:, 0] + q[:, 1] * vt[:, 1] + q[:, 2] * vt[:, 2]
                p = x[live]
                t = (q[:, 3] - (q[:, 0] * p[:, 0] + q[:, 1] * p[:, 1] + q[:, 2] * p[:, 2])) / dn
                t = np.where(t < F(0), F(0), t)
                take = (nbr[c, f] != EMPTY) & (dn > F(0)) & (t < tmin)
                tmin, face = np.where(take, t, tmin), np.where(take, f, face)
            x[live] = x[live] + vt * tmin[:, None]
            tau[live] = tau[live] - tmin
            go = face >= 0
            live, c, face = live[go], c[go], face[go]
            code = nbr[c, face]
            inner = code >= 0
            x[live[inner]] = x[live[inner]] + delta[c[inner], face[inner]]
            cell[live[inner]] = code[inner]
            crossed[live[inner]] += 1
            kind = np.where(inner, -1, kinds[np.where(inner, 0, -1 - code)])
            wall = kind == abi.BND_SPECULAR
            w, q = live[wall], planes[c[wall], face[wall]]
            u = v[w]
            udn = u[:, 0] * q[:, 0] + u[:, 1] * q[:, 1] + u[:, 2] * q[:, 2]
            v[w] = np.where(udn[:, None] > F(0), u - (F(2) * udn)[:, None] * q[:, :3], u)
            hits[w] += 1
            push += np.abs(u.astype(float) - v[w].astype(float)).sum(axis=0)
            stopped[live[kind == abi.BND_DIFFUSE]] = True
            live = live[kind != abi.BND_DIFFUSE]
            if len(live) == 0:
                break
    lost = np.zeros(n, dtype=bool)
    lost[live] = True
    return x, v, cell, crossed, hits, stopped, lost, push


def run(spec, fill, moves, capacity):
    """One step on the GPU and here: the start with every simulator's number in its
    E_rot (exact in FP32, kept by the move, cleared by a diffuse wall), the state
    after the step, and track()'s results."""
    spec = dataclasses.replace(spec, collision_model="none")
    g = Case(spec, precision="fp32", capacity=capacity)
    g.fill(**fill)
    p = g.particles()
    g.close()
    g = Case(spec, precision="fp32", capacity=capacity)
    g.upload(p["velocity"], p["cell"], erot=np.arange(1, len(p["cell"]) + 1, dtype=float), local=p["local"])
    start = g.particles()
    g.step(1)
    end, counters = g.particles(), g.counters()
    counters["push"] = np.abs(g.wall_samples()[:, :, abi.W_FX:abi.W_FX + 3]).sum(axis=(0, 1))
    g.close()
    return start, end, counters, track(spec, start["local"], start["velocity"], start["cell"], moves)


def assert_same(start, end, ref):
    x, v, cell, _, _, stopped = ref[:6]
    # the simulators that met no diffuse wall, in the order of the sort by cell
    ids = start["erot"].astype(int)
    row = np.full(ids.max() + 1, -1)
    row[ids] = np.arange(len(ids))
    got = end["erot"].astype(int)
    kept = got > 0
    r = row[got[kept]]
    assert np.array_equal(np.sort(r), np.flatnonzero(~stopped))
    assert np.array_equal(end["cell"][kept], cell[r])
    assert np.array_equal(end["local"][kept], x[r].astype(float))
    assert np.array_equal(end["velocity"][kept], v[r].astype(float))
    assert np.array_equal(r, r[np.lexsort((r, cell[r]))])


@pytest.mark.parametrize("n_cells, per_cell, dt", [
    (6, 40, 2.0e-6),      # none or one crossing
    (8, 100, 1.0e-5),     # several, and walls straight after them
    (3, 7, 5.0e-4),       # some 150 crossings and as many walls
    (3, 40, 3.0e-3),      # fast simulators run out of crossings
])
def test_box(require_gpu, n_cells, per_cell, dt):
    spec, fill = workloads.heat_bath(n_cells=n_cells, per_cell=per_cell, side=1.0e-3 * n_cells, dt=dt)
    start, end, counters, ref = run(spec, fill, (1, 1, 1), 1 << 23)
    assert_same(start, end, ref)
    assert counters["wall_hits"] == ref[4].sum()
    assert counters["track_errors"] == ref[6].sum()
    # the walls' time sums of the force density, F_N m (U_before - U_after) / A per
    # hit: sums in FP64 of FP32 velocities, in another order (at most 1e5 hits per
    # face: 1e5 x 2^-53 is about 1e-11)
    assert counters["push"] == pytest.approx(ref[7] * spec.n_equivalent_particles * workloads.ARGON.mass / 1.0e-6,
                                             rel=1.0e-10)
    assert (counters["track_errors"] > 0) == (dt > 1.0e-3)
    assert dt < 5.0e-6 or np.any((ref[3] > 1) & (ref[4] > 0))


def test_oblique_faces(require_gpu):
    """Cells of the nozzle's mesh, all walls specular."""
    mesh = workloads.nozzle_mesh(12, 6, 6)
    for p in mesh.patches:
        p.type = abi.WALL
    spec = CaseSpec(mesh=mesh, species=[workloads.ARGON], delta_t=8.0e-6, n_equivalent_particles=2.0e10,
                    collision_model="none", boundaries=[Boundary(p.name, abi.BND_SPECULAR) for p in mesh.patches])
    start, end, counters, ref = run(spec, dict(number_density={"Ar": 1.0e21}, T=600.0), (1, 1, 1), 1 << 20)
    assert len(start["cell"]) > 5000 and ref[3].max() > 3
    assert_same(start, end, ref)
    assert counters["wall_hits"] == ref[4].sum()


def test_channel_with_a_diffuse_wall(require_gpu):
    """Stopped tracks and mirrored ones in one stage, cyclic faces, one moving direction masked."""
    spec, fill = workloads.couette(n_cells=30, per_cell=300, dt=2.0e-7, gas="Ar", periodic="empty")
    spec.boundaries[1].kind = abi.BND_SPECULAR
    start, end, counters, ref = run(spec, fill, (0, 1, 0), 1 << 18)
    assert 50 < ref[5].sum() < len(ref[5]) // 2 and ref[4].sum() > 50
    assert_same(start, end, ref)
