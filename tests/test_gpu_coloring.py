"""Colouring of new constraints against the oracle where its path changes:
lists that one workgroup takes and longer ones, a list that turns out longer
than the step before suggested, and bodies with more constraints than the 64
colours a mask holds (further rounds, colours past 63, a body-plane colour
after them). Colours are whole numbers and compared exactly."""
import numpy as np
import pytest

import oracle_libs as L
import physx_amd as P
from physx_amd import scenes as S

pytestmark = pytest.mark.gpu

DT = 1.0 / 60.0


def _spheres(pos, radius, planes):
    n = len(pos)
    t = np.full(n, S.SPHERE, np.int32)
    dims = np.zeros((n, 4), np.float32)
    dims[:, 0] = radius
    pose = np.concatenate([pos, np.tile([0.0, 0.0, 0.0, 1.0], (n, 1))], 1).astype(np.float32)
    m, inn = S.mass_props(t, dims, 1000.0)
    z = np.zeros((n, 3), np.float32)
    pl = np.asarray(planes, np.float32).reshape(-1, 4)
    return S.Scene(t, dims, pose, z, z.copy(), m, inn, np.zeros(n, np.int32), pl, np.zeros(len(pl), np.int32), 1,
                   "spheres", {})


def _row(n, gap):
    """a row of unit spheres: touching neighbours, or far apart from index `gap` on"""
    x = np.arange(n) * 0.99
    x[gap:] += np.arange(n - gap) * 3.0
    return np.stack([x, np.full(n, 5.0), np.zeros(n)], 1)


def _same(g, o):
    a, b = g.constraints(), np.asarray(o.constraints())
    order = lambda t: t[np.lexsort((t[:, 1], t[:, 0]))]  # noqa: E731
    np.testing.assert_array_equal(order(a)[:, :3], order(b)[:, :3])
    np.testing.assert_allclose(g.bodies()[1], o.bodies()[1], atol=1e-5)


@pytest.mark.parametrize("solver", ["tgs", "pgs"])
@pytest.mark.parametrize("n", [2, 2048, 2049, 2050, 4000])
def test_first_step_lists(cuda, n, solver):
    sc = _spheres(_row(n, n), 0.5, [])
    g = P.Scene(sc, position_iterations=4, velocity_iterations=1,
                solver_type=P.PXH_SOLVER_PGS if solver == "pgs" else P.PXH_SOLVER_TGS)
    o = L.OracleWorld(sc, pos_iters=4, vel_iters=1, solver=solver)
    for _ in range(2):
        g.step(DT, 1)
        o.step(DT, 1)
        assert g.stats()["constraints"] == n - 1
        _same(g, o)


def test_list_longer_than_expected(cuda):
    n = 3000
    sc = _spheres(_row(n, 10), 0.5, [])
    g = P.Scene(sc, position_iterations=4, velocity_iterations=1)
    o = L.OracleWorld(sc, pos_iters=4, vel_iters=1)
    g.step(DT, 1)
    o.step(DT, 1)
    _same(g, o)
    pose = _spheres(_row(n, n), 0.5, []).pose
    z = np.zeros((n, 3), np.float32)
    for w in (g, o):
        w.set_bodies(pose, z, z)
    for _ in range(2):
        g.step(DT, 1)
        o.step(DT, 1)
        _same(g, o)


@pytest.mark.parametrize("solver", ["tgs", "pgs"])
@pytest.mark.parametrize("around", [20, 63, 64, 65, 150])
def test_more_constraints_than_mask_colours(cuda, around, solver):
    """a large sphere on the floor with `around` small ones on its surface"""
    k = np.arange(around)
    y = 0.9 - 1.2 * (k + 0.5) / around
    phi = k * 2.399963
    r = np.sqrt(1.0 - y * y)
    d = np.stack([r * np.cos(phi), y, r * np.sin(phi)], 1)
    pos = np.concatenate([[[0.0, 2.0, 0.0]], [0.0, 2.0, 0.0] + d * 2.05])
    sc = _spheres(pos, 0.06, [[0, 1, 0, 0]])
    sc.dims[0, 0] = 2.0
    sc.mass[:], sc.inertia[:] = S.mass_props(sc.shape_type, sc.dims, 1000.0)
    g = P.Scene(sc, position_iterations=4, velocity_iterations=1,
                solver_type=P.PXH_SOLVER_PGS if solver == "pgs" else P.PXH_SOLVER_TGS)
    g.set_tuning(layout=P.PXH_SOLVE_LAYOUT_COLORS)
    o = L.OracleWorld(sc, pos_iters=4, vel_iters=1, solver=solver)
    for _ in range(3):
        g.step(DT, 1)
        o.step(DT, 1)
        assert g.stats()["constraints"] >= around + 1
        _same(g, o)
