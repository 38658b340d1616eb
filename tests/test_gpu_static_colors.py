"""Colours of bodies that touch planes and a mesh at once: no two constraints of
a body share a colour, and constraints and colours equal the oracle's, exactly;
also past the 64 colours of a mask."""
import numpy as np
import pytest

import oracle_libs as L
import physx_amd as P
from physx_amd import scenes as S
from test_cpu_mesh import IDENT, _flat_grid

pytestmark = pytest.mark.gpu

DT = 1.0 / 60.0
WALLS = [[1, 0, 0, 2.0], [0, 0, 1, 2.0], [0, 1, 0, 0.01], [-1, 0, 0, 2.0]]


def _scene(t, dims, pos, walls):
    n = len(t)
    pose = np.concatenate([pos, np.tile([0.0, 0.0, 0.0, 1.0], (n, 1))], 1).astype(np.float32)
    m, inn = S.mass_props(t, dims, 1000.0)
    z = np.zeros((n, 3), np.float32)
    pl = np.asarray(WALLS[:walls], np.float32).reshape(-1, 4)
    V, T = _flat_grid()
    sc = S.Scene(t, dims, pose, z, z.copy(), m, inn, np.zeros(n, np.int32), pl, np.zeros(len(pl), np.int32), 1,
                 "corner", {})
    sc.meshes = [dict(verts=V, tris=T, pose=IDENT, world=0)]
    return sc


def _run(sc, solver, layout, steps=3):
    g = P.Scene(sc, position_iterations=4, velocity_iterations=1,
                solver_type=P.PXH_SOLVER_PGS if solver == "pgs" else P.PXH_SOLVER_TGS)
    g.set_tuning(layout=layout)
    o = L.OracleWorld(sc, pos_iters=4, vel_iters=1, solver=solver)
    for _ in range(steps):
        g.step(DT)
        o.step(DT)
        a, b = g.constraints(), np.asarray(o.constraints())
        order = lambda t: t[np.lexsort((t[:, 1], t[:, 0]))]  # noqa: E731
        np.testing.assert_array_equal(order(a)[:, :3], order(b)[:, :3])
        held = np.concatenate([a[:, [0, 2]], a[a[:, 1] >= 0][:, [1, 2]]])
        assert len(np.unique(held, axis=0)) == len(held)
        np.testing.assert_allclose(g.bodies()[1], o.bodies()[1], atol=1e-5)
    return a


@pytest.mark.parametrize("layout", [P.PXH_SOLVE_LAYOUT_COLORS, P.PXH_SOLVE_LAYOUT_WORLDS])
@pytest.mark.parametrize("solver", ["tgs", "pgs"])
@pytest.mark.parametrize("walls,bodies", [(0, 6), (1, 1), (1, 2), (2, 1), (3, 9), (4, 14)])
def test_plane_and_mesh_on_one_body(cuda, walls, bodies, solver, layout):
    """boxes and spheres in a row along a wall of a mesh floor, each touching the
    floor, the wall and its neighbours, the first one the corner's walls"""
    i = np.arange(bodies)
    t = np.where(i % 2 == 0, S.BOX, S.SPHERE).astype(np.int32)
    dims = np.zeros((bodies, 4), np.float32)
    dims[t == S.BOX, :3] = 0.25
    dims[t == S.SPHERE, 0] = 0.25
    pos = np.stack([-1.76 + 0.0 * i, np.full(bodies, 0.245), -1.76 + 0.495 * i], 1)
    con = _run(_scene(t, dims, pos, walls), solver, layout)
    n_static = (con[:, 1] < 0).sum()
    assert n_static >= bodies * (1 + (walls > 0))


@pytest.mark.parametrize("solver", ["tgs", "pgs"])
@pytest.mark.parametrize("around", [62, 64, 150])
def test_mesh_patches_past_the_mask(cuda, around, solver):
    """a large sphere on a mesh floor, beside two walls, with `around` small
    spheres on its surface"""
    k = np.arange(around)
    y = 0.9 - 1.2 * (k + 0.5) / around
    phi = k * 2.399963
    r = np.sqrt(1.0 - y * y)
    d = np.stack([r * np.cos(phi), y, r * np.sin(phi)], 1)
    c = np.array([0.0, 2.0, 0.0])
    t = np.full(around + 1, S.SPHERE, np.int32)
    dims = np.zeros((around + 1, 4), np.float32)
    dims[:, 0] = 0.06
    dims[0, 0] = 2.0
    con = _run(_scene(t, dims, np.concatenate([[c], c + d * 2.05]), 2), solver, P.PXH_SOLVE_LAYOUT_COLORS)
    assert len(con) >= around + 2
