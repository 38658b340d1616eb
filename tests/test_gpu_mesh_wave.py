"""Body-mesh contacts at the sizes where the wave's parts have edges: few
triangles a body, more than one round of polytope triangles (16), spheres and
capsules over up to and past 64 triangles (past them the lane form), and more
patches than are kept, against the oracle as in the resting test."""
import numpy as np
import pytest

import oracle_libs as L
import physx_amd as P
from physx_amd import scenes as S
from test_cpu_mesh import IDENT
from test_gpu_mesh import DT, _by_body

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cell,amp", [(2.0, 0.2), (0.5, 0.3), (0.25, 0.1), (0.25, 0.6), (0.18, 0.15), (0.15, 0.05)])
def test_mesh_contacts_by_triangle_size(cuda, cell, amp):
    sc = S.mixed_pile(n_bodies=64, per_side=8, pitch=2.0, n_points=16, seed=3)
    size, a = 20.0, 0.4
    verts, tris = S.terrain_mesh(int(round(size / cell)), size, amp, 5)
    t = sc.shape_type
    sc.dims[t == S.SPHERE, 0] = a
    sc.dims[t == S.CAPSULE, :2] = (0.2, 0.2)
    sc.dims[t == S.BOX, :3] = (a * 0.8, a * 0.6, a * 0.7)
    i = np.arange(sc.n)
    rng = np.random.default_rng(11)
    xz = np.stack([(i % 8 - 3.5) * 2.0, (i // 8 - 3.5) * 2.0], 1) + rng.uniform(-0.3, 0.3, (sc.n, 2))
    near = ((verts[None, :, ::2] - xz[:, None]) ** 2).sum(2).argmin(1)
    sc.pose[:, 0], sc.pose[:, 2] = xz[:, 0], xz[:, 1]
    sc.pose[:, 1] = verts[near, 1] + rng.uniform(0.15, 0.4, sc.n)
    sc.lin_vel[:], sc.ang_vel[:] = 0.0, 0.0
    sc.planes, sc.plane_scene = np.zeros((0, 4), np.float32), np.zeros(0, np.int32)
    sc.meshes = [dict(verts=verts, tris=tris, pose=IDENT, world=0)]
    g = P.Scene(sc)
    g.step(DT)
    o = L.OracleWorld(sc)
    o.step(DT)
    gs, os_ = g.stats(), o.stats()
    print(cell, amp, gs["constraints"], "constraints", flush=True)
    assert gs["constraints"] == os_["constraints"] > 40, (gs, os_)
    gc, oc = _by_body(g.contact_data()), _by_body(o.contact_data())
    assert sorted(gc) == sorted(oc)
    bad = [k for k in gc if L.same_contacts(L.dedupe(gc[k]), L.dedupe(oc[k]))]
    assert not bad, [(k, int(t[k])) for k in bad[:8]]
