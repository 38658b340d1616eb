"""The separation search of box- and convex-convex pairs at the sizes where its
lanes and lists have edges (8 lanes a pair in the support steps with 4 vertices
each in registers; 64 A edges a block and 32 B arcs a piece in the edge search),
over pairs that overlap, touch and lie just apart: the pairs with contacts, their
counts, normals and points against the oracle's, with the tolerances of the
convex one-step tests."""
import numpy as np
import pytest

import oracle_libs as L
import physx_amd as P
from physx_amd import scenes as S
from test_gpu_convex import DT, _compare_contacts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_points,pitch", [(4, 0.5), (5, 0.55), (8, 0.65), (9, 0.7), (17, 0.8), (24, 0.75),
                                            (24, 0.9), (32, 0.8), (33, 0.9), (64, 0.8), (64, 0.9), (70, 0.85)])
def test_convex_search_matches_oracle(cuda, n_points, pitch):
    sc = S.convex_layers(n_bodies=216, per_side=6, pitch=pitch, n_points=n_points, seed=n_points)
    box = np.arange(sc.n) % 3 == 1
    sc.shape_type[box] = S.BOX
    sc.dims[box, :3] = np.random.default_rng(n_points).uniform(0.15, 0.4, (int(box.sum()), 3))
    m, inn = S.mass_props(np.full(sc.n, S.BOX, np.int32), np.abs(sc.dims) + 0.1, 1000.0)
    sc.mass[box], sc.inertia[box] = m[box], inn[box]
    g = P.Scene(sc, position_iterations=4, velocity_iterations=1)
    o = L.OracleWorld(sc, pos_iters=4, vel_iters=1)
    g.step(DT)
    o.step(DT)
    assert g.stats()["bp_pairs"] == o.stats()["bp_pairs"]
    n = _compare_contacts(g, o)
    print(n_points, pitch, g.stats()["bp_pairs"], "pairs,", n, "with contacts", flush=True)
    assert 40 < n < g.stats()["bp_pairs"]


@pytest.mark.parametrize("n_points,pitch", [(4, 0.5), (16, 0.7), (40, 0.65), (90, 0.7)])
def test_round_convex_matches_oracle(cuda, n_points, pitch):
    """Spheres and capsules among hulls, apart, touching and inside."""
    sc = S.convex_layers(n_bodies=216, per_side=6, pitch=pitch, n_points=n_points, seed=n_points)
    i = np.arange(sc.n)
    ball, cap = i % 3 == 1, i % 3 == 2
    rng = np.random.default_rng(n_points)
    sc.shape_type[ball], sc.shape_type[cap] = S.SPHERE, S.CAPSULE
    sc.dims[ball, 0] = rng.uniform(0.1, 0.35, int(ball.sum()))
    sc.dims[cap, 0] = rng.uniform(0.05, 0.2, int(cap.sum()))
    sc.dims[cap, 1] = rng.uniform(0.05, 0.4, int(cap.sum()))
    g = P.Scene(sc, position_iterations=4, velocity_iterations=1)
    o = L.OracleWorld(sc, pos_iters=4, vel_iters=1)
    g.step(DT)
    o.step(DT)
    n = _compare_contacts(g, o)
    print(n_points, pitch, g.stats()["bp_pairs"], "pairs,", n, "with contacts", flush=True)
    assert 40 < n < g.stats()["bp_pairs"]


def test_pairs_about_the_contact_distance_match_oracle(cuda):
    """1,000 pairs of hulls whose vertices are, along the line of their centres, a
    little less, as much or a little more than the contact distance apart:
    whichever the separation search keeps or drops, the support steps, bounding
    spheres and feature bounds before it decide alike. Odd pairs are a hull and a
    capsule."""
    n = 2000
    sc = S.convex_layers(n_bodies=n, per_side=40, n_points=24, seed=21)
    off = np.concatenate([[0], np.cumsum(sc.hull_counts)])
    rng = np.random.default_rng(5)
    cd = 0.04   # two contact offsets

    def turned(i):
        pts = P.cook_convex(sc.hull_points[off[i]:off[i + 1]])["verts"].astype(np.float64)
        q, x = sc.pose[i, 3:6].astype(np.float64), float(sc.pose[i, 6])
        return pts + 2.0 * np.cross(q, np.cross(q, pts) + x * pts)

    for k in range(0, n, 2):
        a, b = k, k + 1
        va = turned(a)
        if k % 4 == 2:
            sc.shape_type[b] = S.CAPSULE
            sc.dims[b] = (0.2, 0.3, 0.0, 0.0)
            reach = 0.5
            sc.pose[b, 3:7] = (0.0, 0.0, 0.0, 1.0)
        else:
            reach = -turned(b)[:, 0].min()
        x = (k // 2) % 32 * 8.0
        y, z = (k // 64) % 32 * 8.0, 0.0
        sc.pose[a, :3] = (x, y, z)
        sc.pose[b, :3] = (x + va[:, 0].max() + reach + cd + rng.uniform(-3e-3, 2e-3), y, z)
    sc.planes, sc.plane_scene = np.zeros((0, 4), np.float32), np.zeros(0, np.int32)
    sc.lin_vel[:], sc.ang_vel[:] = 0.0, 0.0
    g = P.Scene(sc, position_iterations=4, velocity_iterations=1)
    o = L.OracleWorld(sc, pos_iters=4, vel_iters=1)
    g.step(DT)
    o.step(DT)
    assert _compare_contacts(g, o) > 0
    print(g.stats()["bp_pairs"], "pairs,", g.stats()["constraints"], "with contacts", flush=True)


@pytest.mark.parametrize("scale", [0.01, 1.0, 100.0, 1e4, 1e5])
def test_parallel_faces_at_scale_match_oracle(cuda, monkeypatch, scale):
    """400 pairs of bricks with facing faces parallel and less than the contact
    distance apart, lengths in units from 100 m to 10 um: every vertex and
    edge of the facing faces lies at the distance itself, so a feature bound that
    is tighter than the rounding of a height drops them (with a margin of 1e-4
    at every size 6 pairs lost their contact at 1e4 and 1 at 1e5). The tolerances
    scale with the lengths; the rounding of coordinates of 1.5 lengths is 1e-7 of them."""
    pairs = 400
    rng = np.random.default_rng(17)
    half = rng.uniform(0.2, 0.6, (2 * pairs, 3)) * scale
    corner = np.array([[x, y, z] for x in (-1, 1) for y in (-1, 1) for z in (-1, 1)], np.float64)
    pts = (half[:, None, :] * corner).astype(np.float32)
    q = rng.normal(size=(pairs, 4))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    cd = 0.04 * scale
    d = np.zeros((pairs, 3))
    d[:, 0] = half[::2, 0] + half[1::2, 0] + rng.uniform(0.05, 0.95, pairs) * cd
    d[:, 1:] = rng.uniform(-0.15, 0.15, (pairs, 2)) * scale
    qv, w = q[:, :3], q[:, 3:]
    t = 2.0 * np.cross(qv, d)
    at = d + w * t + np.cross(qv, t)
    n = 2 * pairs
    pose = np.zeros((n, 7), np.float32)
    pose[1::2, :3] = at
    pose[::2, 3:] = q
    # the second brick turned about the line between the faces
    a = rng.uniform(0.0, np.pi, (pairs, 1))
    sx, cx = np.sin(a), np.cos(a)
    x, y, z_, w_ = (q[:, k:k + 1] for k in range(4))
    pose[1::2, 3:] = np.concatenate([x * cx + w_ * sx, y * cx + z_ * sx, z_ * cx - y * sx, w_ * cx - x * sx], 1)
    dims = np.zeros((n, 4), np.float32)
    dims[:, 0] = np.arange(n)
    m, inn = S.mass_props(np.full(n, S.BOX, np.int32), np.concatenate([half, half[:, :1]], 1), 1000.0 / scale**3)
    z = np.zeros((n, 3), np.float32)
    sc = S.Scene(np.full(n, S.CONVEX, np.int32), dims, pose, z, z.copy(), m, inn,
                 np.repeat(np.arange(pairs, dtype=np.int32), 2), np.zeros((0, 4), np.float32), np.zeros(0, np.int32),
                 pairs, "bricks", {}, pts.reshape(-1, 3), np.full(n, 8, np.int32))
    desc = L.default_desc

    def scaled(*a):
        c = desc(*a)
        c.contact_offset, c.tolerance_length = 0.02 * scale, scale
        return c

    monkeypatch.setattr(L, "default_desc", scaled)
    g = P.Scene(sc, position_iterations=4, velocity_iterations=1, contact_offset=0.02 * scale, tolerance_length=scale)
    o = L.OracleWorld(sc, pos_iters=4, vel_iters=1)
    g.step(DT)
    o.step(DT)
    assert _compare_contacts(g, o, tol_p=1e-4 * scale) == pairs


@pytest.mark.parametrize("capsules", [False, True])
def test_round_shapes_inside_planes_past_the_vertices(cuda, monkeypatch, capsules):
    """Merged faces of thin blades have planes that meet well outside the hull's
    vertices, farther from its origin than any of them. A small sphere or capsule
    there is inside every plane and has its contact, though the bounding spheres are
    apart."""
    from scipy.spatial import HalfspaceIntersection
    r, cd = 0.001, 0.002
    hulls, at = [], []
    # blades (about one in a thousand) that have such a place within their vertices'
    # box, where the broadphase reports the pair, and past their bounding sphere by
    # more than four times what the planes lie off the vertices
    for points, seed in [(10, 3345), (10, 3851), (10, 3949), (10, 3979), (12, 1244), (12, 1611), (12, 2076),
                         (12, 2468), (12, 3143), (12, 3180), (12, 3979)]:
        v = np.random.default_rng(seed).normal(size=(points, 3))
        v = (v / np.linalg.norm(v, axis=1, keepdims=True) * [0.8, 0.5, 0.015]).astype(np.float32)
        h = P.cook_convex(v)
        pl = np.asarray(h["planes"], np.float64).reshape(-1, 4)
        w = np.asarray(h["verts"], np.float64).reshape(-1, 3)
        face = np.repeat(np.arange(len(pl)), h["poly_counts"])
        slack = -((w[h["vrefs"]] * pl[face, :3]).sum(1) + pl[face, 3]).min()
        c = HalfspaceIntersection(pl, w.mean(0)).intersections * (1.0 - 1e-3)
        far = np.linalg.norm(c, axis=1) > np.linalg.norm(w, axis=1).max() + r + cd + 4.0 * slack + 1e-4
        box = ((c > w.min(0) - r) & (c < w.max(0) + r)).all(1)
        c = c[far & box]
        hulls += [np.concatenate([v, np.repeat(v[:1], 12 - points, 0)])] * len(c)
        at += list(c)
    n = 2 * len(at)
    t = np.full(n, S.CONVEX, np.int32)
    dims = np.zeros((n, 4), np.float32)
    dims[::2, 0] = np.arange(len(at))
    t[1::2] = S.CAPSULE if capsules else S.SPHERE
    dims[1::2, 0] = r
    if capsules:
        dims[1::2, 1] = 1e-4
    pose = np.zeros((n, 7), np.float32)
    pose[:, 6] = 1.0
    pose[1::2, :3] = at
    m, inn = S.mass_props(np.full(n, S.BOX, np.int32), np.full((n, 4), 0.3, np.float32), 1000.0)
    z = np.zeros((n, 3), np.float32)
    sc = S.Scene(t, dims, pose, z, z.copy(), m, inn, np.repeat(np.arange(len(at), dtype=np.int32), 2),
                 np.zeros((0, 4), np.float32), np.zeros(0, np.int32), len(at), "blades", {}, np.concatenate(hulls),
                 np.full(len(at), 12, np.int32))
    desc = L.default_desc

    def small(*a):
        d = desc(*a)
        d.contact_offset = cd / 2
        return d

    monkeypatch.setattr(L, "default_desc", small)
    g = P.Scene(sc, position_iterations=4, velocity_iterations=1, contact_offset=cd / 2)
    o = L.OracleWorld(sc, pos_iters=4, vel_iters=1)
    g.step(DT)
    o.step(DT)
    assert _compare_contacts(g, o) >= 11
