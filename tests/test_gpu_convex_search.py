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
