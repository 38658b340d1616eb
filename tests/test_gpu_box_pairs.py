"""Box-box and plane-box contact generation where a wave shares the search of
several pairs: pair counts around the wave size and pairs that mostly end in
the edge search (clipping leaves no point), against the C oracle. The device
code keeps the oracle's operations and their order with correctly rounded
division and square root, so a few units in the last place of coordinates
below 2 m (2e-7 each) bound the difference."""
import numpy as np
import pytest

import oracle_libs as L
import physx_amd as P

pytestmark = pytest.mark.gpu

BOX, PLANE = P.PXH_GEOM_BOX, P.PXH_GEOM_PLANE


def _quat(rng, n):
    q = rng.normal(size=(n, 4))
    return q / np.linalg.norm(q, axis=1, keepdims=True)


def _pairs(n, seed, lo, hi):
    rng = np.random.default_rng(seed)
    g0, g1 = np.zeros((n, 4)), np.zeros((n, 4))
    g0[:, :3], g1[:, :3] = rng.uniform(0.1, 0.3, (n, 3)), rng.uniform(0.1, 0.3, (n, 3))
    p0 = np.concatenate([rng.uniform(-1, 1, (n, 3)), _quat(rng, n)], 1)
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    p1 = np.concatenate([p0[:, :3] + d * rng.uniform(lo, hi, (n, 1)), _quat(rng, n)], 1)
    f = lambda a: a.astype(np.float32)  # noqa: E731
    return f(g0), f(p0), f(g1), f(p1)


def _compare(t0, g0, p0, t1, g1, p1):
    n = len(t0)
    cnt, out = P.generate_contacts(t0, g0, p0, t1, g1, p1)
    for i in range(n):
        want = L.contacts("pxo", int(t0[i]), g0[i], p0[i], int(t1[i]), g1[i], p1[i])
        assert int(cnt[i]) == len(want), f"pair {i}"
        np.testing.assert_allclose(out[i, :len(want), :7], want[:, :7], atol=2e-6, err_msg=f"pair {i}")
    return cnt


@pytest.mark.parametrize("n", [1, 2, 5, 63, 64, 65, 191, 500])
@pytest.mark.parametrize("share", [1, 9])
def test_box_box_edge_search(cuda, n, share):
    """pairs with a single contact (nearly all of them from the edge search,
    which a few percent of random pairs reach), every pair or one in `share`"""
    g0, p0, g1, p1 = _pairs(60000, 3, 0.3, 0.62)
    t = np.full(60000, BOX, np.int32)
    cnt, _ = P.generate_contacts(t, g0, p0, t, g1, p1)
    one, many = np.flatnonzero(cnt == 1), np.flatnonzero(cnt != 1)
    assert len(one) >= 500
    idx = np.where(np.arange(n) % share == share - 1, one[:n], many[:n])
    _compare(t[:n], g0[idx], p0[idx], t[:n], g1[idx], p1[idx])


@pytest.mark.parametrize("n", [64, 700])
def test_box_box_deep_and_degenerate(cuda, n):
    """overlapping boxes with many clip points, some axis-aligned, equal and
    concentric: ties between features and coplanar faces"""
    g0, p0, g1, p1 = _pairs(n, 7 + n, 0.0, 0.3)
    ident = np.array([0, 0, 0, 1], np.float32)
    p0[::3, 3:], p1[::3, 3:] = ident, ident
    g1[::4] = g0[::4]
    p1[::7, :3] = p0[::7, :3]
    p1[1::5, :3] = p0[1::5, :3] + np.float32([0.0, 0.4, 0.0])
    t = np.full(n, BOX, np.int32)
    _compare(t, g0, p0, t, g1, p1)


@pytest.mark.parametrize("n", [1, 65, 500])
def test_plane_box_more_than_four_corners(cuda, n):
    """thin boxes near the plane: five to eight corners within the contact
    distance, reduced to four"""
    g0, p0, g1, p1 = _pairs(n, 31 + n, 0.0, 0.05)
    g0[:] = 0.0
    g1[:, 1] = 0.01
    p1[::2, 3:] = p0[::2, 3:]
    t0, t1 = np.full(n, PLANE, np.int32), np.full(n, BOX, np.int32)
    _compare(t0, g0, p0, t1, g1, p1)
