"""The radix sort and the scans behind the broadphase at the sizes where their
launches change: one workgroup up to 8,192 keys in four item counts, 4,096-key
tiles beyond, 4,096-element scan tiles. Box counts set the size of the body
sort and of the pair-count scan (six counts per box), the pair counts that of
the pair-key sort; pairs against the oracle's sweep, whole numbers exactly."""
import numpy as np
import pytest

import oracle_libs as L
import physx_amd as P
from physx_amd import scenes as S

pytestmark = pytest.mark.gpu


def _boxes(n, fill, seed, line=False):
    rng = np.random.default_rng(seed)
    side = (n * 0.512 / fill) ** (1 / 3)
    c = rng.uniform(0, side, (n, 3))
    if line:   # one row of boxes: every key in the same grid row, many equal coordinates
        c[:, 0] = np.floor(rng.uniform(0, n * 0.1, n) * 4) / 4
        c[:, 1:] = 0.25
    h = rng.uniform(0.1, 0.3, (n, 3))
    return np.concatenate([c - h, c + h], 1).astype(np.float32)


def _check(bp, bounds, prev, cuda):
    import torch
    n = len(bounds)
    dist = np.full(n, 0.02, np.float32)
    bp.update(torch.from_numpy(bounds).to(cuda), torch.from_numpy(dist).to(cuda),
              torch.arange(n, dtype=torch.int32, device=cuda))
    created, deleted = bp.fetch_results()
    want = np.asarray(L.bp_pairs_pxo(bounds, dist)).reshape(-1, 2).astype(np.int64)
    want = np.unique(np.sort(want, 1), axis=0)
    key = lambda p: np.asarray(p, np.int64)[:, 0] * (1 << 32) + np.asarray(p, np.int64)[:, 1]  # noqa: E731
    now = key(want)
    np.testing.assert_array_equal(key(created), np.setdiff1d(now, prev))
    np.testing.assert_array_equal(key(deleted), np.setdiff1d(prev, now))
    return now


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 682, 683, 1023, 1024, 1025, 2048, 2049, 4095, 4096, 4097, 8191, 8192,
                               8193, 12288, 12289, 20011])
def test_broadphase_sizes(cuda, n):
    bp = P.BroadPhase()
    prev = np.zeros(0, np.int64)
    for k in range(2):
        prev = _check(bp, _boxes(n, 4.0, n + k), prev, cuda)


@pytest.mark.parametrize("n", [300, 3000])
def test_broadphase_one_row(cuda, n):
    bp = P.BroadPhase()
    prev = np.zeros(0, np.int64)
    for k in range(2):
        prev = _check(bp, _boxes(n, 4.0, n + k, line=True), prev, cuda)


@pytest.mark.parametrize("n", [384 * 4096, 384 * 4096 + 1, 17_000_000])
def test_broadphase_many_tiles(cuda, n):
    """The last size whose sort tiles add up each other's counts, the first whose
    counts are scanned, and one whose pair counts take a scan of scanned sums (more
    than 4,096 tiles of 4,096): boxes in a shuffled order along rows, each one
    overlapping the next of its row and no other."""
    import torch
    row = 4096
    g = torch.Generator(device="cuda").manual_seed(n)
    place = torch.randperm(n, generator=g, device="cuda")   # box -> place
    x, y = (place % row).float(), (place // row).float() * 2.0
    z = torch.zeros_like(x)
    bounds = torch.stack([x - 0.6, y - 0.5, z - 0.5, x + 0.6, y + 0.5, z + 0.5], 1).contiguous()
    torch.cuda.synchronize()   # the update reads the bounds on its own stream
    bp = P.BroadPhase()
    bp.update(bounds)
    created, deleted = bp.fetch_results()
    box = torch.empty_like(place)
    box[place] = torch.arange(n, device="cuda")
    k = torch.arange(n - 1, device="cuda")
    k = k[k % row != row - 1]
    a, b = torch.minimum(box[k], box[k + 1]), torch.maximum(box[k], box[k + 1])
    want = torch.sort(a * (1 << 32) + b).values
    got = torch.from_numpy(created.astype(np.int64)).cuda()
    assert len(deleted) == 0
    assert torch.equal(got[:, 0] * (1 << 32) + got[:, 1], want)
    bp.close()


@pytest.mark.parametrize("per_body", [1, 800, 1000])
def test_constraint_list_many_tiles(cuda, per_body):
    """more contact slots than 4,096 tiles of 1,024 (from the room for pairs asked
    for): the same bits as with the least room"""
    sc = S.batched_piles(n_scenes=1, nmin=5000, nmax=5000, seed=5)
    a, b = P.Scene(sc), P.Scene(sc, max_pairs_per_body=per_body)
    for _ in range(12):
        a.step(1.0 / 60.0)
        b.step(1.0 / 60.0)
    assert a.stats()["constraints"] == b.stats()["constraints"] > 0
    for u, v in zip(a.bodies(), b.bodies()):
        np.testing.assert_array_equal(u, v)


@pytest.mark.parametrize("n", [2, 65, 700, 3000])
@pytest.mark.parametrize("extent", [(60.0, 0.0, 0.0), (20.0, 50.0, 0.0), (20.0, 0.0, 50.0), (10.0, 50.0, 50.0)])
def test_broadphase_few_rows(cuda, n, extent):
    """One box so wide that the grid has one, two or four rows: of a body's nine
    lanes in the sweep one, two or four have candidates, and only lanes before
    another one count theirs again to place them."""
    rng = np.random.default_rng(n)
    bp = P.BroadPhase()
    prev = np.zeros(0, np.int64)
    for _ in range(2):
        c = rng.uniform(0.0, 1.0, (n, 3)) * extent
        h = rng.uniform(0.1, 0.6, (n, 3))
        h[n // 2] = 20.0
        prev = _check(bp, np.concatenate([c - h, c + h], 1).astype(np.float32), prev, cuda)
    assert len(prev) > 0
