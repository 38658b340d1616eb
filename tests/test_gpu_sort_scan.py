"""The radix sort and the scans behind the broadphase at the sizes where their
launches change: one workgroup up to 8,192 keys in four item counts, 4,096-key
tiles beyond, 4,096-element scan tiles. Box counts set the size of the body
sort and of the pair-count scan (six counts per box), the pair counts that of
the pair-key sort; pairs against the oracle's sweep, whole numbers exactly."""
import numpy as np
import pytest

import oracle_libs as L
import physx_amd as P

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
