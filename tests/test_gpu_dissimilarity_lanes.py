"""The dissimilarity where its lanes per edge change (128 / 129 runs, whole
waves of runs) and where edges fill a step (8 and 16), bit for bit against the
oracle: missing and unassigned entries, equal edges, infinite distances."""
import numpy as np
import pytest

import kodama_amd as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("runs", [1, 127, 128, 129, 256, 257, 300])
@pytest.mark.parametrize("k", [1, 7, 8, 9, 16, 17, 64, 65, 130])
def test_matches_oracle(oracle, runs, k):
    rng = np.random.default_rng(1000 * runs + k)
    n = 37
    idx = rng.integers(1, n + 1, (n, k)).astype(np.int32)
    dist = np.sort(rng.random((n, k)).astype(np.float32), axis=1)
    idx[3, : k // 2] = -1
    dist[5, k // 2:] = np.inf
    dist[7] = 0.5
    idx[7] = 9  # equal edges keep their order
    idx[8, 0] = n + 40  # outside the samples
    res = rng.integers(0, 4, (runs, n)).astype(np.int32)  # 0 = unassigned
    gi, gd = K.KODAMA_dissimilarity(idx, dist, res)
    wi, wd = oracle.dissimilarity(idx, dist, res)
    assert np.array_equal(gi, wi) and np.array_equal(gd, wd)
