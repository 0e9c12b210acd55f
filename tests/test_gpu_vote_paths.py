"""The vote where its labels and results take another way: labels staged from
pinned host memory (all blocks together read at most 128 KiB of them) or copied
first, staged in LDS or not (12288 rows), the last labels of a run (a
multiple of four or not) -- against the oracle's vote, with ties and missing
neighbours; and the reductions of repeated votes (cycles) on each."""
import numpy as np
import pytest

import kodama_amd as K
from kodama_amd import datasets as D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 2, 3, 4, 5, 255, 256, 257, 1022, 1023, 1025, 2816, 2817, 4097, 12288, 12289])
@pytest.mark.parametrize("k", [3, 30])
def test_vote_matches_oracle(oracle, rows, k):
    rng = np.random.default_rng(rows + k)
    nbr = rng.integers(0, rows, (rows, k)).astype(np.int32)
    nbr[rng.random((rows, k)) < 0.1] = -1
    score = -np.sort(rng.integers(0, 4, (rows, k)).astype(np.float32), axis=1)
    folds = np.zeros(rows, np.int32)
    g = K.KnnVoteGraph(nbr, score)
    for _ in range(3):
        labels = rng.integers(0, 6, rows).astype(np.int32)
        got = g.predict(labels, fallback_code=-7)
        want = oracle.knn_vote(nbr, score, folds, labels)
        some = (nbr >= 0).any(axis=1)
        assert np.array_equal(got[some], want[some])
        assert (got[~some] == -7).all()
    g.close()


@pytest.mark.parametrize("rows", [253, 1001, 2816, 2817])
def test_repeated_votes_reduce_alike(oracle, rows):
    """CoreKNN's cycles read the counts, first rows and matches of every vote."""
    import oracle as O
    x, _, _ = D.config1(n=rows, seed=9)
    labels = D.randint(4, 1, rows, 1, 9).astype(np.int32)
    kw = dict(cycles=12, k=10, folds=5, seed=7, cv_seed=8)
    got = K.core_knn(x, labels, K.core_options(**kw))
    want = oracle.core_knn(x, labels, O.core_options(**kw))
    for name in ("clbest", "vect_acc", "active_classes"):
        assert np.array_equal(got[name], want[name]), name
