"""KODAMA.matrix kernels where their layouts change, bit for bit against the
oracle's KODAMA.matrix (atlas, landmarks, starting labels, projection): the
k-means assignment by matrix-core scores with exact re-evaluation, the sorted
cluster sums, and the projection with a lane per run."""
import numpy as np
import pytest

import kodama_amd as K
from kodama_amd import datasets as D

pytestmark = pytest.mark.gpu


def _check(oracle, x, **kw):
    o = dict(runs=2, cycles=2, landmarks=300, splitting=40, folds=3, k=8, graph_neighbors=30, seed=11)
    o.update(kw)
    got = K.KODAMA_matrix(x, M=o["runs"], Tcycle=o["cycles"], landmarks=o["landmarks"], splitting=o["splitting"],
                          folds=o["folds"], k=o["k"], graph_neighbors=o["graph_neighbors"], seed=o["seed"])
    want = oracle.kodama_matrix(x, **o)
    for f in ("res", "acc", "v"):
        assert np.array_equal(got[f], want[f]), f


# Columns at the edges of the operand steps and of the reference's blocks of 16.
@pytest.mark.parametrize("p", [1, 15, 16, 20, 21, 62, 63, 129, 256])
def test_columns(oracle, p):
    x, _ = D.gaussian_mixture(700, p, 6, seed=p)
    _check(oracle, x)


# Clusters at the edges of an LDS chunk (64) and past a workgroup's threads (256);
# rows at the edges of a segment (1024) of the counting sort.
@pytest.mark.parametrize("n,splitting", [(1023, 63), (1024, 64), (1025, 65), (2049, 257)])
def test_clusters_and_segments(oracle, n, splitting):
    x, _ = D.gaussian_mixture(n, 12, 5, seed=n)
    _check(oracle, x, splitting=splitting)


def test_equal_rows_and_ties(oracle):
    """Rows on a small integer grid: equal rows and equal distances (the first
    cluster wins), empty clusters to split, candidates that fill the queue."""
    rng = np.random.default_rng(4)
    x = rng.integers(0, 3, (900, 5)).astype(np.float32)
    _check(oracle, x, splitting=100)


def test_rows_without_spread(oracle):
    """All rows equal but one: every centroid ties for nearly every row."""
    x = np.ones((400, 7), np.float32)
    x[17] = 2.0
    _check(oracle, x, landmarks=150, splitting=70)


@pytest.mark.parametrize("value", [7.0, 1e-3])
def test_many_splits_of_one_donor(oracle, value):
    """Nearly all rows equal and far more clusters than distinct rows: each
    round splits the same donors over and over, which scales centroids by
    (1 + 1 / 1024) each time, past every row's norm; the bound of the scores
    follows them. One column, so that every product is rounded alone."""
    rng = np.random.default_rng(3)
    x = np.full((3000, 1), value, np.float32)
    x[::100] += rng.normal(0.0, value / 100, (30, 1)).astype(np.float32)
    _check(oracle, x, landmarks=1500, splitting=200)


@pytest.mark.parametrize("scale", [1e-18, 1e18])
def test_scales_outside_the_scores(oracle, scale):
    """Norms the FP16 scores do not serve: every pair is evaluated exactly."""
    x, _ = D.gaussian_mixture(500, 9, 4, seed=2)
    _check(oracle, (x * np.float32(scale)).astype(np.float32), landmarks=200, splitting=30)


# 1 to 32 lanes a row, then one lane per run in groups of 64; votes at both ends;
# an odd number of rows (16-bit entries in whole words).
@pytest.mark.parametrize("runs,k", [(1, 1), (1, 64), (2, 30), (3, 7), (5, 64), (16, 9), (17, 30), (32, 64), (33, 12),
                                    (63, 64), (64, 30), (65, 5), (130, 20)])
def test_projection_runs_and_votes(oracle, runs, k):
    x, _ = D.gaussian_mixture(501, 6, 4, seed=runs)
    _check(oracle, x, runs=runs, cycles=1, landmarks=150, splitting=10, k=k, graph_neighbors=100)
