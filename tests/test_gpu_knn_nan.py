"""Rows with a NaN or an infinity on the matrix-core kNN path: a query with a
NaN has no neighbours, a train row with one is nobody's, and the others are the
oracle's as if that row were not there; infinite rows are left to the scan."""
import numpy as np
import pytest

import kodama_amd as K
from kodama_amd import datasets as D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("row", [2, 700, 4299])
@pytest.mark.parametrize("k", [5, 40])
def test_nan_rows(oracle, row, k):
    x, _ = D.config3(n=4600, p=20, seed=k)
    train, query = x[:4300].copy(), x[4300:].copy()
    train[row, 19] = np.nan
    query[[0, 7, 299], 3] = np.nan
    idx, dist = K.exact_knn_search(train, query, k, "euclidean")
    bad = np.isnan(query).any(axis=1)
    assert (idx[bad] == -1).all() and np.isinf(dist[bad]).all()
    rest = np.delete(np.arange(4300), row)
    want_i, want_d = oracle.exact_knn(train[rest], query[~bad], k, K._metric("euclidean"))
    assert np.array_equal(idx[~bad], rest[want_i])
    assert np.array_equal(dist[~bad], want_d)


@pytest.mark.parametrize("where", ["query", "train"])
def test_infinite_rows(oracle, where):
    x, _ = D.config3(n=4600, p=20, seed=1)
    train, query = x[:4300].copy(), x[4300:].copy()
    (query if where == "query" else train)[90, 4] = -np.inf
    idx, dist = K.exact_knn_search(train, query, 5, "euclidean")
    want_i, want_d = oracle.exact_knn(train, query, 5, K._metric("euclidean"))
    assert np.array_equal(idx, want_i) and np.array_equal(dist, want_d)
