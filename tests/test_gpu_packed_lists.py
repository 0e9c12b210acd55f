"""kNN shapes around the sizes of the candidate buffers and train sets, and the
setting of the candidate lists' form, which is kept for callers and changes
nothing: neighbours bit for bit the oracle's for the global search and the
per-fold tables of a batch of runs (the rerank finds each query's run), both
buffer sizes, negative scores (inner product), train sets past 32768 rows, and
rows equal often enough to fill the buffers."""
import numpy as np
import pytest

import kodama_amd as K
from kodama_amd import datasets as D

from test_gpu_fold_tables import _runs

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _restore():
    yield
    K.set_mfma_packed_lists(True)
    K.set_fold_table_schedule("tuned", 0, 0)


@pytest.mark.parametrize("k,metric,name", [(20, 2, "euclidean"), (20, 1, "inner_product"), (100, 0, "cosine")])
def test_graph_lists_match_oracle(oracle, k, metric, name):
    x, _ = D.config3(n=6000, p=50, seed=k + metric)
    g = K.KODAMA_knn_graph(x, k=k, metric=name)
    assert 0 <= K.last_knn_fallbacks() < 600
    idx, dist = oracle.knn_graph(x, k, metric)
    assert np.array_equal(g["indices"], idx)
    assert np.array_equal(g["distances"], dist)


@pytest.mark.parametrize("list_", [8, 16])
def test_fold_table_lists_match_oracle(oracle, list_):
    x, _ = D.config3(n=6000, p=50, seed=3)
    rows, fids = _runs(x, [2500, 700, 1800, 64], folds=10, seed=list_)
    want = [oracle.precompute_knn_cv(x[rw], f, 30, K._metric("euclidean")) for rw, f in zip(rows, fids)]
    K.set_fold_table_schedule("tuned", list_, 0)
    nbr, score, used = K.knn_fold_tables(x, rows, fids, 30, "euclidean", path="mfma")
    assert used == "mfma" and K.last_fold_table_schedule()["list"] == list_
    for r, (wn, ws) in enumerate(want):
        assert np.array_equal(nbr[r], wn), r
        assert np.array_equal(score[r], ws), r


@pytest.mark.parametrize("train_rows", [32768, 32769])
def test_neighbours_among_the_last_train_rows(oracle, train_rows):
    """A whole number of 64-row chunks and one row more; queries near the last
    train rows."""
    x, _ = D.config3(n=train_rows + 400, p=32, seed=train_rows)
    train = x[:train_rows]
    rng = np.random.default_rng(7)
    query = np.concatenate([train[-300:] + rng.normal(0.0, 1e-3, size=(300, 32)).astype(np.float32),
                            x[train_rows:train_rows + 100]]).astype(np.float32)
    want_idx, want_dist = oracle.exact_knn(train, query, 16, 2)
    idx, dist = K.exact_knn_search(train, query, 16, "euclidean")
    assert 0 <= K.last_knn_fallbacks() < 100
    assert np.array_equal(idx, want_idx)
    assert np.array_equal(dist, want_dist)
    assert np.any(want_idx[:300] >= train_rows - 16)


@pytest.mark.parametrize("k,metric,name", [(20, 1, "inner_product"), (32, 2, "euclidean"), (40, 2, "euclidean")])
def test_lists_with_exclusion(oracle, k, metric, name):
    """40000 train rows cut into slices whose candidates the rerank merges, both
    buffer sizes, negative scores; every query excludes one train row."""
    x, _ = D.config3(n=40600, p=50, seed=k)
    train, query = x[:40000], x[40000:]
    ex = (np.arange(600, dtype=np.int32) * 61) % 40000
    want_idx, want_dist = oracle.exact_knn(train, query, k, metric, exclude=ex)
    idx, dist = K.exact_knn_search(train, query, k, name, exclude=ex)
    assert 0 <= K.last_knn_fallbacks() < 300
    assert np.array_equal(idx, want_idx)
    assert np.array_equal(dist, want_dist)
    assert not np.any(idx == ex[:, None])


def test_duplicates_fall_back(oracle):
    """1000 copies of each row: every query has more rows inside its bound than
    either buffer holds and takes the exact scan."""
    base, _, _ = D.config1(n=5, seed=11)
    x = np.repeat(base, 1000, axis=0)
    g = K.KODAMA_knn_graph(x, k=24)
    assert K.last_knn_fallbacks() == x.shape[0]
    idx, dist = oracle.knn_graph(x, 24, 2)
    assert np.array_equal(g["indices"], idx)
    assert np.array_equal(g["distances"], dist)


def test_second_pass_certifies_what_the_first_buffers_cannot(oracle):
    """150 copies of each of 40 rows do not fit the first pass's 128 entries per
    slice; the second pass's 256 hold them (ties at distance 0 ranked by index)
    and nothing reaches the scan."""
    base, _ = D.config3(n=40, p=24, seed=5)
    x = np.repeat(base, 150, axis=0)
    g = K.KODAMA_knn_graph(x, k=20)
    assert K.last_knn_fallbacks() == 0
    idx, dist = oracle.knn_graph(x, 20, 2)
    assert np.array_equal(g["indices"], idx)
    assert np.array_equal(g["distances"], dist)


def test_the_form_setting_is_accepted_and_changes_nothing():
    x, _ = D.config3(n=5000, p=20, seed=1)
    out = []
    for on in (True, False):
        K.set_mfma_packed_lists(on)
        out.append(K.KODAMA_knn_graph(x, k=10))
    assert np.array_equal(out[0]["indices"], out[1]["indices"])
    assert np.array_equal(out[0]["distances"], out[1]["distances"])


def test_packed_list_control_rejects_out_of_range():
    with pytest.raises(ValueError):
        K.N.call("kodama_hip_set_mfma_packed_lists", K.C.c_int32(2))
