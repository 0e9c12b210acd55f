"""FP16 matrix-core candidates of the exact kNN (class maxima, threshold,
candidates, exact rerank): neighbours and distances bit-identical to the
oracle's exhaustive search where the operand width, the number of parts, the
sample, the slices and the candidate buffers change."""
import ctypes
import threading

import numpy as np
import pytest

import kodama_amd as K
from kodama_amd import datasets as D

pytestmark = pytest.mark.gpu


def _check(oracle, train, query, k, name, exclude=None, most=0):
    idx, dist = K.exact_knn_search(train, query, k, name, exclude=exclude)
    fb = K.last_knn_fallbacks()
    want = oracle.exact_knn(train, query, k, K._metric(name), exclude=exclude)
    assert np.array_equal(idx, want[0])
    assert np.array_equal(dist, want[1])
    assert 0 <= fb <= most, fb


# Columns at the edges of the operand: one step (three parts up to 9 columns,
# one part up to 30), two (20 / 21: three parts or one; 62 / 63), the widths
# past 64 (from 1024 queries on) up to nine steps, where the second pass with
# three parts ends (95 / 96).
@pytest.mark.parametrize("p", [1, 9, 10, 20, 21, 30, 31, 62, 63, 64, 65, 95, 96, 126, 127, 200, 256])
@pytest.mark.parametrize("name", ["euclidean", "inner_product"])
def test_operand_widths(oracle, p, name):
    queries = 257 if p <= 64 else 1024
    x, _ = D.config3(n=4099 + queries, p=p, seed=p)
    # Very few columns put many rows within the rounding bound of each other.
    _check(oracle, x[:4099], x[4099:], 7, name, most=0 if p > 2 else queries)


# k at the edges of the buffers (32 / 33), of the class maxima (1, 15, 16, 121,
# 128) and of the sample (16 k chunks of 64 rows: 4100 to 20000 rows are a
# sample below k = 20 and all rows above); queries at the edges of a tile, a
# wave and a workgroup.
@pytest.mark.parametrize("k", [1, 2, 15, 16, 32, 33, 121, 128])
@pytest.mark.parametrize("rows,queries", [(4096, 1), (4161, 255), (20000, 17)])
def test_neighbour_counts_and_ragged_sizes(oracle, k, rows, queries):
    x, _ = D.config3(n=rows + queries, p=50, seed=k)
    ex = (np.arange(queries, dtype=np.int32) * 37) % rows
    _check(oracle, x[:rows], x[rows:], k, "euclidean", exclude=ex, most=queries // 20)


def test_rows_sorted_by_distance_refill_the_buffers(oracle):
    """Train rows that come ever closer: the evenly spread sample sets a bound
    that the last rows all pass, so the buffers fill and are tightened."""
    x, _ = D.config3(n=60000, p=24, seed=3)
    query = x[:64] * np.float32(0.01)
    order = np.argsort(-np.linalg.norm(x - query.mean(0), axis=1), kind="stable")
    _check(oracle, np.ascontiguousarray(x[order]), query, 2, "euclidean")


def test_cosine_graph_prepares_rows_as_the_host(oracle):
    x, _ = D.config3(n=4500, p=37, seed=8)
    x[17] = 0.0  # a row without a norm keeps its values
    g = K.KODAMA_knn_graph(x, k=12, metric="cosine")
    idx, dist = oracle.knn_graph(x, 12, 0)
    assert np.array_equal(g["indices"], idx) and np.array_equal(g["distances"], dist)


@pytest.mark.parametrize("scale", [1e-14, 1e17, 1e-17, 1e19])
def test_extreme_scales(oracle, scale):
    """Norms at both ends of the served range, and past it, where every query
    takes the scan."""
    x, _ = D.config3(n=4300, p=16, seed=2)
    x = (x * np.float32(scale)).astype(np.float32)
    _check(oracle, x[:4200], x[4200:], 9, "euclidean", most=100)


def test_outlying_rows_loosen_the_bound_but_not_the_result(oracle):
    """One train row 1000 times the others: the bound follows its norm, so the
    first pass certifies little and the others answer."""
    x, _ = D.config3(n=5000, p=50, seed=12)
    x[40] *= 1000.0
    _check(oracle, x[:4900], x[4900:], 20, "euclidean", most=100)


def _uneven(x, sizes, folds, seed):
    """Runs whose first fold holds nine rows in ten."""
    rng = np.random.default_rng(seed)
    rows, fids = [], []
    for n in sizes:
        rows.append(np.sort(rng.choice(x.shape[0], n, replace=False)).astype(np.int32))
        f = np.where(rng.random(n) < 0.9, 0, rng.integers(0, folds, n)).astype(np.int32)
        f[:folds] = np.arange(folds)
        fids.append(f)
    return rows, fids


# Run sizes at the edges of a chunk (64), the padding (256) and a slice; wide
# rows; a fold that leaves a query few candidates (fewer than k in the small
# runs); every k class.
@pytest.mark.parametrize("p", [2, 21, 65, 200])
@pytest.mark.parametrize("k", [1, 32, 33, 64])
def test_fold_tables_match_oracle(oracle, p, k):
    x, _ = D.config3(n=2500, p=p, seed=p + k)
    rows, fids = _uneven(x, [64, 3, 255, 256, 257, 63, 1025], folds=3, seed=k)
    for name in ("euclidean", "cosine"):
        nbr, score, used = K.knn_fold_tables(x, rows, fids, k, name, path="mfma")
        assert used == "mfma"
        for r, (rw, f) in enumerate(zip(rows, fids)):
            wn, ws = oracle.precompute_knn_cv(x[rw], f, k, K._metric(name))
            assert np.array_equal(nbr[r], wn), (name, r)
            assert np.array_equal(score[r], ws), (name, r)


def test_fold_tables_rule_by_run_size(oracle):
    """The scan below 64 rows in the largest run, the matrix cores from there."""
    x, _ = D.config3(n=400, p=12, seed=1)
    for n, path in ((63, "scan"), (64, "mfma")):
        rows, fids = _uneven(x, [n, 20], folds=4, seed=n)
        nbr, score, used = K.knn_fold_tables(x, rows, fids, 6, "euclidean")
        assert used == path
        for r, (rw, f) in enumerate(zip(rows, fids)):
            wn, ws = oracle.precompute_knn_cv(x[rw], f, 6, 2)
            assert np.array_equal(nbr[r], wn) and np.array_equal(score[r], ws)


def test_fold_tables_of_equal_rows(oracle):
    """Forty copies of each row fill no buffer; 300 copies fill them all, the
    wider second pass too, and the scan answers."""
    base, _ = D.config3(n=6, p=30, seed=4)
    for copies in (40, 300):
        x = np.repeat(base, copies, axis=0)
        rows, fids = [np.arange(x.shape[0], dtype=np.int32)], [(np.arange(x.shape[0]) % 5).astype(np.int32)]
        nbr, score, _ = K.knn_fold_tables(x, rows, fids, 20, "euclidean", path="mfma")
        assert (K.last_knn_fallbacks() == 0) == (copies == 40)
        wn, ws = oracle.precompute_knn_cv(x, fids[0], 20, 2)
        assert np.array_equal(nbr[0], wn) and np.array_equal(score[0], ws)


def test_fold_tables_of_many_runs_in_several_launches(oracle):
    """1.07M padded rows with the larger buffers (2 KiB a row): three launches of
    524288 rows at most, the last of a part, on 1 GiB of candidates. Equal to
    the scan everywhere, and to the oracle in the runs around the seams."""
    x, _ = D.config3(n=6000, p=4, seed=9)
    rng = np.random.default_rng(1)
    rows = [np.sort(rng.choice(6000, 5000, replace=False)).astype(np.int32) for _ in range(210)]
    fids = [rng.integers(0, 7, 5000).astype(np.int32) for _ in rows]
    K.release_memory()
    least = _least_free()
    with least:
        nbr, score, used = K.knn_fold_tables(x, rows, fids, 40, "euclidean", path="mfma")
    assert used == "mfma" and least.used < 2_000_000_000, least.used
    sn, ss, used = K.knn_fold_tables(x, rows, fids, 40, "euclidean", path="scan")
    assert used == "scan"
    for r in range(210):
        assert np.array_equal(nbr[r], sn[r]) and np.array_equal(score[r], ss[r]), r
    for r in (0, 102, 204, 209):
        wn, ws = oracle.precompute_knn_cv(x[rows[r]], fids[r], 40, 2)
        assert np.array_equal(nbr[r], wn) and np.array_equal(score[r], ws), r


class _least_free:
    """The most device memory in use above the start while the block runs, as
    the HIP runtime that the library is linked to reports it."""

    def _free(self):
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert self._hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    def __enter__(self):
        self._hip, self.used, self._stop = ctypes.CDLL("libamdhip64.so.7"), 0, threading.Event()
        start = self._free()

        def watch():
            while not self._stop.is_set():
                self.used = max(self.used, start - self._free())

        self._thread = threading.Thread(target=watch)
        self._thread.start()

    def __exit__(self, *_):
        self._stop.set()
        self._thread.join()


# Rows far from the origin against their spread, on both sides of the width
# where the second pass can take three parts (95 / 96 columns).
@pytest.mark.parametrize("p", [50, 95, 96, 128, 256])
@pytest.mark.parametrize("offset", [10.0, 1000.0])
def test_rows_away_from_the_origin(oracle, p, offset):
    rng = np.random.default_rng(p)
    x = (rng.standard_normal((6100, p), dtype=np.float32) + np.float32(offset)).astype(np.float32)
    x[:, 0] -= np.float32(2 * offset)  # columns of both signs
    ex = (np.arange(1100, dtype=np.int32) * 37) % 5000
    _check(oracle, x[:5000], x[5000:], 30, "euclidean", exclude=ex)
    _check(oracle, x[:5000], x[5000:], 30, "inner_product")
    g = K.KODAMA_knn_graph(x[:5000], k=30)
    assert K.last_knn_fallbacks() == 0
    idx, dist = oracle.knn_graph(x[:5000], 30, 2)
    assert np.array_equal(g["indices"], idx) and np.array_equal(g["distances"], dist)


def test_cosine_rows_around_one_direction(oracle):
    rng = np.random.default_rng(2)
    x = (rng.standard_normal((6000, 110), dtype=np.float32) + np.float32(10)).astype(np.float32)
    g = K.KODAMA_knn_graph(x, k=20, metric="cosine")
    assert K.last_knn_fallbacks() == 0
    idx, dist = oracle.knn_graph(x, 20, 0)
    assert np.array_equal(g["indices"], idx) and np.array_equal(g["distances"], dist)


@pytest.mark.parametrize("name", ["euclidean", "cosine", "inner_product"])
def test_fold_tables_away_from_the_origin(oracle, name):
    rng = np.random.default_rng(4)
    x = (rng.standard_normal((3000, 150), dtype=np.float32) + np.float32(20)).astype(np.float32)
    rows, fids = _uneven(x, [900, 257, 1500], folds=5, seed=8)
    nbr, score, used = K.knn_fold_tables(x, rows, fids, 20, name, path="mfma")
    assert used == "mfma" and K.last_knn_fallbacks() == 0
    for r, (rw, f) in enumerate(zip(rows, fids)):
        wn, ws = oracle.precompute_knn_cv(x[rw], f, 20, K._metric(name))
        assert np.array_equal(nbr[r], wn) and np.array_equal(score[r], ws), r


@pytest.mark.parametrize("name", ["euclidean", "inner_product"])
@pytest.mark.parametrize("what", ["huge_row", "nan_column", "equal_rows", "overflow"])
def test_centres_that_help_nothing(oracle, name, what):
    """A sample whose mean is useless or undefined changes no result: one row
    that outweighs all others, a column without a finite value in the sample
    (its rows are nobody's neighbours), rows that are all the same away from
    the origin, and sums past the largest float."""
    x, _ = D.config3(n=5200, p=40, seed=6)
    train, query = x[:5000].copy(), x[5000:].copy()
    if what == "huge_row":
        train[0] = 1e15
    elif what == "nan_column":
        train[:, 3] = np.nan
    elif what == "equal_rows":
        train[:] = query[0] + np.float32(30)
    else:
        train[:, 5] = 3e38
        query[:, 5] = 3e38
    idx, dist = K.exact_knn_search(train, query, 6, name)
    if what == "nan_column":
        assert (idx == -1).all() and np.isinf(dist).all()
        return
    want = oracle.exact_knn(train, query, 6, K._metric(name))
    assert np.array_equal(idx, want[0]) and np.array_equal(dist, want[1])


def test_inner_product_rows_larger_than_what_is_left_of_them(oracle):
    """Train rows whose offset is 30000 times their spread: the products' own
    rounding hides their order from the scores, and the scan answers."""
    rng = np.random.default_rng(9)
    x = (rng.standard_normal((5200, 100), dtype=np.float32) + np.float32(30000)).astype(np.float32)
    idx, dist = K.exact_knn_search(x[:4100], x[4100:], 12, "inner_product")
    want = oracle.exact_knn(x[:4100], x[4100:], 12, 1)
    assert np.array_equal(idx, want[0]) and np.array_equal(dist, want[1])
