"""Host side of the calls: memory and streams kept between calls (several
threads, sizes that shrink and grow), and label encoding by table or by sort."""
import ctypes
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import kodama_amd as K
from kodama_amd import datasets as D

pytestmark = pytest.mark.gpu


def _work(seed):
    """Calls of every kind that allocates, with sizes that differ by seed."""
    n = 4200 + 700 * (seed % 4)
    x, comp = D.config3(n=n, p=20 + seed % 3, seed=seed % 4)
    g = K.KODAMA_knn_graph(x, k=10 + seed % 5)
    rows = [np.arange(seed % 7, 900 + 50 * (seed % 4), dtype=np.int32), np.arange(1000, 1600, dtype=np.int32)]
    init = [comp[r] for r in rows]
    o = K.core_options(cycles=4, k=8, folds=5, stratified=0, evolutionary_search=1, guarded_diversity=1,
                       many_to_one_absorption=1)
    b = K.core_knn_batch(x, rows, init, o, mode=("plain", "device")[seed % 2])
    p = K.PLSLDACV(x[:800], comp[:800], ncomp=3, folds=4)
    return [g["indices"], g["distances"], *b["clbest"], b["vect_acc"], p["predicted_labels"]]


def test_threads_share_the_kept_memory():
    """Eight threads, three calls each, against the same calls in sequence."""
    seeds = list(range(8))
    want = [_work(s) for s in seeds]
    with ThreadPoolExecutor(8) as pool:
        got = list(pool.map(_work, seeds * 3))
    for i, out in enumerate(got):
        for a, b in zip(out, want[i % 8]):
            assert np.array_equal(a, b), i % 8


def test_a_resident_graph_survives_other_calls():
    """A vote graph keeps its memory while other calls take and give theirs."""
    rng = np.random.default_rng(3)
    nbr = rng.integers(0, 3000, (3000, 12), dtype=np.int32)
    score = -np.sort(rng.random((3000, 12), dtype=np.float32), axis=1)
    codes = rng.integers(0, 9, 3000, dtype=np.int32)
    graph = K.KnnVoteGraph(nbr, score)
    first = graph.predict(codes)
    for s in range(4):
        _work(s)
        assert np.array_equal(graph.predict(codes), first)
    graph.close()
    _work(1)


@pytest.mark.parametrize("spread", [1, 7, 1_000_003])
def test_label_values_do_not_matter(spread):
    """Labels close together are encoded by a table, far apart by a sort; the
    votes depend on their order only."""
    x, comp = D.config3(n=600, p=10, seed=6)
    base = K.KNNCV(x, comp, k=7, metric="euclidean", folds=5)
    lab = (comp - 9) * spread
    out = K.KNNCV(x, lab, k=7, metric="euclidean", folds=5)
    assert np.array_equal(out["predicted_labels"], (base["predicted_labels"] - 9) * spread)
    assert np.array_equal(out["fold_assignments"], base["fold_assignments"])


def _free_bytes():
    """Free device memory, from the HIP runtime that the library is linked to."""
    K.version()
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL("libamdhip64.so.7").hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_released_memory_is_free_for_others():
    """What a call leaves in the pool comes back with release_memory; a resident
    handle keeps its own, and later calls allocate again."""
    rng = np.random.default_rng(5)
    nbr = rng.integers(0, 3000, (3000, 12), dtype=np.int32)
    score = -np.sort(rng.random((3000, 12), dtype=np.float32), axis=1)
    codes = rng.integers(0, 9, 3000, dtype=np.int32)
    x, _ = D.config3(n=60000, p=50, seed=3)
    graph = K.KnnVoteGraph(nbr, score)
    votes = graph.predict(codes)
    K.release_memory()
    before = _free_bytes()
    want = K.KODAMA_knn_graph(x, k=20)
    kept = before - _free_bytes()
    K.release_memory()
    assert kept > 30 << 20
    assert before - _free_bytes() <= kept // 8
    assert np.array_equal(graph.predict(codes), votes)
    graph.close()
    again = K.KODAMA_knn_graph(x, k=20)
    assert np.array_equal(again["indices"], want["indices"])
    with pytest.raises(K.NoDevice):
        K.release_memory(gpu_device=99)


def test_an_error_in_a_parallel_loop_is_an_error_of_the_call():
    """20 runs, enough rows for the parallel preparation, and a fold count that
    the fold dealer refuses inside it."""
    x, comp = D.config3(n=3000, p=8, seed=2)
    rows = [np.arange(r, 1000 + r, dtype=np.int32) for r in range(20)]
    o = K.core_options(cycles=1, k=5, folds=1, stratified=0, evolutionary_search=1, guarded_diversity=1)
    with pytest.raises(ValueError, match="Number of folds must be at least 2"):
        K.core_knn_batch(x, rows, [comp[r] for r in rows], o)
