"""The workloads whose speed is measured: calls that a user of kodama_amd makes,
through its public entry points, from the smallest vote to a 1M-row graph.

A case is a dict of plain values. prepare() makes what a program has in hand
before the call (host arrays, since the entry points take host arrays, and the
vote-graph handle that such a program keeps), run() is one call, work() what the
call cannot do without. Sizes are those of the repository's benchmark and tests
(n = 2000 to 1M rows, p = 50, k = 10 to 100, 100 runs of 1000-5000 landmarks) and
ragged ones between them.

Every result here is fixed by the inputs: the neighbours and distances are
defined bit for bit (one float32 summation order, ties by index), the votes are
counts with a fixed tie order, the plain evolutions replay named random streams,
and the device evolutions draw from counters. So the tolerance is "exact".
"""
from __future__ import annotations

import math

import numpy as np
import torch

import kodama_amd as K


# ---- inputs ---------------------------------------------------------------------

def _gen(seed, stream=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000003 + stream)
    return g


def _mixture(n, p, seed, centers=20):
    """Rows of a Gaussian mixture (Zipf(1.1) cluster sizes, unit variance, means
    U[-4, 4]^p) and their components, the shape of the benchmark's data."""
    g = _gen(seed, 1)
    means = (torch.rand(centers, p, generator=g, device="cuda") * 2.0 - 1.0) * 4.0
    w = 1.0 / torch.arange(1, centers + 1, device="cuda", dtype=torch.float32) ** 1.1
    comp = torch.multinomial(w, n, replacement=True, generator=g)
    x = means[comp] + torch.randn(n, p, generator=g, device="cuda")
    return x.cpu().numpy(), comp.to(torch.int32).cpu().numpy() + 1


def _latent(n, p, seed):
    """Latent Gaussian of variance 1 / i in dimension i, eight clusters shifted
    along three directions: the PLS-LDA data."""
    g = _gen(seed, 2)
    sd = 1.0 / torch.sqrt(torch.arange(1, p + 1, device="cuda", dtype=torch.float32))
    comp = torch.randint(0, 8, (n,), generator=g, device="cuda")
    dirs = torch.randn(3, p, generator=g, device="cuda")
    dirs = dirs / dirs.norm(dim=1, keepdim=True)
    signs = torch.rand(8, 3, generator=g, device="cuda") * 2.0 - 1.0
    x = torch.randn(n, p, generator=g, device="cuda") * sd + (2.0 * (signs @ dirs) * sd)[comp]
    return x.cpu().numpy(), comp.to(torch.int32).cpu().numpy() + 1


def _runs(x, comp, case, seed):
    """Landmark rows, uneven folds and starting labels of a batch of runs (the
    run sizes belong to the case, not to the seed). The starting labels split each component into pieces by random landmark centres
    (nearest centre, as one k-means step leaves them), or are the components
    with 5 % label noise."""
    rng = np.random.default_rng(seed + 17)
    sizes = np.random.default_rng(case["lo"] + case["runs"]).integers(case["lo"], case["hi"] + 1, case["runs"])
    xg = torch.from_numpy(x).cuda()
    n = x.shape[0]
    rows, folds, init = [], [], []
    for r in range(case["runs"]):
        size = int(sizes[r])
        rw = np.sort(rng.choice(n, size, replace=False)).astype(np.int32)
        share = rng.dirichlet(np.ones(case["folds"]))
        cnt = np.maximum(1, np.floor(share * (size - case["folds"])).astype(np.int64) + 1)
        cnt[np.argmax(cnt)] += size - cnt.sum()
        f = rng.permutation(np.repeat(np.arange(case["folds"], dtype=np.int32), cnt)).astype(np.int32)
        if case["start"] == "noisy":
            lab = comp[rw].copy()
            flip = rng.random(size) < 0.05
            lab[flip] = rng.integers(1, int(comp.max()) + 1, int(flip.sum()))
        else:
            idx = torch.from_numpy(rw.astype(np.int64)).cuda()
            pts = xg[idx]
            pick = torch.from_numpy(rng.choice(size, min(case["centres"], size), replace=False)).cuda()
            lab = torch.cdist(pts, pts[pick]).argmin(dim=1).to(torch.int32).cpu().numpy() + 1
        rows.append(rw)
        folds.append(f)
        init.append(lab.astype(np.int32))
    return rows, folds, init


def _network(case, seed):
    """A proposal network trained on accept/reject traces of a few other runs."""
    sub = dict(case, runs=4, start="centres", centres=100)
    x, comp = _mixture(20000, case["p"], seed + 5)
    rows, folds, init = _runs(x, comp, sub, seed + 5)
    feat, tgt, _ = K.mlp_collect_traces(x, rows, init, _options(case, cycles=20), fold_ids=folds, max_samples=20000)
    params, _ = K.mlp_train(feat, tgt, epochs=3, batch=256, learning_rate=0.05, momentum=0.9, seed=seed + 1)
    return params


def _options(case, cycles=None):
    kw = dict(cycles=case["cycles"] if cycles is None else cycles, folds=case["folds"], stratified=0, seed=1,
              cv_seed=1, evolutionary_search=1, guarded_diversity=1, n_threads=0)
    if case["kind"] == "batch_pls":
        kw.update(classifier=0, max_components=case["ncomp"], fixed_components=case["ncomp"],
                  auto_class_coarsening=1)
    else:
        kw.update(k=case["k"], many_to_one_absorption=1)
    return K.core_options(**kw)


# ---- the cases ------------------------------------------------------------------

_BATCH = dict(n=100000, p=50, k=30, runs=100, lo=1000, hi=5000, folds=10, cycles=20, start="centres", centres=300)


def listed():
    return [
        # One vote of a resident graph, the call inside a caller's own label
        # search: a launch and two small copies, latency above all.
        dict(name="vote_2k", kind="vote", n=2000, k=10, classes=5),
        # The cross-validated classifier on a small table with its defaults
        # (cosine, stratified): the first call of most users.
        dict(name="knncv_2k", kind="knncv", n=2000, p=50, k=10, metric="cosine", folds=10),
        # One label evolution of a small table with the reference's random
        # streams: 100 cycles of host proposals and tiny votes.
        dict(name="core_2k", kind="core", n=2000, p=50, k=10, folds=10, cycles=100),
        # New rows against a reference set, more columns than the mixture's
        # (spectra, gene panels), odd sizes.
        dict(name="search_wide", kind="search", train=30011, query=10007, p=100, k=30, metric="euclidean"),
        # The 100-neighbour graph that the matrix construction uses by default.
        dict(name="graph_100k", kind="graph", n=100000, p=50, k=100, metric="euclidean"),
        # The largest graph of the repository's benchmark.
        dict(name="graph_1m", kind="graph", n=1000000, p=50, k=30, metric="euclidean"),
        # The headline batch: 100 runs of 1000-5000 landmarks, k = 30, in the
        # form with the reference's streams, ...
        dict(name="batch_plain", kind="batch_plain", **_BATCH),
        # ... resident on the device, ...
        dict(name="batch_device", kind="batch_device", **_BATCH),
        # ... and with the learned proposal on labels that are mostly right,
        # 100 cycles.
        dict(name="batch_learned", kind="batch_learned",
             **dict(_BATCH, n=200000, cycles=100, start="noisy")),
        # The PLS-LDA batch of the benchmark: 100 runs of 2000 landmarks.
        dict(name="batch_pls", kind="batch_pls", n=10000, p=50, ncomp=5, runs=100, lo=2000, hi=2000, folds=10,
             cycles=20, start="centres", centres=8),
        # The whole construction on 100k rows: atlas, graph, landmarks, Core,
        # projection.
        dict(name="matrix_100k", kind="matrix", n=100000, p=50, k=30, runs=100, cycles=50, landmarks=3000,
             splitting=300, folds=5, neighbors=100, form="device"),
        # The graph rewritten by the runs' labels, what the construction ends with.
        dict(name="dissimilarity_100k", kind="dissimilarity", n=100000, k=100, runs=100),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: a kind of the list, its sizes spread over what it takes."""
    kind = rng.choice(["vote", "knncv", "core", "search", "search", "graph", "graph", "graph", "batch_plain",
                       "batch_device", "batch_device", "batch_learned", "batch_pls", "matrix", "dissimilarity"])
    metric = rng.choice(["euclidean", "euclidean", "cosine", "inner_product"])
    if kind == "vote":
        return dict(kind=kind, n=_log(rng, 500, 100000), k=_log(rng, 5, 64), classes=_log(rng, 2, 300))
    if kind == "knncv":
        return dict(kind=kind, n=_log(rng, 500, 40000), p=_log(rng, 4, 200), k=_log(rng, 3, 60), metric=metric,
                    folds=rng.choice([3, 5, 10]))
    if kind == "core":
        return dict(kind=kind, n=_log(rng, 500, 8000), p=_log(rng, 4, 64), k=_log(rng, 5, 50),
                    folds=rng.choice([5, 10]), cycles=_log(rng, 10, 100))
    if kind == "search":
        p = _log(rng, 4, 256)
        return dict(kind=kind, train=_log(rng, 1000, 100000), query=_log(rng, 100, 50000), p=p,
                    k=_log(rng, 1, 128 if p <= 128 else 64), metric=metric)
    if kind == "graph":
        n = _log(rng, 1000, 500000)
        p = _log(rng, 4, 64 if n > 60000 else 256)
        top = 128 if p <= 128 else 64
        return dict(kind=kind, n=n, p=p, k=_log(rng, 5, 30 if n > 200000 else top), metric=metric)
    if kind.startswith("batch"):
        lo = _log(rng, 200, 2000)
        case = dict(kind=kind, n=_log(rng, 6000, 200000), p=_log(rng, 8, 64), runs=_log(rng, 4, 100), lo=lo,
                    hi=lo + _log(rng, 1, 3000), folds=rng.choice([5, 10]), cycles=_log(rng, 5, 100))
        if kind == "batch_pls":
            return dict(case, n=10000 + rng.randrange(5000), ncomp=rng.randrange(2, 7),
                        cycles=_log(rng, 5, 20), start="centres", centres=8)
        return dict(case, k=_log(rng, 5, 60), start=rng.choice(["centres", "noisy"]), centres=_log(rng, 20, 300))
    if kind == "matrix":
        n = _log(rng, 1500, 100000)
        return dict(kind=kind, n=n, p=_log(rng, 8, 64), k=_log(rng, 5, 50), runs=_log(rng, 4, 100),
                    cycles=_log(rng, 10, 50), landmarks=min(_log(rng, 500, 4000), int(0.7 * n)),
                    splitting=_log(rng, 30, 300), folds=5, neighbors=_log(rng, 50, 110),
                    form=rng.choice(["device", "plain"]))
    return dict(kind=kind, n=_log(rng, 1000, 100000), k=_log(rng, 10, 110), runs=_log(rng, 4, 130))


# ---- one pass -------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "vote":
        n, k = case["n"], case["k"]
        nbr = rng.integers(0, n, (n, k), dtype=np.int32)
        score = -np.sort(rng.random((n, k), dtype=np.float32) * 50.0, axis=1)
        codes = rng.integers(0, case["classes"], n, dtype=np.int32)
        return dict(kind=kind, graph=K.KnnVoteGraph(nbr, score), codes=codes)
    if kind == "dissimilarity":
        # A graph of near neighbours with the labels that runs of the evolution
        # give: mostly the component, split and merged differently in each run.
        n, k, runs = case["n"], case["k"], case["runs"]
        g = _gen(seed, 3)
        comp = torch.sort(torch.randint(0, 20, (n,), generator=g, device="cuda"))[0]
        step = torch.randint(1, 400, (n, k), generator=g, device="cuda")
        sign = torch.randint(0, 2, (n, k), generator=g, device="cuda") * 2 - 1
        ids = (torch.arange(n, device="cuda")[:, None] + step * sign) % n + 1
        dist = torch.sort(torch.rand(n, k, generator=g, device="cuda") * 4.0 + 6.0, dim=1)[0]
        split = torch.randint(1, 40, (runs, 20), generator=g, device="cuda", dtype=torch.int32)
        noise = torch.rand(runs, n, generator=g, device="cuda") < 0.03
        res = torch.where(noise, torch.randint(1, 40, (runs, n), generator=g, device="cuda", dtype=torch.int32),
                          split[:, comp])
        return dict(kind=kind, indices=ids.to(torch.int32).cpu().numpy(), distances=dist.cpu().numpy(),
                    res=res.cpu().numpy())
    if kind == "search":
        x, _ = _mixture(case["train"] + case["query"], case["p"], seed)
        if case["metric"] == "cosine":  # the call takes normalised rows
            x = x / np.maximum(np.linalg.norm(x, axis=1, keepdims=True), 1e-12).astype(np.float32)
        return dict(case, x=np.ascontiguousarray(x[:case["train"]]), q=np.ascontiguousarray(x[case["train"]:]))
    if kind == "graph":
        return dict(case, x=_mixture(case["n"], case["p"], seed)[0])
    if kind in ("knncv", "core"):
        x, comp = _mixture(case["n"], case["p"], seed, centers=5)
        labels = comp if kind == "knncv" else rng.integers(1, 6, case["n"]).astype(np.int32)
        return dict(case, x=x, labels=labels)
    if kind == "matrix":
        return dict(case, x=_mixture(case["n"], case["p"], seed)[0])
    x, comp = (_latent if kind == "batch_pls" else _mixture)(case["n"], case["p"], seed)
    rows, fold_ids, init = _runs(x, comp, case, seed)
    state = dict(case, x=x, rows=rows, fold_ids=fold_ids, init=init, options=_options(case))
    if kind == "batch_learned":
        state["params"] = _network(case, seed)
    return state


def _batch_out(out):
    return dict(clbest=np.concatenate(out["clbest"]), accbest=out["accbest"], vect_acc=out["vect_acc"])


def run(state):
    s, kind = state, state["kind"]
    if kind == "vote":
        return s["graph"].predict(s["codes"])
    if kind == "knncv":
        out = K.KNNCV(s["x"], s["labels"], folds=s["folds"], k=s["k"], metric=s["metric"])
        return dict(predicted=out["predicted_labels"], folds=out["fold_assignments"],
                    accuracy=out["global_accuracy"])
    if kind == "core":
        out = K.CoreKNN(s["x"], s["labels"], cycles=s["cycles"], folds=s["folds"], k=s["k"])
        return {f: v for f, v in out.items() if f != "backend"}
    if kind == "search":
        idx, dist = K.exact_knn_search(s["x"], s["q"], s["k"], metric=s["metric"])
        return dict(indices=idx, distances=dist)
    if kind == "graph":
        out = K.KODAMA_knn_graph(s["x"], k=s["k"], metric=s["metric"])
        return dict(indices=out["indices"], distances=out["distances"])
    if kind in ("batch_plain", "batch_device"):
        return _batch_out(K.core_knn_batch(s["x"], s["rows"], s["init"], s["options"], mode=kind[6:],
                                           fold_ids=s["fold_ids"]))
    if kind == "batch_learned":
        return _batch_out(K.core_knn_batch_learned(s["x"], s["rows"], s["init"], s["options"], s["params"],
                                                   fallback=0.25, fold_ids=s["fold_ids"]))
    if kind == "batch_pls":
        return _batch_out(K.core_plslda_batch(s["x"], s["rows"], s["init"], s["options"], fold_ids=s["fold_ids"]))
    if kind == "matrix":
        out = K.KODAMA_matrix(s["x"], M=s["runs"], Tcycle=s["cycles"], landmarks=s["landmarks"],
                              splitting=s["splitting"], folds=s["folds"], k=s["k"], graph_neighbors=s["neighbors"],
                              form=s["form"])
        return {f: out[f] for f in ("res", "acc", "v", "landmarks", "knn_indices", "knn_distances")}
    idx, dist = K.KODAMA_dissimilarity(s["indices"], s["distances"], s["res"])
    return dict(indices=idx, distances=dist)


# ---- what a pass needs ------------------------------------------------------------

def _pairs(sizes_lo, sizes_hi, runs):
    """Mean sum of squared run sizes, sizes uniform between the two."""
    a, b = float(sizes_lo), float(sizes_hi)
    return runs * (a * a + a * b + b * b) / 3.0


def work(case):
    """Inputs read once, outputs written once; two operations per column of each
    pair of rows that a search compares."""
    kind = case["kind"]
    if kind == "vote":
        n, k = case["n"], case["k"]
        return dict(bytes=8 * n * k + 8 * n, flops=2 * n * k)
    if kind == "dissimilarity":
        n, k, runs = case["n"], case["k"], case["runs"]
        return dict(bytes=16 * n * k + 4 * n * runs, flops=2 * n * k * runs)
    if kind == "search":
        t, q, p, k = case["train"], case["query"], case["p"], case["k"]
        return dict(bytes=4 * (t + q) * p + 8 * q * k, flops=2 * t * q * p)
    n, p = case["n"], case["p"]
    if kind == "graph":
        return dict(bytes=4 * n * p + 8 * n * case["k"], flops=2 * n * n * p)
    if kind == "knncv":
        return dict(bytes=4 * n * p + 16 * n, flops=2 * n * n * p)
    if kind == "core":
        k, c = case["k"], case["cycles"]
        return dict(bytes=4 * n * p + 8 * n * k * (c + 1), flops=2 * n * n * p + 2 * n * k * (c + 1))
    if kind == "matrix":
        k, c, runs, L = case["k"], case["cycles"], case["runs"], case["landmarks"]
        return dict(bytes=4 * n * p + 8 * n * case["neighbors"] + 4 * n * runs + 8 * runs * L * k * (c + 1),
                    flops=2 * n * n * p + 2 * runs * L * L * p + 2 * runs * L * k * (c + 1))
    rows = case["runs"] * (case["lo"] + case["hi"]) / 2.0
    c = case["cycles"]
    if kind == "batch_pls":
        # Per cycle and fold: the class sums of the training rows (one add per
        # value) and ncomp products of the validation rows.
        return dict(bytes=int(4 * n * p + 12 * rows + 8 * rows * (c + 1)),
                    flops=int(rows * (c + 1) * p * (case["folds"] - 1 + 2 * case["ncomp"])))
    return dict(bytes=int(4 * n * p + 12 * rows + 8 * rows * case["k"] * (c + 1)),
                flops=int(2 * _pairs(case["lo"], case["hi"], case["runs"]) * p + 2 * rows * case["k"] * (c + 1)))


def tolerance(case):
    return "exact"


# ---- 64-bit values ----------------------------------------------------------------

def _sorted_distances(q, x, k, metric, skip_self):
    """The k smallest internal distances of each query row, float64."""
    xt = x.T.contiguous()
    xn = (x * x).sum(1)
    rows = max(1, int(4e8) // x.shape[0])
    out = []
    for a in range(0, q.shape[0], rows):
        b = q[a:a + rows]
        d = b @ xt
        d = (b * b).sum(1)[:, None] + xn - 2.0 * d if metric == "euclidean" else -d
        if skip_self:
            i = torch.arange(b.shape[0], device=d.device)
            d[i, a + i] = math.inf
        out.append(torch.topk(d, k, dim=1, largest=False)[0])
    return torch.cat(out)


def exact(case, seed):
    """Distances in 64 bits; indices, votes and labels have no such value, and the
    evolutions' accuracies are counts along random trajectories."""
    kind = case["kind"]
    if kind == "search":
        if case["train"] * case["query"] > 3e10:
            return None
        s = prepare(case, seed)
        x, q = (torch.from_numpy(s[f]).cuda().double() for f in ("x", "q"))
        k = min(case["k"], case["train"])
        return dict(indices=None, distances=_sorted_distances(q, x, k, case["metric"], False).cpu().numpy())
    if kind == "graph":
        n = case["n"]
        if n * n > 3e10:
            return None
        x = torch.from_numpy(prepare(case, seed)["x"]).cuda().double()
        if case["metric"] == "cosine":
            x = x / x.norm(dim=1, keepdim=True)
        d = _sorted_distances(x, x, min(case["k"], n - 1), case["metric"], True)
        d = torch.sqrt(d.clamp_min(0.0)) if case["metric"] == "euclidean" else 1.0 + d
        if case["metric"] == "cosine":
            d = d.clamp_min(0.0)
        return dict(indices=None, distances=d.cpu().numpy())
    if kind == "dissimilarity":
        s = prepare(case, seed)
        idx = torch.from_numpy(s["indices"]).cuda().long() - 1
        dist = torch.from_numpy(s["distances"]).cuda().double()
        lab = torch.from_numpy(s["res"]).cuda().T.contiguous()  # every label is a class (none 0)
        same = torch.empty_like(dist)
        for j in range(idx.shape[1]):
            same[:, j] = (lab == lab[idx[:, j]]).sum(1).double()
        if bool((same == 0).any()):
            return None  # infinite distances
        d = torch.sort((1.0 + dist) / (same / case["runs"]) ** 2, dim=1)[0]
        return dict(indices=None, distances=d.cpu().numpy())
    return None
