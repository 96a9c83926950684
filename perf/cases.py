"""Timed cases: the counting calls a program makes through this package.

Each case is a dict of plain values: a seeded graph family with its sizes and
one query on it.  prepare() builds the graph (and what a program keeps beside
it: a trained cost model, a batch, a step-API state), run() is one counting
call, work() the bytes of the graph and of the results and one operation per
adjacency entry, exact() an independent count where plain numpy is quick.
All results are whole numbers: clique counts or motif histograms.
"""
import math

import numpy as np

import dumato_amd as dm


def listed():
    return [
        # the smallest call: triangles of a 2,000-vertex random graph, where
        # launches, copies and the persistent kernel's start and end count
        dict(name="er2k-clique3", family="er", n=2000, m=20000, query="clique", k=3),
        # a citation-network-sized sparse graph, five-vertex patterns
        dict(name="sparse3k-motif5", family="chunglu", n=3301, m=4603, gamma=2.6, wmax=90.0, query="motif", k=5),
        # flat degrees, odd sizes: no hubs for the schedulers to split
        dict(name="er5k-motif4", family="er", n=5003, m=60011, query="motif", k=4),
        # the benchmark's headline query: power-law graph, four-vertex patterns
        dict(name="chunglu18k-motif4", family="chunglu", n=18000, m=200000, gamma=2.3, wmax=500.0,
             query="motif", k=4),
        # preferential attachment with planted cliques: many vertices, strong hubs
        dict(name="ba100k-motif4", family="ba", n=100000, m=10, planted=200, query="motif", k=4),
        # deep motifs beside hubs: the longest enumeration
        dict(name="ba12k-motif5", family="ba", n=12007, m=10, planted=40, query="motif", k=5),
        # a large sparse graph, triangles: reading the graph matters most
        dict(name="rmat18-clique3", family="rmat", scale=18, ef=16, query="clique", k=3),
        # skewed graph, mid-size cliques, plain scheduling
        dict(name="rmat17-clique5", family="rmat", scale=17, ef=8, query="clique", k=5),
        # the same family with the learned scheduler (cost model trained once)
        dict(name="rmat17-clique6-learned", family="rmat", scale=17, ef=8, query="clique", k=6, learned=True),
        # cliques beyond the bitmap sizes
        dict(name="rmat13-clique7", family="rmat", scale=13, ef=8, query="clique", k=7),
        # a service's mixed batch: several graphs and patterns in one launch
        dict(name="batch12", family="batch", graphs=12, nmin=500, nmax=10000, query="batch", k=5),
        # the step API (user kernels, host-driven balancing): near-cliques
        dict(name="dfs-near5", family="rmat", scale=12, ef=8, query="near_clique", k=5),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.randrange(9)
    if kind == 0:
        n = _log_int(rng, 500, 50000)
        return dict(family="er", n=n, m=int(n * rng.uniform(2, 20)), query="clique", k=rng.randint(3, 6))
    if kind == 1:
        n, avg = _log_int(rng, 1000, 30000), rng.uniform(4, 24)
        return dict(family="chunglu", n=n, m=int(n * avg / 2), gamma=round(rng.uniform(2.1, 2.8), 3),
                    wmax=round(min(n / 8.0, rng.uniform(4, 20) * avg), 1), query="motif", k=rng.randint(3, 4))
    if kind == 2:
        n = _log_int(rng, 1000, 20000)
        return dict(family="er", n=n, m=int(n * rng.uniform(2, 12)), query="motif", k=rng.randint(3, 4))
    if kind == 3:
        n = _log_int(rng, 500, 4000)
        return dict(family="chunglu", n=n, m=int(n * rng.uniform(1.0, 1.5)), gamma=round(rng.uniform(2.4, 2.8), 3),
                    wmax=round(rng.uniform(15, 60), 1), query="motif", k=rng.randint(5, 6))
    if kind == 4:
        return dict(family="ba", n=_log_int(rng, 2000, 100000), m=rng.randint(3, 10), planted=rng.randint(0, 200),
                    query="motif", k=4)
    if kind == 5:
        return dict(family="ba", n=_log_int(rng, 1000, 10000), m=rng.randint(3, 9), planted=rng.randint(0, 40),
                    query="motif", k=5)
    if kind == 6:
        return dict(family="rmat", scale=rng.randint(12, 17), ef=rng.randint(4, 8), query="clique",
                    k=rng.randint(3, 6), learned=rng.random() < 0.4)
    if kind == 7:
        return dict(family="rmat", scale=rng.randint(9, 12), ef=rng.randint(4, 8),
                    query=rng.choice(["clique", "near_clique"]), k=rng.choice([5, 7]))
    return dict(family="batch", graphs=rng.randint(3, 10), nmin=rng.randint(300, 700), nmax=_log_int(rng, 2000, 10000),
                query="batch", k=rng.randint(4, 5))


def _er_edges(n, m, seed):
    """m distinct undirected edges of n vertices, uniformly at random (numpy)."""
    rng = np.random.default_rng(seed)
    keys = np.zeros(0, np.int64)
    while len(keys) < m:
        a, b = rng.integers(0, n, (2, 2 * m), dtype=np.int64)
        ok = a != b
        new = (np.minimum(a, b) * n + np.maximum(a, b))[ok]
        keys = np.unique(np.concatenate([keys, new]))
    keys = rng.permutation(keys)[:m]
    return (keys // n).astype(np.int32), (keys % n).astype(np.int32)


def _graph(c, seed):
    if c["family"] == "er":
        s, d = _er_edges(c["n"], c["m"], seed)
        return dm.Graph.from_edges(s, d, c["n"])
    if c["family"] == "chunglu":
        return dm.Graph.chung_lu(c["n"], c["m"], c["gamma"], c["wmax"], seed + 1)
    if c["family"] == "ba":
        return dm.Graph.barabasi_albert(c["n"], c["m"], c["planted"], 8, 12, seed + 1)
    return dm.Graph.rmat(c["scale"], c["ef"], 0.57, 0.19, 0.19, seed + 1)


def _batch_specs(c, seed):
    """The graphs of a batch: half Erdos-Renyi, half Chung-Lu, sizes log-uniform."""
    rng = np.random.default_rng(seed)
    out = []
    for i in range(c["graphs"]):
        n = int(round(math.exp(rng.uniform(math.log(c["nmin"]), math.log(c["nmax"])))))
        avg = float(rng.uniform(4, 20))
        spec = dict(family="er", n=n, m=int(n * avg / 2))
        if i % 2:
            spec = dict(family="chunglu", n=n, m=int(n * avg / 2), gamma=float(rng.uniform(2.1, 2.8)),
                        wmax=float(min(n / 8.0, 4.0 * avg)))
        out.append(spec)
    return out


def prepare(case, seed):
    st = dict(case=case)
    if case["family"] == "batch":
        graphs = [_graph(s, seed * 1000 + i) for i, s in enumerate(_batch_specs(case, seed))]
        st["graphs"], st["batch"] = graphs, dm.Batch(graphs)
        st["queries"] = [(g, mode, k) for g in range(len(graphs))
                         for mode, ks in (("clique", range(3, 7)), ("motif", range(3, case["k"] + 1))) for k in ks]
        return st
    g = st["graph"] = _graph(case, seed)
    st["cfg"] = None
    if case["query"] == "near_clique":
        st["dfs"] = dm.Dfs(g, case["k"], dm.DM_PATTERN_NEAR_CLIQUE)
    elif case.get("learned"):
        g.sched_train(False, 4, epochs=30, seed=1)
        st["cfg"] = dm.config(sched=dm.DM_SCHED_LEARNED)
    return st


def run(state):
    c = state["case"]
    if c["query"] == "batch":
        res, _ = state["batch"].run(state["queries"])
        return np.concatenate([np.atleast_1d(np.asarray(r, np.uint64)) for r in res])
    if c["query"] == "near_clique":
        return state["dfs"].run()[0]
    if c["query"] == "clique":
        return state["graph"].clique_count(c["k"], state["cfg"])
    return state["graph"].motif_count(c["k"], state["cfg"])[1]


def _edges(c):
    if c["family"] == "ba":
        return c["n"], c["n"] * c["m"] + 45 * c["planted"]
    if c["family"] == "rmat":
        return 1 << c["scale"], c["ef"] << c["scale"]
    return c["n"], c["m"]


_CLASSES = {3: 3, 4: 10, 5: 33, 6: 155, 7: 1043}  # histogram slots


def work(case):
    """Each adjacency list read once (32-bit ids, two 64-bit offsets per
    vertex), each result written once; one operation per adjacency entry."""
    if case["family"] == "batch":
        sizes = [_edges(s) for s in _batch_specs(case, 0)]
        queries, outs = 4 + case["k"] - 2, 4 + sum(_CLASSES[k] for k in range(3, case["k"] + 1))
    else:
        sizes, queries = [_edges(case)], 1
        outs = _CLASSES[case["k"]] if case["query"] == "motif" else 1
    return {"bytes": sum(8 * m + 16 * n + 8 * outs for n, m in sizes),
            "flops": sum(2 * m * queries for _, m in sizes)}


def exact(case, seed):
    """Triangles and three-vertex motifs of the numpy-made random graphs, from
    the adjacency matrix in 64-bit floats (exact at these sizes)."""
    if case["family"] != "er" or case["k"] != 3 or case["n"] > 6000:
        return None
    s, d = _er_edges(case["n"], case["m"], seed)
    a = np.zeros((case["n"], case["n"]))
    a[s, d] = a[d, s] = 1.0
    triangles = int(round(float(((a @ a) * a).sum()) / 6))
    if case["query"] == "clique":
        return triangles
    deg = a.sum(1)
    wedges = int(round(float((deg * (deg - 1) / 2).sum()))) - 3 * triangles
    hist = np.zeros(3, np.uint64)  # histogram slots: one edge (never connected), wedge, triangle
    hist[1], hist[2] = wedges, triangles
    return hist
