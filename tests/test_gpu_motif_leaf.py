"""The motif leaf node (pair counts over a hash table of U) where it can go
wrong: U at the edges of a wave, of a table size, and past the LDS table (the
table in the arena), for every width and size it is compiled for.

Friendship graphs (a hub, n disjoint leaf pairs joined to it) have closed
forms: every connected K-subset with K >= 4 is the hub and K-1 leaves, and its
class is fixed by how many of the pairs it holds whole."""
import math

import numpy as np
import pytest

import dumato_amd as dm
from oracle import pyoracle as O
from tests import graphs as G

pytestmark = pytest.mark.gpu


def friendship(n):
    hub = np.zeros(2 * n, np.int32)
    leaf = np.arange(1, 2 * n + 1, dtype=np.int32)
    a = np.arange(1, 2 * n + 1, 2, dtype=np.int32)
    return np.concatenate([hub, a]), np.concatenate([leaf, a + 1]), 2 * n + 1


def closed_form(n, k):
    """{whole pairs held: subsets} of k - 1 of the 2n leaves."""
    return {p: math.comb(n, p) * math.comb(n - p, k - 1 - 2 * p) * 2 ** (k - 1 - 2 * p)
            for p in range((k - 1) // 2 + 1)}


def classes(k):
    """{whole pairs: class id}, from the oracle on a friendship graph whose counts differ."""
    n = 2 * k
    s, d, nv = friendship(n)
    _, hist = O.motif_count(O.csr_from_edges(s, d, nv), k)
    want = closed_form(n, k)
    ids = {p: [i for i in range(len(hist)) if int(hist[i]) == c] for p, c in want.items()}
    assert all(len(v) == 1 for v in ids.values())
    return {p: v[0] for p, v in ids.items()}


@pytest.mark.parametrize("w", [8, 64])
@pytest.mark.parametrize("n", [31, 32, 33, 63, 65, 438, 439, 560, 877, 878, 1100])
def test_closed_forms_at_table_edges_k4(n, w):
    print("case friendship n=%d k=4 w=%d" % (n, w), flush=True)
    s, d, nv = friendship(n)
    tot, hist = dm.Graph.from_edges(s, d, nv).motif_count(4, dm.config(vwave=w, watchdog_s=60.0))
    want = closed_form(n, 4)
    assert tot == sum(want.values())
    assert {i: int(c) for i, c in enumerate(hist) if c} == {classes(4)[p]: c for p, c in want.items() if c}


@pytest.mark.parametrize("n", [31, 33, 219, 220, 438, 439, 600])
def test_closed_forms_at_table_edges_k5(n):
    print("case friendship n=%d k=5" % n, flush=True)
    s, d, nv = friendship(n)
    tot, hist = dm.Graph.from_edges(s, d, nv).motif_count(5, dm.config(watchdog_s=60.0))
    want = closed_form(n, 5)
    assert tot == sum(want.values())
    assert {i: int(c) for i, c in enumerate(hist) if c} == {classes(5)[p]: c for p, c in want.items() if c}


@pytest.mark.parametrize("k,n,p", [(3, 150, 0.5), (4, 70, 0.5), (5, 40, 0.5), (6, 26, 0.4)])
@pytest.mark.parametrize("lds", [0, 256])
def test_dense_graphs_against_the_oracle(k, n, p, lds):
    # dense: many elements of U hold several lists' bits, half the pairs are
    # adjacent; lds = 256: no table in LDS
    s, d, nv = G.gnp(n, p, 40 + k)
    g, ref = dm.Graph.from_edges(s, d, nv), O.csr_from_edges(s, d, nv)
    wt, wh = O.motif_count(ref, k)
    for w in (8, 16, 32, 64):
        print("case gnp n=%d p=%.1f k=%d w=%d lds=%d" % (n, p, k, w, lds), flush=True)
        tot, hist = g.motif_count(k, dm.config(vwave=w, lds_bytes=lds, watchdog_s=60.0))
        assert tot == wt and np.array_equal(hist, wh)
        if k <= 5:
            assert g.last_stats()["alg_bytes"] == O.motif_bytes(ref, k)


def test_learned_pieces_split_a_k3_root():
    # k = 3: the root is the leaf node; a learned partition cuts it by children
    s, d, nv = G.gnp(200, 0.4, 71)
    g, ref = dm.Graph.from_edges(s, d, nv), O.csr_from_edges(s, d, nv)
    g.sched_train(True, 3, epochs=3, seed=2)
    wt, wh = O.motif_count(ref, 3)
    for w in (16, 64):
        print("case learned motif k=3 w=%d" % w, flush=True)
        tot, hist = g.motif_count(3, dm.config(sched=dm.DM_SCHED_LEARNED, vwave=w, watchdog_s=60.0))
        assert tot == wt and np.array_equal(hist, wh)
        assert g.last_stats()["alg_bytes"] == O.motif_bytes(ref, 3)
