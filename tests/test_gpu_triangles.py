"""k = 3 cliques: the table of N+(root) at its size steps and past the LDS
slice (list intersection there), out-lists longer than a stream chunk, root
ranges and learned pieces; counts and algorithmic bytes."""
import math

import numpy as np
import pytest

import dumato_amd as dm
from oracle import pyoracle as O
from tests import graphs as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3, 65, 154, 155, 309, 310, 615, 1231, 2200])
def test_complete_graphs(n):
    # root 0 of K_n has n - 1 out-neighbours
    s, d, nv = G.complete(n)
    g = dm.Graph.from_edges(s, d, nv)
    for w, lds in ((64, 0), (64, 256), (16, 0), (8, 2048)):
        print("case K%d triangles w=%d lds=%d" % (n, w, lds), flush=True)
        assert g.clique_count(3, dm.config(vwave=w, lds_bytes=lds, watchdog_s=60.0)) == math.comb(n, 3)


@pytest.mark.parametrize("n,p", [(50, 0.5), (400, 0.1), (700, 0.3)])
def test_random_graphs_against_the_oracle(n, p):
    s, d, nv = G.gnp(n, p, 500 + n)
    g, ref = dm.Graph.from_edges(s, d, nv), O.csr_from_edges(s, d, nv)
    _, ro = O.relabel(ref, oriented=True)
    want, by = O.clique_count(ref, 3), O.clique_bytes(ro, 3)
    g.sched_train(False, 3, epochs=3, seed=1)
    for kw in (dict(), dict(vwave=32), dict(vwave=8), dict(steal=0), dict(steal_min=2, steal_period=0),
               dict(sched=dm.DM_SCHED_LEARNED)):
        print("case gnp n=%d triangles %s" % (n, kw), flush=True)
        assert g.clique_count(3, dm.config(watchdog_s=60.0, **kw)) == want
        assert g.last_stats()["alg_bytes"] == by
    h = nv // 3
    a = g.clique_count(3, dm.config(root_end=h))
    assert a + g.clique_count(3, dm.config(root_begin=h)) == want
    g.clique_count(3, dm.config(per_root=1))
    assert int(g.last_root_counts().sum()) == want
