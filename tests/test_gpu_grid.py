"""The default grid on graphs with fewer vertices than the workers that fit:
at least a block per CU at every width, all that fits for a long motif query,
no more workers than vertices for a short one."""
import numpy as np
import pytest

import dumato_amd as dm
from oracle import pyoracle as O
from tests import graphs as G

pytestmark = pytest.mark.gpu


def reference(g):
    off, adj = (np.array(x) for x in g.csr()[:2])
    src = np.repeat(np.arange(len(off) - 1), np.diff(off))
    up = src < adj
    return O.csr_from_edges(src[up].astype(np.int32), adj[up].astype(np.int32), len(off) - 1)


@pytest.mark.parametrize("w", [8, 16, 32, 64])
def test_narrow_widths_use_every_cu(w):
    g = dm.Graph.erdos_renyi(1000, 5000, 21)
    ref = reference(g)
    print("case grid w=%d" % w, flush=True)
    assert g.clique_count(4, dm.config(vwave=w)) == O.clique_count(ref, 4)
    assert g.last_stats()["blocks"] >= 256
    tot, hist = g.motif_count(4, dm.config(vwave=w))
    wt, wh = O.motif_count(ref, 4)
    assert tot == wt and np.array_equal(hist, wh)
    assert g.last_stats()["blocks"] >= 256


def test_a_long_query_takes_what_fits():
    s, d, n = G.gnp(90, 0.5, 4)
    g, ref = dm.Graph.from_edges(s, d, n), O.csr_from_edges(s, d, n)
    print("case long query", flush=True)
    tot, hist = g.motif_count(5, dm.config(vwave=64))
    wt, wh = O.motif_count(ref, 5)
    assert tot == wt and np.array_equal(hist, wh)
    assert g.last_stats()["workers"] >= 6144


def test_a_short_query_keeps_to_the_vertices():
    g = dm.Graph.erdos_renyi(3000, 6000, 8)
    ref = reference(g)
    print("case short query", flush=True)
    tot, hist = g.motif_count(4, dm.config(vwave=64))
    wt, wh = O.motif_count(ref, 4)
    assert tot == wt and np.array_equal(hist, wh)
    assert 2048 <= g.last_stats()["workers"] <= 3072
