"""The bitmap clique path's stages (k >= 6, every k past 6 included): set
widths of 1, 2 and 4 words, stages narrowed by small LDS slices or in the
arena, every worker width; counts and algorithmic bytes against the oracle or
closed forms."""
import math

import numpy as np
import pytest

import dumato_amd as dm
from oracle import pyoracle as O
from tests import graphs as G

pytestmark = pytest.mark.gpu

SHAPES = [(64, 0), (64, 256), (64, 4096), (32, 0), (16, 1024), (8, 0)]


@pytest.mark.parametrize("n,p", [(60, 0.5), (110, 0.4), (170, 0.25)])
@pytest.mark.parametrize("w,lds", SHAPES)
def test_random_graphs_against_the_oracle(n, p, w, lds):
    s, d, nv = G.gnp(n, p, 300 + n)
    g, ref = dm.Graph.from_edges(s, d, nv), O.csr_from_edges(s, d, nv)
    _, ro = O.relabel(ref, oriented=True)
    for k in (4, 5, 6, 7, 8, 9):
        print("case gnp n=%d clique k=%d w=%d lds=%d" % (n, k, w, lds), flush=True)
        assert g.clique_count(k, dm.config(vwave=w, lds_bytes=lds, watchdog_s=60.0)) == O.clique_count(ref, k)
        assert g.last_stats()["alg_bytes"] == O.clique_bytes(ro, k)


def bipartite_with_clique(a, b, c):
    """Complete bipartite graph (sides a and b) plus a clique on c vertices of
    side a: wide out-neighbourhoods (b) that hold few edges."""
    x, y = np.meshgrid(np.arange(a), a + np.arange(b), indexing="ij")
    i, j = np.triu_indices(c, 1)
    src = np.concatenate([x.ravel(), a - c + i])
    dst = np.concatenate([y.ravel(), a - c + j])
    return src.astype(np.int32), dst.astype(np.int32), a + b


@pytest.mark.parametrize("b", [100, 128, 129, 250, 256, 257])
def test_wide_roots_closed_form(b):
    # word counts 2 and 4, the last bitmap root and the first past it
    c = 11
    s, d, nv = bipartite_with_clique(b, b, c)
    g = dm.Graph.from_edges(s, d, nv)
    for k in (4, 5, 6, 7, 9, 12):
        want = math.comb(c, k) + b * math.comb(c, k - 1)
        for w, lds in ((64, 0), (64, 2048), (16, 0)):
            print("case bipartite b=%d clique k=%d w=%d lds=%d" % (b, k, w, lds), flush=True)
            assert g.clique_count(k, dm.config(vwave=w, lds_bytes=lds, watchdog_s=60.0)) == want


def test_complete_graph_every_size():
    s, d, n = G.complete(26)
    g = dm.Graph.from_edges(s, d, n)
    for k in range(3, 13):
        print("case K26 clique k=%d" % k, flush=True)
        assert g.clique_count(k, dm.config(watchdog_s=60.0)) == math.comb(26, k)


@pytest.mark.parametrize("n,p", [(64, 0.8), (120, 0.6), (220, 0.35)])
def test_pairs_of_a_child_given_away(n, p):
    # few dense roots, many idle workers, the smallest pieces: children's pairs
    # travel as jobs of their own; with a learned partition too
    s, d, nv = G.gnp(n, p, 70 + n)
    ref = O.csr_from_edges(s, d, nv)
    _, ro = O.relabel(ref, oriented=True)
    for k in (6, 7):
        want, by = O.clique_count(ref, k), O.clique_bytes(ro, k)
        g = dm.Graph.from_edges(s, d, nv)
        g.sched_train(False, 4, epochs=3, seed=1)
        for w, kw in ((64, {}), (16, {}), (64, dict(sched=dm.DM_SCHED_LEARNED))):
            print("case gnp n=%d clique k=%d w=%d %s" % (n, k, w, kw), flush=True)
            cfg = dm.config(vwave=w, blocks=64, steal_min=2, steal_period=0, watchdog_s=60.0, **kw)
            for _ in range(2):
                assert g.clique_count(k, cfg) == want
                assert g.last_stats()["alg_bytes"] == by


@pytest.mark.parametrize("n,p", [(70, 0.75), (115, 0.6), (150, 0.45)])
def test_narrow_stages_beside_a_childs_bitmap(n, p):
    # slices where a child's own bitmap fits LDS but its stages are narrowed,
    # down to those too small for the prefix of k = 6's last step
    s, d, nv = G.gnp(n, p, 500 + n)
    ref = O.csr_from_edges(s, d, nv)
    _, ro = O.relabel(ref, oriented=True)
    want, by = O.clique_count(ref, 6), O.clique_bytes(ro, 6)
    g = dm.Graph.from_edges(s, d, nv)
    for lds in range(1536, 9216, 192):
        print("case gnp n=%d clique k=6 lds=%d" % (n, lds), flush=True)
        assert g.clique_count(6, dm.config(vwave=64, lds_bytes=lds, watchdog_s=60.0)) == want
        assert g.last_stats()["alg_bytes"] == by
