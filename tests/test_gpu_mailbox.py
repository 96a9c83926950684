"""The workers' mailboxes: grids smaller and larger than what is resident (the
queues of blocks that start late are found by idle workers), one worker per
wave up to eight, stealing on and off, one heavy root shared by everybody;
counts and algorithmic bytes stay exact."""
import math

import numpy as np
import pytest

import dumato_amd as dm
from oracle import pyoracle as O
from tests import graphs as G

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def graph():
    g = dm.Graph.chung_lu(4000, 24000, 2.3, 200.0, 11)
    n = g.info()[0]
    return g, O.CSR(n, *g.csr())


@pytest.mark.parametrize("blocks", [1, 5, 333, 4096])
@pytest.mark.parametrize("w", [16, 64])
def test_grid_sizes(graph, blocks, w):
    g, ref = graph
    _, ro = O.relabel(ref, oriented=True)
    wt, wh = O.motif_count(ref, 4)
    for steal in (1, 0):
        print("case blocks=%d w=%d steal=%d" % (blocks, w, steal), flush=True)
        cfg = dm.config(blocks=blocks, vwave=w, steal=steal, watchdog_s=60.0)
        for k in (3, 5):
            assert g.clique_count(k, cfg) == O.clique_count(ref, k)
            assert g.last_stats()["alg_bytes"] == O.clique_bytes(ro, k)
        tot, hist = g.motif_count(4, cfg)
        assert tot == wt and np.array_equal(hist, wh)


@pytest.mark.parametrize("waves", [1, 2, 4])
def test_one_heavy_root(waves):
    # a clique on 60 vertices beside isolated edges: almost all the work is in
    # a few roots, every other worker asks for a share
    s, d, n = G.complete(60)
    e = np.arange(60, 3060, 2, dtype=np.int32)
    g = dm.Graph.from_edges(np.concatenate([s, e]), np.concatenate([d, e + 1]), 3060)
    for k in (4, 6, 7):
        for period in (0, 2):
            print("case heavy root k=%d waves=%d period=%d" % (k, waves, period), flush=True)
            cfg = dm.config(waves_per_block=waves, steal_min=2, steal_period=period, watchdog_s=60.0)
            assert g.clique_count(k, cfg) == math.comb(60, k)
    tot, hist = g.motif_count(5, dm.config(waves_per_block=waves, watchdog_s=60.0))
    assert tot == math.comb(60, 5) and int(hist[32]) == tot


def test_repeated_launches_alternate_pattern_and_grid(graph):
    # slots, mailboxes and tags are reused by every launch
    g, ref = graph
    want = {k: O.clique_count(ref, k) for k in (3, 4)}
    wt, wh = O.motif_count(ref, 3)
    for i in range(12):
        print("case relaunch %d" % i, flush=True)
        cfg = dm.config(blocks=(0, 3, 700)[i % 3], watchdog_s=60.0)
        assert g.clique_count(3 + i % 2, cfg) == want[3 + i % 2]
        tot, hist = g.motif_count(3, cfg)
        assert tot == wt and np.array_equal(hist, wh)
