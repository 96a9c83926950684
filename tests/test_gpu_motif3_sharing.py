"""k = 3 motifs share work: workers without a root are given children of the
others' roots; the pieces of a root add up."""
import math

import numpy as np
import pytest

import dumato_amd as dm
from oracle import pyoracle as O
from tests import graphs as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w", [64, 16])
def test_children_are_given_away(w):
    # 1,500 roots of up to 1,499 children, more workers than roots
    s, d, n = G.complete(1500)
    g = dm.Graph.from_edges(s, d, n)
    print("case K1500 motif k=3 w=%d" % w, flush=True)
    tot, hist = g.motif_count(3, dm.config(vwave=w, blocks=1024, watchdog_s=60.0))
    assert tot == math.comb(n, 3) and int(hist[2]) == tot
    assert g.last_stats()["donations"] > 0


def test_untouched_roots_of_a_range_are_given_away():
    # a batch's ranges of 32 roots, fewer ranges than workers
    g = dm.Graph.erdos_renyi(16000, 640000, 5)
    batch = dm.Batch([g])
    want, hist = g.motif_count(3)
    print("case batch ER motif k=3", flush=True)
    res, _ = batch.run([(0, "motif", 3)])
    assert np.array_equal(res[0], hist)
    assert batch.last_stats()["donations"] > 0


@pytest.mark.parametrize("n,p", [(600, 0.3), (1100, 0.1)])
def test_chunks_and_pieces_against_the_oracle(n, p):
    s, d, nv = G.gnp(n, p, 900 + n)
    g, ref = dm.Graph.from_edges(s, d, nv), O.csr_from_edges(s, d, nv)
    wt, wh = O.motif_count(ref, 3)
    for kw in (dict(), dict(steal=0), dict(steal_period=0, blocks=512), dict(vwave=8), dict(lds_bytes=256)):
        print("case gnp n=%d motif k=3 %s" % (n, kw), flush=True)
        tot, hist = g.motif_count(3, dm.config(watchdog_s=60.0, **kw))
        assert tot == wt and np.array_equal(hist, wh)
        assert g.last_stats()["alg_bytes"] == O.motif_bytes(ref, 3)
