"""The clique list path (roots past 256 out-neighbours, bitmaps off): counts and
algorithmic bytes for every width, with the children given away as often and as
finely as may be, and with nobody to give them to."""
import math

import numpy as np
import pytest

import dumato_amd as dm
from oracle import pyoracle as O
from tests import graphs as G

pytestmark = pytest.mark.gpu

OPTIONS = [dict(), dict(steal=0), dict(steal_min=2, steal_period=0), dict(lds_bytes=256), dict(blocks=1, waves_per_block=1),
           dict(blocks=1024, steal_min=2)]


@pytest.mark.parametrize("w", [64, 32, 16, 8])
@pytest.mark.parametrize("n,p", [(60, 0.5), (300, 0.08), (1000, 0.02)])
def test_bitmaps_off(n, p, w):
    s, d, nv = G.gnp(n, p, 700 + n)
    g, ref = dm.Graph.from_edges(s, d, nv), O.csr_from_edges(s, d, nv)
    _, ro = O.relabel(ref, oriented=True)
    for k in (4, 5, 6):
        want, by = O.clique_count(ref, k), O.clique_bytes(ro, k)
        for kw in OPTIONS:
            print("case lists n=%d k=%d w=%d %s" % (n, k, w, kw), flush=True)
            assert g.clique_count(k, dm.config(vwave=w, clique_bitmap=0, watchdog_s=60.0, **kw)) == want
            assert g.last_stats()["alg_bytes"] == by


@pytest.mark.parametrize("w", [64, 8])
def test_roots_past_the_bitmaps(w):
    s, d, n = G.complete(300)
    g = dm.Graph.from_edges(s, d, n)
    for kw in (dict(), dict(steal_min=2, steal_period=0)):
        print("case K300 k=4 w=%d %s" % (w, kw), flush=True)
        assert g.clique_count(4, dm.config(vwave=w, watchdog_s=60.0, **kw)) == math.comb(300, 4)
