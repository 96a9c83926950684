"""k = 3 motifs of roots whose table lies in the arena, past the sizes where the
table's power of two steps up: complete graphs (a root of n - 1 out-neighbours,
no wedge) against the closed form."""
import math

import pytest

import dumato_amd as dm
from tests import graphs as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1367, 2732, 2733, 2800, 2843, 4200])
@pytest.mark.parametrize("w", [64, 16])
def test_complete_graphs(n, w):
    print("case K%d motif k=3 w=%d" % (n, w), flush=True)
    s, d, nv = G.complete(n)
    tot, hist = dm.Graph.from_edges(s, d, nv).motif_count(3, dm.config(vwave=w, watchdog_s=60.0))
    assert tot == math.comb(n, 3) and int(hist[2]) == tot
