"""Class counters that all workers of a block add to: one block, many workers
whose leaf nodes fall into the same classes at the same time."""
import numpy as np
import pytest

import dumato_amd as dm
from oracle import pyoracle as O
from tests import graphs as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,waves", [(64, 4), (64, 2), (8, 4), (16, 4)])
def test_one_block(w, waves):
    # 300 copies of a random graph on 12 vertices
    s, d, n = G.gnp(12, 0.5, 9)
    src = np.concatenate([s + i * n for i in range(300)]).astype(np.int32)
    dst = np.concatenate([d + i * n for i in range(300)]).astype(np.int32)
    g, ref = dm.Graph.from_edges(src, dst, 300 * n), O.csr_from_edges(s, d, n)
    for k in (3, 4, 5, 6):
        print("case one block w=%d waves=%d k=%d" % (w, waves, k), flush=True)
        wt, wh = O.motif_count(ref, k)
        tot, hist = g.motif_count(k, dm.config(vwave=w, blocks=1, waves_per_block=waves, watchdog_s=60.0))
        assert tot == 300 * wt and np.array_equal(hist, 300 * wh)
