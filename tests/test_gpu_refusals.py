"""Requests that are turned down: many idle workers beside a few busy ones,
whose blocks run out of work over and over; counts stay exact."""
import math

import numpy as np
import pytest

import dumato_amd as dm
from tests import graphs as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w", [8, 64])
def test_few_busy_workers_many_askers(w):
    # many small complete graphs' roots in few blocks' worth of workers
    parts, at = [], 0
    for n in [40] * 12 + [5] * 200:
        s, d, _ = G.complete(n)
        parts.append((s + at, d + at))
        at += n
    g = dm.Graph.from_edges(np.concatenate([p[0] for p in parts]).astype(np.int32),
                            np.concatenate([p[1] for p in parts]).astype(np.int32), at)
    for k in (4, 5, 6):
        want = 12 * math.comb(40, k) + 200 * math.comb(5, k)
        for rep in range(3):
            print("case refusals k=%d w=%d rep=%d" % (k, w, rep), flush=True)
            cfg = dm.config(vwave=w, blocks=128, steal_min=2, steal_period=0, watchdog_s=60.0)
            assert g.clique_count(k, cfg) == want
