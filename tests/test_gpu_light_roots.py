"""Light clique roots that share one bitmap, and the rows of wide ones: counts
and algorithmic bytes against the oracle for every worker width, static, range
and learned queues, slices too small for the shared bitmap, and record_costs
(which runs roots one by one)."""
import numpy as np
import pytest

import dumato_amd as dm
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu

OPTIONS = [{}, dict(blocks=8), dict(blocks=2), dict(blocks=8, lds_bytes=2112), dict(blocks=8, lds_bytes=1024),
           dict(blocks=8, record_costs=1), dict(blocks=4, steal_min=2, steal_period=0)]


def reference(g):
    off, adj = (np.array(x) for x in g.csr()[:2])
    src = np.repeat(np.arange(len(off) - 1), np.diff(off))
    up = src < adj
    return O.csr_from_edges(src[up].astype(np.int32), adj[up].astype(np.int32), len(off) - 1)


@pytest.mark.parametrize("w", [64, 32, 16, 8])
@pytest.mark.parametrize("scale,ef", [(11, 4), (12, 8), (9, 16)])
def test_counts_and_bytes(scale, ef, w):
    g = dm.Graph.rmat(scale, ef, .57, .19, .19, 3)
    ref = reference(g)
    _, ro = O.relabel(ref, oriented=True)
    g.sched_train(False, 4, epochs=3, seed=1)
    for k in (3, 4, 5, 6, 7):
        want, by = O.clique_count(ref, k), O.clique_bytes(ro, k)
        for kw in OPTIONS + [dict(blocks=8, sched=dm.DM_SCHED_LEARNED)]:
            print("case rmat s%d clique k=%d w=%d %s" % (scale, k, w, kw), flush=True)
            assert g.clique_count(k, dm.config(vwave=w, watchdog_s=60.0, **kw)) == want
            assert g.last_stats()["alg_bytes"] == by


@pytest.mark.parametrize("sizes", [(1, 1, 62), (31, 33), (32, 32, 1), (64,), (63, 2), (65, 3), (129, 30)])
def test_batches_at_the_lanes_edge(sizes):
    # disjoint complete graphs: their roots' out-degrees run from 0 to size - 1
    src, dst, at, want = [], [], 0, {}
    for n in sizes:
        i, j = np.triu_indices(n, 1)
        src.append(at + i), dst.append(at + j)
        at += n
    g = dm.Graph.from_edges(np.concatenate(src).astype(np.int32), np.concatenate(dst).astype(np.int32), at)
    from math import comb
    for k in (3, 4, 5):
        want = sum(comb(n, k) for n in sizes)
        for blocks in (0, 1):
            print("case complete %s clique k=%d blocks=%d" % (sizes, k, blocks), flush=True)
            assert g.clique_count(k, dm.config(blocks=blocks, watchdog_s=60.0)) == want
