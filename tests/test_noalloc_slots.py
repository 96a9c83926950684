"""Static scratch: every worker of a launch has a job slot, so that all can ask
for work, at every width (host arithmetic); narrow launches of more than 8,192
workers count right and share work (GPU)."""
import math

import numpy as np
import pytest

import dumato_amd as dm
from oracle import pyoracle as O
from tests import graphs as G, hostcc


def test_every_worker_has_a_slot(tmp_path):
    out = hostcc.run(tmp_path, r"""
    const int64_t scratch = (int64_t)64 << 20;  // more than the arenas have
    for (int motif = 0; motif < 2; motif++)
        for (int K = 3; K <= (motif ? 7 : 12); K++)
            for (int vw = 8; vw <= 64; vw *= 2) {
                const int wpb = 256 / vw;
                const int64_t arena = arena_bound_for(1, 1, K, motif);
                // what fits the 256 CUs, 8 blocks of 4 waves each, and the scratch
                const int64_t blocks = std::min<int64_t>(2048, scratch / (arena * wpb)), workers = blocks * wpb;
                if (scratch_slots((int)workers, (int)blocks) != workers)
                    printf("motif %d k=%d width %d: %lld workers\n", motif, K, vw, (long long)workers);
            }
    printf("all\n");
""", include="runtime.h", link=True)
    assert out == "all\n"


@pytest.mark.gpu
def test_more_than_8192_narrow_workers():
    s, d, n = G.gnp(400, 0.25, 12)
    g, ref = dm.Graph.from_edges(s, d, n), O.csr_from_edges(s, d, n)
    g.clique_count(3)  # uploads the graph
    wt, wh = O.motif_count(ref, 3)
    for blocks, w in ((330, 8), (660, 16), (0, 8)):
        print("case noalloc motif k=3 w=%d blocks=%d" % (w, blocks), flush=True)
        for _ in range(3):
            t, h = g.count_noalloc(True, 3, dm.config(vwave=w, blocks=blocks, watchdog_s=60.0))
            assert t == wt and np.array_equal(h, wh)
            if blocks:
                assert g.last_stats()["workers"] > 8192


@pytest.mark.gpu
def test_as_many_one_wave_blocks_as_arenas_fit():
    # 10,000 blocks of one worker: fewer slots than workers
    s, d, n = G.complete(30)
    g = dm.Graph.from_edges(s, d, n)
    g.clique_count(3)
    print("case noalloc 10000 blocks", flush=True)
    t, _ = g.count_noalloc(True, 3, dm.config(vwave=64, waves_per_block=1, blocks=10000, watchdog_s=60.0))
    assert t == math.comb(30, 3)
