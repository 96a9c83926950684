"""The default shape of every motif size leaves the leaf room for a table in
LDS beside its fixed part (at size 7 the 6-wave kernel's slice does not)."""
import numpy as np
import pytest

import dumato_amd as dm
from oracle import pyoracle as O
from tests import graphs as G, hostcc

pytestmark = pytest.mark.gpu

SMALLEST_TABLE = 1024  # 2^7 buckets of 8 bytes


def test_default_slices_hold_a_table(tmp_path):
    fixed = [int(x) for x in hostcc.run(tmp_path, 'for (int k = 3; k <= 7; k++) printf("%d ", motif_leaf_fixed(64, k));').split()]
    s, d, n = G.gnp(20, 0.3, 1)
    g, ref = dm.Graph.from_edges(s, d, n), O.csr_from_edges(s, d, n)
    for k in (3, 4, 5, 6, 7):
        print("case default slice k=%d" % k, flush=True)
        table = (dm.pattern_table(7)[0], dm.num_classes(7)) if k == 7 else None
        want = O.motif_count(ref, k, table=table) if table else O.motif_count(ref, k)
        tot, hist = g.motif_count(k, dm.config(vwave=64, watchdog_s=60.0))
        assert tot == want[0] and np.array_equal(hist, want[1])
        assert g.last_stats()["lds_bytes"] >= fixed[k - 3] + SMALLEST_TABLE


@pytest.mark.parametrize("w,k", [(8, 4), (8, 5), (8, 7), (16, 7), (32, 7)])
def test_narrow_slices_hold_a_table(tmp_path, w, k):
    fixed = int(hostcc.run(tmp_path, 'printf("%%d", motif_leaf_fixed(%d, %d));' % (w, k)))
    s, d, n = G.gnp(24, 0.3, 2 + k)
    g, ref = dm.Graph.from_edges(s, d, n), O.csr_from_edges(s, d, n)
    print("case narrow slice w=%d k=%d" % (w, k), flush=True)
    table = dict(table=(dm.pattern_table(7)[0], dm.num_classes(7))) if k == 7 else {}
    wt, wh = O.motif_count(ref, k, **table)
    for kw in (dict(), dict(lds_bytes=256)):
        tot, hist = g.motif_count(k, dm.config(vwave=w, watchdog_s=60.0, **kw))
        assert tot == wt and np.array_equal(hist, wh)
        assert (g.last_stats()["lds_bytes"] >= fixed + SMALLEST_TABLE) == (not kw)
