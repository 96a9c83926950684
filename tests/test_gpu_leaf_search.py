"""The motif leaf's count of a neighbour list's entries above the root: hubs
whose lists below them have every length from 0 to past the last round's
remainders, against the oracle."""
import numpy as np
import pytest

import dumato_amd as dm
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3, 4, 5, 7, 8, 13, 16, 17, 33])
@pytest.mark.parametrize("w", [64, 16])
def test_lists_of_every_length(n, w):
    # vertex i of a chain of hubs joins all before it but every third: lists of
    # lengths 0..n-1 in ascending ids, with gaps that the root's id falls into
    s, d = zip(*[(j, i) for i in range(n) for j in range(i) if (i + j) % 3 or j + 1 == i])
    s, d = np.array(s, np.int32), np.array(d, np.int32)
    g, ref = dm.Graph.from_edges(s, d, n), O.csr_from_edges(s, d, n)
    for k in (3, 4, 5):
        print("case chain n=%d motif k=%d w=%d" % (n, k, w), flush=True)
        _, got = g.motif_count(k, dm.config(vwave=w, watchdog_s=60.0))
        _, want = O.motif_count(ref, k)
        assert np.array_equal(got, want)
        assert g.last_stats()["alg_bytes"] == O.motif_bytes(ref, k)
