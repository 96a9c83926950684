"""Step-API kernels of a user's own (tests/user_kernels.hip), which mix the steps
in ways the library's kernels do not."""
import ctypes
import os

import numpy as np
import pytest

import dumato_amd as dm
from tests import graphs as G

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "libuser_kernels.so")


def union_pairs(s, d, n):
    """In degree-rank ids: pairs x < y of (N(a) | N(b)) above a, b in N(a) above
    a, y in N(a) & N(b)."""
    adj = np.zeros((n, n), bool)
    adj[s, d] = adj[d, s] = True
    order = np.lexsort((np.arange(n), adj.sum(1)))
    adj = adj[np.ix_(order, order)]
    total = 0
    for a in range(n):
        for b in np.nonzero(adj[a])[0]:
            if b > a:
                union = np.nonzero((adj[a] | adj[b]) & (np.arange(n) > a))[0]
                both = adj[a] & adj[b]
                total += sum(i for i, y in enumerate(union) if both[y])
    return total


@pytest.mark.parametrize("w", [8, 64])
@pytest.mark.parametrize("n,p", [(40, 0.3), (150, 0.2)])
def test_pairs_of_a_union_in_id_order(w, n, p):
    dm.lib()
    f = ctypes.CDLL(LIB).user_union_pairs
    f.restype = ctypes.c_void_p
    s, d, nv = G.gnp(n, p, 33 + n)
    print("case user kernel union pairs n=%d w=%d" % (n, w), flush=True)
    st = dm.Dfs(dm.Graph.from_edges(s, d, nv), 4, dm.DM_PATTERN_MOTIF, dm.dfs_config(vwave=w, threshold=100))
    tot, out, _ = st.run(f(w))
    assert int(out[0]) == tot == union_pairs(s, d, nv)
