"""Leaf nodes of more than 2,730 elements, whose edge counts go to the class
counters in parts: a hub behind a path, its other neighbours a circulant graph.

Every connected K-subset with the path's end r (the lowest rank) is the path,
the hub and three of the hub's other neighbours; its class is fixed by the
edges among the three."""
import math

import numpy as np
import pytest

import dumato_amd as dm
from tests import hostcc
from tests.test_gpu_motif_leaf import classes, closed_form, friendship


def hub_behind_a_path(K, n):
    path = K - 4
    ring = path + 1 + np.arange(n)
    src = [np.arange(path), np.full(n, path), ring, ring]
    dst = [np.arange(path) + 1, ring, path + 1 + (np.arange(n) + 1) % n, path + 1 + (np.arange(n) + 2) % n]
    return np.concatenate(src).astype(np.int32), np.concatenate(dst).astype(np.int32), path + 1 + n


def class_of(K, edges, q2c):
    adj = np.zeros((K, K), bool)
    for i in range(K - 4):
        adj[i, i + 1] = True
    for x in (K - 3, K - 2, K - 1):
        adj[K - 4, x] = True
    for a, b in edges:
        adj[K - 3 + a, K - 3 + b] = True
    adj |= adj.T
    q = sum(1 << ((s - 2) * (s + 1) // 2 + t) for s in range(2, K) for t in range(s) if adj[s, t])
    return int(q2c[q])


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2740, 4100])
@pytest.mark.parametrize("k", [5, 6, 7])
def test_hub_behind_a_path(k, n):
    print("case hub behind a path n=%d k=%d" % (n, k), flush=True)
    s, d, nv = hub_behind_a_path(k, n)
    tot, hist = dm.Graph.from_edges(s, d, nv).motif_count(k, dm.config(root_begin=0, root_end=1, watchdog_s=60.0))
    tri, path3 = n, 3 * n
    one = 2 * n * (n - 2) - 2 * path3 - 3 * tri
    q2c = dm.pattern_table(k)[0]
    want = {class_of(k, [(0, 1), (1, 2), (0, 2)], q2c): tri, class_of(k, [(0, 1), (1, 2)], q2c): path3,
            class_of(k, [(0, 1)], q2c): one, class_of(k, [], q2c): math.comb(n, 3) - one - path3 - tri}
    assert {i: int(c) for i, c in enumerate(hist) if c} == want
    assert tot == math.comb(n, 3)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1365, 1366, 2049, 2600])
@pytest.mark.parametrize("w", [64, 16])
def test_friendship_k4(n, w):
    print("case friendship n=%d k=4 w=%d" % (n, w), flush=True)
    s, d, nv = friendship(n)
    tot, hist = dm.Graph.from_edges(s, d, nv).motif_count(4, dm.config(vwave=w, watchdog_s=60.0))
    want = closed_form(n, 4)
    assert tot == sum(want.values())
    assert {i: int(c) for i, c in enumerate(hist) if c} == {classes(4)[p]: c for p, c in want.items() if c}


def test_counts_between_flushes_fit_32_bits(tmp_path):
    out = hostcc.run(tmp_path, r"""
    // the most elements of a node that is not flushed, by its table's slots
    int64_t most = 0;
    while (leaf_table_bits(most + 1) < kLeafWideBits) most++;
    if (most * (most - 1) / 2 > UINT32_MAX) printf("narrow\n");
    // a flush's elements times the largest out-degree of 2^43 edges
    if ((uint64_t)kLeafFlush << 22 > 1ull << 32 || kLeafFlush % 64) printf("wide\n");
    printf("fit\n");
""")
    assert out == "fit\n"
