"""The per-worker arena holds the motif leaf's table at every size: the table
is the smallest power of two of 4-byte slots that is at least 1.5 per element
(512 slots at least), over the levels above the leaf."""
from tests import hostcc


def test_motif_arena_holds_the_leaf_table(tmp_path):
    out = hostcc.run(tmp_path, r"""
    auto table = [](int64_t tot) {
        int64_t s = 512;
        while (s < tot + tot / 2) s *= 2;
        return 4 * s;
    };
    for (int K = 3; K <= 7; K++)
        for (int64_t md = 1, step = 1; md < 4000000; md += step, step = 1 + md / 700) {
            int64_t above = 0;
            for (int l = 1; l <= K - 4; l++) above += 10 * (l + 1) * md + 64;
            const int64_t need = above + table(K == 3 ? md : (K - 2) * md);
            if (arena_bound_for((int32_t)md, (int32_t)md, K, true) < need) {
                printf("k=%d degree %lld\n", K, (long long)md);
                break;
            }
            if (leaf_table_bytes(md) != table(md)) printf("table of %lld\n", (long long)md);
        }
    printf("holds\n");
""", include="runtime.h", link=True)
    assert out == "holds\n"
