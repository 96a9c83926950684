// User kernels against include/dumato_device.h that mix its steps in ways the
// library's own kernels do not (built by dumato_amd/Makefile, run by
// test_gpu_user_kernels.py).
#include "../include/dumato_device.h"

// Pairs x < y of the union of N(id[0]) and N(id[1]) above id[0], y adjacent to
// both: the union's list (extend) does not ascend, extend_q takes the entries
// above the vertex placed, whatever their order.
template <int W>
__global__ __launch_bounds__(256) void union_pairs(dm_dfs_data d) {
    dm_device::Worker<W> DM;
    DM.start(d);
    while (DM.active() && DM.balanced()) {
        if (DM.getCurrentNumberOfExtensions() == -1) {
            if (DM.k() <= 1) {
                DM.extend(0, DM.k());
            } else {
                DM.extend_q();
                DM.filterClique();
            }
        }
        if (DM.getCurrentNumberOfExtensions() != 0 && !DM.last_level()) {
            DM.forward();
        } else {
            if (DM.last_level()) DM.aggregate_counter();
            DM.backward();
        }
    }
    DM.end();
}

extern "C" const void *user_union_pairs(int w) {
    return w == 8 ? (const void *)union_pairs<8> : w == 64 ? (const void *)union_pairs<64> : nullptr;
}
