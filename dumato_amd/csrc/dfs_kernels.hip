// Kernels written against the step API of include/dumato_device.h, in the
// shape of the reference's user kernels:
//   dfs_clique_pa   src/main/clique_PA.cu:9-32
//   dfs_clique_wc   src/DM_WCV/clique_DM_WCV8.cu:8-34
//   dfs_motifs      src/main/motifs_DM_WCLB.cu:9-36
//   dfs_q_pa        src/main/q4_PA.cu:9-32 .. q13_PA.cu (near-clique query)
// They run under dm_dfs_run (host-driven load balancing).  The fused kernels
// of enum_kernel.hip compute the same counts faster; these exist so that the
// reference's programming model, and its stop/snapshot/donate balancing,
// have a drop-in here.
#include "../../include/dumato_device.h"
#include "internal.h"

namespace dm {

template <int W>
__global__ __launch_bounds__(256) void dfs_clique_pa(dm_dfs_data d) {
    dm_device::Worker<W> DM;
    DM.start_clique(d);
    while (DM.active() && DM.balanced()) {
        if (DM.getCurrentNumberOfExtensions() == -1) DM.extend_clique();
        if (DM.getCurrentNumberOfExtensions() != 0) {
            if (DM.last_level()) {
                DM.aggregate_counter();
                DM.backward_clique();
            } else {
                DM.forward();
            }
        } else {
            DM.backward_clique();
        }
    }
    DM.end();
}

template <int W>
__global__ __launch_bounds__(256) void dfs_clique_wc(dm_dfs_data d) {
    dm_device::Worker<W> DM;
    DM.start(d);
    while (DM.active() && DM.balanced()) {
        if (DM.getCurrentNumberOfExtensions() == -1) {
            DM.extend();
            if (DM.k() > 0) DM.filterClique();
        }
        if (DM.getCurrentNumberOfExtensions() != 0) {
            if (DM.last_level()) {
                DM.aggregate_counter();
                DM.backward();
            } else {
                DM.forward();
            }
        } else {
            DM.backward();
        }
    }
    DM.end();
}

template <int W>
__global__ __launch_bounds__(256) void dfs_motifs(dm_dfs_data d) {
    dm_device::Worker<W> DM;
    DM.start_induce(d);
    while (DM.active() && DM.balanced()) {
        if (DM.getCurrentNumberOfExtensions() == -1) {
            DM.extend(0, DM.k());
            if (DM.k() > 0) DM.canonicalFilter2();
        }
        if (DM.getCurrentNumberOfExtensions() != 0) {
            if (DM.last_level()) {
                DM.aggregate_pattern();
                DM.backward_induce();
            } else {
                DM.forward_induce();
            }
        } else {
            DM.backward_induce();
        }
    }
    DM.end();
}

// q4_PA .. q13_PA (src/main/q4_PA.cu:9-32): the near-clique query with the
// state's K
template <int W>
__global__ __launch_bounds__(256) void dfs_q_pa(dm_dfs_data d) {
    dm_device::Worker<W> DM;
    DM.start_q(d);
    while (DM.active() && DM.balanced()) {
        if (DM.getCurrentNumberOfExtensions() == -1) DM.extend_q();
        if (DM.getCurrentNumberOfExtensions() != 0) {
            if (DM.last_level()) {
                DM.aggregate_counter();
                DM.backward_q();
            } else {
                DM.forward();
            }
        } else {
            DM.backward_q();
        }
    }
    DM.end();
}

// ---- state kept on the device between launches (dfs.cpp) ----
// The initial state: nobody working, root t of `roots` in slot t / workers of
// worker t mod workers, everything else clear.
__global__ __launch_bounds__(256) void dfs_reset_kernel(dm_dfs_data d, const int32_t *roots, int nroots) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x, step = (size_t)gridDim.x * blockDim.x;
    const size_t W = (size_t)d.workers, J = (size_t)d.jobs_per_worker;
    for (size_t t = i; t < W * DM_DFS_MAXK; t += step) d.next[t] = d.fixed[t] = 0;
    for (size_t w = i; w < W; w += step) {
        d.k[w] = -1;
        d.status[w] = 1;
        d.job_valid[w] = (size_t)nroots > w ? (int)(((size_t)nroots - 1 - w) / W) + 1 : 0;
        d.job_cur[w] = 0;
    }
    for (size_t t = i; t < (size_t)nroots; t += step) {
        const size_t j = (t % W) * J + t / W;
        d.jobs[j * DM_DFS_MAXK] = roots[t];
        d.job_level[j] = 0;
        d.job_ind[j] = 0;
    }
    for (size_t t = i; t < (size_t)(d.ncls > 1 ? d.ncls : 1); t += step) d.result[t] = 0;
}

// The unspent extensions of the busy workers' levels below the last one, end
// to end from at[w] (< 0: not wanted), one block per worker.
__global__ __launch_bounds__(64) void dfs_gather_kernel(dm_dfs_data d, const int64_t *at, int32_t *out) {
    const size_t w = blockIdx.x;
    int64_t o = at[w];
    if (o < 0) return;
    for (int l = 0; l <= d.k[w] && l < d.K - 2; l++) {
        const int n = d.next[w * DM_DFS_MAXK + l];
        if (n <= 0) continue;
        const size_t lo = d.motif ? (size_t)d.cap_base * (size_t)(l * (l + 1) / 2) : (size_t)d.cap_base * (size_t)l;
        const int32_t *src = d.ext + w * (size_t)d.ext_per_worker + lo;
        for (int t = threadIdx.x; t < n; t += 64) out[o + t] = src[t];
        o += n;
    }
}

// Writes moved jobs (slot, level, induction, prefix) into the workers' queues.
__global__ __launch_bounds__(256) void dfs_scatter_kernel(dm_dfs_data d, const DfsMove *mv, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const size_t s = (size_t)mv[i].slot;
    d.job_level[s] = mv[i].level;
    d.job_ind[s] = mv[i].ind;
    for (int l = 0; l < DM_DFS_MAXK; l++) d.jobs[s * DM_DFS_MAXK + l] = mv[i].id[l];
}

static int launched(const char *what) {
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? DM_OK : set_error(DM_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
}
int dfs_reset_launch(const dm_dfs_data &d, const int32_t *roots, int nroots, void *stream) {
    const size_t work = (size_t)d.workers * DM_DFS_MAXK;
    hipLaunchKernelGGL(dfs_reset_kernel, dim3((unsigned)((work + 255) / 256)), dim3(256), 0, (hipStream_t)stream, d,
                       roots, nroots);
    return launched("step-API reset");
}
int dfs_gather_launch(const dm_dfs_data &d, const int64_t *at, int32_t *out, void *stream) {
    hipLaunchKernelGGL(dfs_gather_kernel, dim3(d.workers), dim3(64), 0, (hipStream_t)stream, d, at, out);
    return launched("step-API gather");
}
int dfs_scatter_launch(const dm_dfs_data &d, const DfsMove *mv, int n, void *stream) {
    hipLaunchKernelGGL(dfs_scatter_kernel, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, d, mv, n);
    return launched("step-API scatter");
}

template <int W>
static const void *dfs_kernel_w(int kind) {
    switch (kind) {
        case DM_DFS_CLIQUE_PA: return (const void *)dfs_clique_pa<W>;
        case DM_DFS_CLIQUE_WC: return (const void *)dfs_clique_wc<W>;
        case DM_DFS_MOTIF: return (const void *)dfs_motifs<W>;
        case DM_DFS_NEAR_CLIQUE: return (const void *)dfs_q_pa<W>;
        default: return nullptr;
    }
}

}  // namespace dm

extern "C" int dm_dfs_kernel(int kind, int vwave, const void **kernel) {
    using namespace dm;
    if (!kernel) return set_error(DM_ERR_ARG, "kernel is NULL");
    const void *k = nullptr;
    switch (vwave) {
        case 8: k = dfs_kernel_w<8>(kind); break;
        case 16: k = dfs_kernel_w<16>(kind); break;
        case 32: k = dfs_kernel_w<32>(kind); break;
        case 64: k = dfs_kernel_w<64>(kind); break;
        default: return set_error(DM_ERR_ARG, "vwave must be 8, 16, 32 or 64 (got %d)", vwave);
    }
    if (!k) return set_error(DM_ERR_ARG, "unknown step-API kernel %d", kind);
    *kernel = k;
    return DM_OK;
}
