// Internal declarations shared by the host runtime (C++) and the HIP kernels.
#ifndef DM_INTERNAL_H
#define DM_INTERNAL_H

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <string>
#include <vector>

#include "../../include/dumato.h"

namespace dm {

// ---- limits ---------------------------------------------------------------
constexpr int kMaxK = 12;              // largest clique size; motifs stop at 7
constexpr int kMaxMotifK = 7;
constexpr int kMaxLevels = kMaxK - 2;  // stack levels 0..K-3 (+1 spare)
constexpr int kJobIds = 12;

// ---- errors ---------------------------------------------------------------
int set_error(int code, const char *fmt, ...);
int last_code();

// ---- host graph -------------------------------------------------------------
struct HostCSR {
    int32_t n = 0;
    std::vector<int64_t> off;  // n + 1
    std::vector<int32_t> adj;  // sorted neighbour lists
    int32_t maxdeg = 0;
    int64_t nnz() const { return off.empty() ? 0 : off.back(); }
};

int parse_edgelist(const char *path, std::vector<int32_t> &src, std::vector<int32_t> &dst);
int build_csr(int32_t n_hint, const int32_t *src, const int32_t *dst, size_t m, HostCSR &out);

// ---- pattern tables -----------------------------------------------------------
struct PatternTable {
    int k = 0;
    int ncls = 0;
    std::vector<uint16_t> q2c;       // quick code -> class id
    std::vector<uint64_t> cls_code;  // class id -> canonical code
};
const PatternTable *pattern_table(int k);

// ---- random numbers (xoshiro256**, seeded by splitmix64) ---------------------
struct Rng {
    uint64_t s[4];
    explicit Rng(uint64_t seed) {
        for (int i = 0; i < 4; i++) {
            seed += 0x9E3779B97F4A7C15ull;
            uint64_t z = seed;
            z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
            z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
            s[i] = z ^ (z >> 31);
        }
    }
    static inline uint64_t rotl(uint64_t x, int k) { return (x << k) | (x >> (64 - k)); }
    inline uint64_t next() {
        uint64_t r = rotl(s[1] * 5, 7) * 9, t = s[1] << 17;
        s[2] ^= s[0];
        s[3] ^= s[1];
        s[1] ^= s[2];
        s[0] ^= s[3];
        s[2] ^= t;
        s[3] = rotl(s[3], 45);
        return r;
    }
    inline double uniform() { return (next() >> 11) * (1.0 / 9007199254740992.0); }
    inline uint64_t below(uint64_t n) { return (uint64_t)(uniform() * (double)n) % (n ? n : 1); }
};

// ---- device-side structures (identical layout on host and device) ----------
// A job given away: children [lo, hi) of the node with prefix ids[0..lvl] in
// query q.  Word j holds (tag << 32 | value): words 0..3 = lvl, lo, hi, q;
// words 4.. = ids; of a job on a root's children or their pairs, the last two
// = where the root's rows are published (worker + 1, number; 0: nowhere).
constexpr int kJobWords = 4 + kJobIds;
constexpr int kJobPub = kJobWords - 2;
struct Job {
    uint64_t w[kJobWords];
};

// Scheduler words that workers update while a launch runs, each on its own
// 128-byte line, so that traffic on one never stalls the others.
struct SchedStats {
    unsigned long long donations;
    unsigned long long jobs;
    unsigned long long alg_bytes;
    unsigned long long busy_sum;     // sum over workers of cycles spent in jobs
    unsigned long long busy_max;     // largest per-worker busy cycles
    // timeline (wall-clock ticks): first block start, then the latest worker
    // to start its first job, to find its static queue exhausted, to end its
    // last job and to exit
    unsigned long long t_start, t_first_job, t_static_done, t_last_job, t_exit;
    unsigned long long job_max;         // cycles of the longest single job
    unsigned long long active_workers;  // workers that ran at least one job
    unsigned long long pad[4];
};
static_assert(sizeof(SchedStats) == 128, "one line per copy of the statistics");
// Every block adds its statistics once, when it ends: to one of these copies,
// which the host sums (one copy: 13 same-line atomics of 768 blocks took the
// last 50 us of every clique launch, of 1,536 blocks 125 us of a k >= 5 motif's).
constexpr int kStatCopies = 32;
struct SchedCounters {
    unsigned long long outstanding;  // unfinished jobs (static + donated)
    char pad0[120];
    int32_t started;                 // blocks that have begun to run
    char pad2[124];
    int32_t error;                   // 1 watchdog, 2 arena overflow, 3 bad job
    char pad5[124];
    SchedStats st[kStatCopies];
};
SchedStats sched_totals(const SchedCounters &c);
// Word 0 of a job in a worker's slot is its level, or kStaticJobs: the records
// [word 1, word 2) of the static queue that starts at record (or, strided, at
// worker) word 4 | word 5 << 32; or kNoJob: the request was not taken.
// Every answer, a refusal too, writes all kJobWords words with the request's
// tag, and none is taken before all of them carry it.  So one writer at a time
// has a worker's slot, all its words carry the tag of the request before (none
// at first: the init kernel clears the slots), and a partly written answer
// never matches, although tags repeat after 255 requests and 2^24 launches.
constexpr int32_t kStaticJobs = 0x100;
constexpr int32_t kNoJob = 0x200;
// a worker's seq-th request of a launch; never 0, and never the one before's
constexpr uint32_t request_tag(uint32_t epoch, uint32_t seq) { return (epoch << 8) | (seq % 255u + 1); }
constexpr uint64_t slot_word(uint32_t tag, int32_t value) { return ((uint64_t)tag << 32) | (uint32_t)value; }
constexpr bool slot_word_of(uint64_t word, uint32_t tag) { return (uint32_t)(word >> 32) == tag; }
constexpr int32_t refusal_value(int word) { return word == 0 ? kNoJob : 0; }
constexpr int kRefusalWords = kJobWords;
// A block's mailbox, a line: kMailSlots words that hold 0 (open), a request
// (asking worker + 1, its tag in the high half) or kMailIdle (no worker of the
// block has work); word kMailOver is the epoch of a launch that is over.
constexpr int kMailStride = 16;
constexpr int kMailSlots = 8;
constexpr int kMailOver = 8;
// words kMailPub..: which publication of its root's rows each worker's arena
// holds (blocks of at most kMailPubs workers)
constexpr int kMailPub = 9;
constexpr int kMailPubs = kMailStride - kMailPub;
constexpr unsigned long long kMailIdle = 0xffffffffull;
// The static scratch holds a launch's mailboxes and, after them, job slots in
// this many lines: a slot for every worker of a default launch, whose arenas
// (4,864 B at least) limit them to 13,400 in at most 2,048 blocks.  Of larger
// grids that a caller asks for the last workers never ask for work.
constexpr int kScratchLines = 16384;
static_assert(sizeof(Job) == kMailStride * 8, "a slot and a mailbox are a line each");
constexpr int scratch_slots(int workers, int blocks) { return std::min(workers, kScratchLines - blocks); }

// One counting query of a launch.  A single-graph call has one; a batch
// has one per (graph, pattern, k).
struct QueryDesc {
    int32_t K;
    int32_t motif;
    int32_t ncls;
    int32_t graph;                    // graph index in a batch (latency grouping)
    const uint16_t *lut;              // quick code -> class (motif)
    unsigned long long *out;          // clique: out[0]; motif: out[0 .. ncls)
    unsigned long long *done_ticks;   // nullable: wall clock of the query's last job end
};

struct EnumParams {
    // graph: symmetric CSR in degree-rank ids (a batch concatenates its graphs,
    // each relabelled inside its own id range); ostart[v] = first index of
    // N(v) above v
    const int64_t *off;
    const int32_t *adj;
    const int64_t *ostart;
    int32_t n;
    int32_t nq;                       // queries
    const QueryDesc *qd;
    int32_t kmax;                     // largest k of the queries (LDS record size)
    int32_t hist_slots;               // per-worker class counters (batch launches)
    int32_t nworkers;
    int32_t pad1;
    // static partition: worker w owns records sq_jobs[4*sq_off[w] .. 4*sq_off[w+1]):
    //   (root, lo, hi, q)   children [lo, hi) of root (q = query), or
    //   (r0, -1, r1, q)     every root of [r0, r1), all children
    // sq_jobs == nullptr: the strided partition of one query, with no arrays:
    // worker w's j-th job is root r = n-1 - (w + j*nworkers) as the range
    // (r, -1, r+1, 0) -- the reference's v -> warp v % W deal, heaviest
    // (highest degree rank) first
    const int64_t *sq_off;
    const int32_t *sq_jobs;
    int32_t *sq_cur;
    // a slot per worker for the jobs it is given (workers past q_cap never
    // ask), and a mailbox per block
    Job *q;
    uint32_t q_cap;
    int32_t pad2;
    unsigned long long *mail;
    const int32_t *epoch;             // launch epoch in device memory (set by the init kernel)
    unsigned long long *start_ticks;  // wall clock of the first block start
    SchedCounters *sc;
    // per-worker stacks: LDS slice of lds_per_worker bytes, then global arena
    char *arena;
    int64_t arena_per_worker;
    int32_t lds_per_worker;
    int32_t pad3;
    unsigned long long *root_cost;    // nullable, per vertex
    unsigned long long *root_count;   // nullable
    int32_t steal, steal_min, bitmap, pad4;
    uint64_t poll_ticks;              // wall-clock ticks between a worker's looks at its mailbox
    uint64_t watchdog_ticks;          // wall-clock ticks
    // local bitmaps prebuilt for some roots (cliques, k = 4..6): pre_roots
    // ascending (npre entries), root pre_roots[i]'s rows (d x NW uint64) and
    // out-degrees (d int32) at pre + pre_offs[i]
    const int32_t *pre_roots;
    const int64_t *pre_offs;
    const char *pre;
    // per prebuilt root: the next child its shared-cursor jobs claim (zeroed
    // before each launch); a static job (root, -2, P, q) is one of the P
    // jobs that share root's cursor
    int32_t *pre_cursor;
    int32_t npre;
    // workers per static queue (0 or 1: one queue per worker): worker w
    // claims from queue w / q_group of the (nworkers + q_group - 1) / q_group
    // queues
    int32_t q_group;
    // copies of a single query's results that the blocks add to (summed by
    // the host), and the words from one copy to the next
    int32_t res_copies, res_stride;
    int32_t pad6;
};
// One copy per block, 32 at most, in at most 8 KB unless one copy is larger.
inline int result_stride(size_t nres) { return (int)((nres + 15) & ~(size_t)15); }
inline int result_copies(size_t nres) { return std::max(1, std::min(32, 1024 / result_stride(nres))); }

// A static or donated job's query word: bits 0..15 the query index, bits
// 16..23 the job's own donation threshold (0: the launch's steal_min).
constexpr int kQueryBits = 16;
constexpr int job_query(int32_t q) { return q & ((1 << kQueryBits) - 1); }
constexpr int job_steal_min(int32_t q) { return (q >> kQueryBits) & 0xff; }
constexpr int32_t make_job_query(int q, int steal_min) { return q | (steal_min << kQueryBits); }

// kernels (enum_kernel.hip)
// mode: 0 cliques, 1 motifs, 2 motifs of sizes 5 and 6 (a motif kernel budgeted
// for more waves per SIMD: 6, 4 in mode 1).  Size 7's class counters and fixed
// leaf part leave a worker at 6 waves 800 B for the leaf's table, less than the
// smallest one, so every table was built in memory; at 4 waves it has 4 KB
// (Barabasi-Albert 600 of 3 edges a vertex, full grid, 48.9 -> 42.2 ms; Chung-Lu
// 3,000 of 4,000 edges 13.6 -> 11.7, 8,000 of 10,000 28.9 -> 25.5).  Size 6 has a
// 2 KB table at 6 waves and stays there: Barabasi-Albert 1,500 19.9 ms, 22.4 at 4;
// Chung-Lu 12,000 8.6, 9.2; light ones the other way round, Chung-Lu 1,000 1.37, 1.12.
inline int launch_mode(bool motif, int K) { return !motif ? 0 : K == 5 || K == 6 ? 2 : 1; }
// The motif leaf's LDS without its table, per worker of W lanes: recs u64[W] |
// bits u64[kLeafCap / 64 + 4] | qs u64[npm] | n u32[npm] | e u32[copies][npm * npm]
// (k = 7: [npm (npm + 1) / 2]), npm = 2^(K-2) mask values.  A motif launch gives
// each worker at least this.
constexpr int kLeafCap = 2048;  // stream positions per chunk
// A leaf node's edges are counted in 32 bits: where its table has fewer than
// 2^kLeafWideBits slots its elements have fewer than 2^32 pairs; of a wider node
// the sums go to the 64-bit class counters after every kLeafFlush elements, whose
// out-lists have fewer than 2^32 entries together (with ids in degree order an
// out-degree is at most sqrt(2E): 2^22 from 2^43 edges on).
constexpr int kLeafWideBits = 13;
constexpr int kLeafFlush = 1024;
constexpr int leaf_copies(int K) { return K <= 4 ? 8 : K == 5 ? 2 : 1; }
constexpr int motif_leaf_fixed(int W, int K) {
    return (W * 8 + kLeafCap / 8 + 32 + (1 << (K - 2)) * 12 +
            (K <= 6 ? leaf_copies(K) * (4 << (2 * (K - 2))) : (1 << (K - 2)) * ((1 << (K - 2)) + 1) * 2) + 15) & ~15;
}
// The leaf's table in the arena, where the LDS slice does not hold it: 2^bits
// slots of 4 B for `tot` elements, between 1/3 and 2/3 full (512 slots at least).
constexpr int leaf_table_bits(int64_t tot) {
    int b = 9;
    while (((int64_t)1 << b) < tot + tot / 2) b++;
    return b;
}
constexpr int64_t leaf_table_bytes(int64_t tot) { return (int64_t)4 << leaf_table_bits(tot); }
constexpr int kLeafTableMin = 1024;  // the smallest table in LDS
size_t enum_lds_bytes(int vwave, int threads, int kmax, int ncls_single, int hist_slots, int lds_per_worker);
int enum_occupancy(int vwave, int mode, int threads, size_t lds, int *blocks_per_cu);
int enum_launch(const EnumParams &p, int mode, int vwave, int blocks, int threads, size_t lds,
                void *stream);
// resets the scheduler state of a launch (graph-capturable: kernels only)
int enum_init_launch(const EnumParams &p, unsigned long long njobs, int32_t *epoch, unsigned long long *results,
                     size_t nresults, unsigned long long *done_ticks, int nq, int launch_blocks, void *stream);
int fill_u32_launch(void *ptr, uint32_t value, size_t count, void *stream);
// builds the local bitmaps of p.pre_roots into p.pre (one block per root)
int prebuild_launch(const EnumParams &p, void *stream);
// bytes of a prebuilt bitmap of a root with out-degree d (0: not on the bitmap path)
constexpr int64_t prebuilt_bytes(int32_t d) {
    const int nw = d <= 64 ? 1 : d <= 128 ? 2 : d <= 256 ? 4 : 0;
    return nw ? (((int64_t)d * nw * 8 + (int64_t)d * 4 + 15) & ~(int64_t)15) : 0;
}

// step-API state kernels (dfs_kernels.hip)
struct DfsMove {  // a job moved to another worker's queue
    int64_t slot;
    uint64_t ind;
    int32_t level;
    int32_t id[DM_DFS_MAXK];
    int32_t pad;
};
int dfs_reset_launch(const dm_dfs_data &d, const int32_t *roots, int nroots, void *stream);
int dfs_gather_launch(const dm_dfs_data &d, const int64_t *at, int32_t *out, void *stream);
int dfs_scatter_launch(const dm_dfs_data &d, const DfsMove *mv, int n, void *stream);

}  // namespace dm

#endif
