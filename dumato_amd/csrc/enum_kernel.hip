// DFS-wide subgraph enumeration on gfx950: k-clique counting and k-motif
// histograms.
//
// Reference semantics (what is computed):
//   clique  src/main/clique_PA.cu:9-32 with extend_clique / forward / backward /
//           aggregate_counter (src/main/DuMatoGPU.cu:1194-1220, 836-844, 745-750,
//           1769-1771): C_{l+1} = N+(last) & C_l, the last level adds |C|.
//   motif   src/main/motifs_DM_WCLB.cu:9-36 with extend(0,k) (:1702-1721),
//           canonicalFilter2 (:989-1012), forward_induce (:846-869) and
//           aggregate_pattern (:930-967).
//
// How it runs here (MI355X-first, not a translation):
//   * A worker is a virtual wave of W = 8/16/32/64 lanes of a wave64.  All
//     cross-lane steps (compaction, counts) use 64-bit ballots masked to the
//     worker's lanes, mbcnt-style prefix popcounts and shuffles of width W.
//   * Graph: symmetric CSR in degree-rank ids.  Cliques use the oriented view
//     N+(v) = the suffix of N(v) above v (ostart[v]), so "u > last" is the
//     degree orientation.
//   * Stack levels l = 0..K-3 live in a per-worker LDS slice and spill to a
//     per-worker global arena when a level does not fit.
//   * Motif extend keeps, per level, U_l = sorted union of N(id[0..l]) above
//     id[0], each element with the mask of the lists containing it (bit 7 =
//     passes the canonical rule).  The valid elements E_l are exactly the
//     reference's extensions after canonicalFilter2; the mask bits are the
//     reference's induction bits (forward_induce / aggregate_pattern).
//   * The last two levels are never materialised.  A leaf of a node of level
//     K-3 is an unordered pair of valid elements of U_{K-3}, or a valid
//     element and a new neighbour of it; its class follows from the two masks
//     and the pair's adjacency through the class table.  One pass over the
//     out-neighbours N+(x) of U_{K-3}'s elements finds the edges inside U_{K-3}
//     (motif_leaf); everything else is counted in closed form.
//   * Work: static per-worker queues of (root, lo, hi) jobs.  A worker that
//     runs out asks a random block through the block's mailbox; a busy worker
//     there answers with a share of its static jobs, or of the remaining
//     children of its job's lowest level (the reference's donate(),
//     src/main/DuMatoCPU.cu:463-539, done on the device instead of by the host).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <type_traits>

#include "internal.h"

namespace dm {

#define DEV __device__ __forceinline__

// Largest block (4 waves); a launch may use 1, 2 or 4 waves per block.
constexpr int kThreads = 256;
// Waves per SIMD each instantiation is compiled for: 3 (168 VGPRs) for the
// clique kernel, whose bitmap roots need the LDS of three blocks a CU, 4 (128
// VGPRs) for the full-wave motif kernel.  Motif sizes 5 and 6 get a second
// full-wave motif kernel at 6 waves (80 VGPRs; what is spilled belongs to the
// levels above the leaf, whose own registers fit).  k = 4 has larger tables,
// which 4 waves leave room for: at 5 / 6 waves Chung-Lu 18K 1.225 -> 1.193 /
// 1.199 ms, Barabasi-Albert 100K 4.82 -> 5.19 / 5.20.
template <int W, int MODE>
constexpr int min_waves() { return W == 64 && MODE == 1 ? 4 : 3; }
constexpr int kDeepMotifWaves = 6;

// ---------------------------------------------------------------------------
// virtual-wave primitives
template <int W>
struct Grp {
    int gl;  // lane within the worker
    int sh;  // first wave lane of the worker
    DEV Grp() {
        int l = __lane_id();
        gl = l & (W - 1);
        sh = l & ~(W - 1);
    }
    DEV uint64_t ballot(bool p) const {
        uint64_t b = __ballot(p);
        if constexpr (W == 64) return b;
        else return (b >> sh) & ((1ull << W) - 1);
    }
    DEV int below(uint64_t m) const { return __popcll(m & ((1ull << gl) - 1)); }
    DEV int isum(int x) const {
#pragma unroll
        for (int o = W / 2; o > 0; o >>= 1) x += __shfl_xor(x, o, W);
        return x;
    }
    DEV unsigned long long lsum(unsigned long long x) const {
#pragma unroll
        for (int o = W / 2; o > 0; o >>= 1) x += __shfl_xor(x, o, W);
        return x;
    }
    // src is the same for every lane of the worker at every call site; for a
    // full wave the value is then read into a scalar register
    DEV int bcast(int x, int src) const {
        if constexpr (W == 64) return __builtin_amdgcn_readlane(x, src);
        else return __shfl(x, src, W);
    }
    DEV int iscan(int x) const {  // inclusive prefix sum over the worker's lanes
        if constexpr (W == 64) {
            // within rows of 16 lanes (row_shr 1, 2, 4, 8), then the row ends
            // added to the rows above them (row_bcast 15, 31)
            x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);
            x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);
            x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);
            x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);
            x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);
            x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
            return x;
        } else {
#pragma unroll
            for (int o = 1; o < W; o <<= 1) {
                int y = __shfl_up(x, o, W);
                if (gl >= o) x += y;
            }
            return x;
        }
    }
    DEV unsigned long long bcast64(unsigned long long x, int src) const {
        if constexpr (W == 64) {
            const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, src);
            const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), src);
            return ((unsigned long long)hi << 32) | lo;
        } else {
            return __shfl(x, src, W);
        }
    }
};

template <int W>
DEV int uni(int x) {
    if constexpr (W == 64) return __builtin_amdgcn_readfirstlane(x);
    else return x;
}

// The same for 64-bit values and pointers: what a worker's lanes share and
// read from memory stays in scalar registers for a full wave.
template <int W, class T>
DEV T unil(T x) {
    if constexpr (W == 64) {
        const uint64_t v = (uint64_t)x;
        const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
        return (T)(((uint64_t)hi << 32) | lo);
    } else {
        return x;
    }
}

DEV void wsync() { __threadfence_block(); }

// Orders a wave's LDS accesses (executed in order per wave) for the compiler.
DEV void lsync() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

// LDS words addressed as such (ds instructions; a generic pointer takes flat ones)
using lds_u8 = __attribute__((address_space(3))) uint8_t;
using lds_u32 = __attribute__((address_space(3))) uint32_t;
using lds_u64 = __attribute__((address_space(3))) uint64_t;
// global memory addressed as such: a generic pointer takes flat loads, which
// the LDS counter waits for too, so LDS reads between them end their overlap
using glb_i32 = const __attribute__((address_space(1))) int32_t;
using glb_i64 = const __attribute__((address_space(1))) int64_t;
using glb_u8 = const __attribute__((address_space(1))) uint8_t;
using glb_u16 = const __attribute__((address_space(1))) uint16_t;
using glb_u32 = __attribute__((address_space(1))) uint32_t;
using glb_u64 = __attribute__((address_space(1))) uint64_t;
// waits until the wave's memory operations have been performed
DEV void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// The atomic that returned x has been performed before any access that
// follows in the program (its result is waited for here).
template <class T>
DEV void landed(T &x) { asm volatile("" : "+v"(x)::"memory"); }
// LDS address of a generic pointer into LDS
DEV uint32_t lds_at(const void *a) { return (uint32_t)(uintptr_t)(lds_u32 *)a; }
template <class P, class T>
DEV void ladd(P *a, T v) {
    (void)__hip_atomic_fetch_add(a, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}
// to LDS words that other waves of the block add to as well
template <class P, class T>
DEV void badd(P *a, T v) {
    (void)__hip_atomic_fetch_add(a, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
template <class P>
DEV void lor(P *a, uint64_t v) {
    (void)__hip_atomic_fetch_or(a, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}
template <class P>
DEV int lower_bound(P a, int n, int32_t x) {
    int lo = 0, hi = n;
    while (lo < hi) {
        int mid = (lo + hi) >> 1;
        if (a[mid] < x) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

DEV int quick_off(int s) { return ((s - 2) * (s + 1)) >> 1; }

DEV uint64_t now_ticks() { return wall_clock64(); }

// ---------------------------------------------------------------------------
// per-worker state in LDS
struct Lvl {
    int32_t *uid;     // U_l ids (motif) / C_l (clique)
    uint8_t *upm;     // U_l masks; nullptr = level 0 (mask 1, valid)
    int32_t *eid;     // E_l ids (motif)
    uint8_t *epm;     // E_l masks; nullptr = level 0
    char *mark_lds;   // allocator tops before this level's buffers
    char *mark_glb;
    uint64_t ind;     // induction (quick bits) of the prefix id[0..l]
    int32_t nu, ne;   // |U_l|, |E_l|
    int32_t cur, end; // children cursor / end
    int32_t vtx;      // vertex placed at level l
    int32_t sdeg;     // sum of degrees of id[0..l] (algorithmic bytes)
};

// Per-worker LDS record, at fixed offsets from one base so that a worker
// holds a single pointer to it: uint64 st[kStats] (the worker's statistics),
// int32 jid[kJobIds] (the prefix of the current job), then Lvl lv[nlv], nlv =
// max(K-2, 1).
enum { kStBusy, kStJobs, kStFirst, kStStatic, kStLast, kStQCount, kStDonated, kStT0, kStJobMax, kStats };
constexpr int kJidOff = 80;
constexpr int kLvOff = (kJidOff + kJobIds * 4 + 15) & ~15;
static_assert(kStats * 8 <= kJidOff, "worker statistics overlap the job prefix");
struct WorkerLDS {
    char *b;
    DEV unsigned long long *st() const { return (unsigned long long *)b; }
    DEV int32_t *jid() const { return (int32_t *)(b + kJidOff); }
    DEV Lvl *lv() const { return (Lvl *)(b + kLvOff); }
};
DEV int nlevels(int K) { return K - 2 > 1 ? K - 2 : 1; }
__host__ __device__ inline size_t worker_lds_bytes(int K) {
    int nlv = K - 2 > 1 ? K - 2 : 1;
    return ((size_t)kLvOff + (size_t)nlv * sizeof(Lvl) + 15) & ~(size_t)15;
}
DEV WorkerLDS worker_lds(char *base, int K) {
    (void)K;
    WorkerLDS w;
    w.b = base;
    return w;
}

// ---------------------------------------------------------------------------
// The motif leaf node: a node of level K-3 with prefix id[0..K-3], U = U_{K-3},
// npm = 2^(K-2) mask values, E = the valid elements of U.  Each of its
// K-subgraphs is the prefix plus either two elements of E, or an element of E
// and one of its neighbours above id[0] outside U; the class depends on the
// two masks and the adjacency alone, not on which is the child and which the
// leaf.  So the counts per class need only, per mask i:
//   n_i   elements of E with mask i,
//   q_i   sum of |N(x) above id[0]| over them,
//   e_ij  edges between E-elements of masks i and j (e_i0: to U \ E),
// as pairs(i, j) = e_ij adjacent, n_i n_j - e_ij (C(n_i, 2) - e_ii) not, and
// new(i) = q_i - sum_j e_ij - e_ii.
// Every edge {x, y} inside U, x < y, is found once, from N+(x): the work is
// sum over U of |N+(x)| membership tests of U, not sum over E of |N(x)|.  A
// degree-ordered N+ is short where N is long, so beside hubs this is 3-5x
// fewer (over the leaf nodes of Chung-Lu 18K k = 4: 305 M against 1,116 M;
// Barabasi-Albert 100K k = 4: 678 M against 3,557 M).  Calls against the
// leaf that streamed every child's N(c): Chung-Lu 18K k = 4 4.76 -> 2.12 ms,
// Barabasi-Albert 100K k = 4 16.5 -> 5.9 ms, 12K k = 5 167 -> 43 ms; with the
// steps described at their places now 1.25, 4.79 and 34 ms.
//
// U is held in a hash table for these tests: buckets of two 32-bit slots, two
// buckets per element, so a test is two 8-byte LDS reads and no loop.  With h =
// id * odd (a bijection of 32 bits) the top b bits of h name the first bucket;
// a slot holds the other 32 - b bits in place (h << b), whether it sits in its
// second bucket (the first one xor the next b bits of h), and its 6-bit code
// ^ 63 (code: its mask if valid, 32 if not; 63 marks an empty slot), which
// fits from b = 7 on.  The table is in LDS, or in the worker's arena where U is
// too large for that.
constexpr uint32_t kEmpty = 63;

struct LeafSum {
    unsigned long long cnt, bytes;  // this lane's share
    int big;                        // > 0: needs a table of 2^big slots in memory
};

// The table's b and hash split; slots are reached through lds (LDS) or glb.
template <bool LDS>
struct LeafTab {
    using P32 = std::conditional_t<LDS, lds_u32 *, glb_u32 *>;
    using P64 = std::conditional_t<LDS, lds_u64 *, glb_u64 *>;
    P32 t;
    int b, sh;     // 2^b buckets, sh = 32 - b
    uint32_t mul;  // odd
    // code of x (0: not in U)
    DEV int find(int32_t x) const {
        const uint32_t h = (uint32_t)x * mul, b1 = h >> sh, k1 = h << b, b2 = b1 ^ (k1 >> sh);
        const uint64_t s1 = ((P64)t)[b1], s2 = ((P64)t)[b2];
        const uint32_t a0 = (uint32_t)s1 ^ k1, a1 = (uint32_t)(s1 >> 32) ^ k1;
        const uint32_t a2 = (uint32_t)s2 ^ (k1 | 64), a3 = (uint32_t)(s2 >> 32) ^ (k1 | 64);
        const uint32_t m0 = a0 < a1 ? a0 : a1, m1 = a2 < a3 ? a2 : a3;
        const uint32_t m = m0 < m1 ? m0 : m1;
        return m < 63 ? (int)(m ^ 63) : 0;
    }
    // where x lies, of a table whose codes are all 1 (-1: not in it)
    DEV int slot(int32_t x) const {
        const uint32_t h = (uint32_t)x * mul, b1 = h >> sh, k1 = h << b, b2 = b1 ^ (k1 >> sh);
        const uint64_t s1 = ((P64)t)[b1], s2 = ((P64)t)[b2];
        const uint32_t w = k1 | (1 ^ 63);
        int at = -1;
        at = (uint32_t)s1 == w ? 2 * (int)b1 : at;
        at = (uint32_t)(s1 >> 32) == w ? 2 * (int)b1 + 1 : at;
        at = (uint32_t)s2 == (w | 64) ? 2 * (int)b2 : at;
        at = (uint32_t)(s2 >> 32) == (w | 64) ? 2 * (int)b2 + 1 : at;
        return at;
    }
    // adds mask bit `bit` to x, which is in U, if it is valid
    DEV void mark(int32_t x, uint32_t bit) const {
        const uint32_t h = (uint32_t)x * mul, b1 = h >> sh, k1 = h << b, b2 = b1 ^ (k1 >> sh);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            P32 s = t + 2 * (i < 2 ? b1 : b2) + (i & 1);
            const uint32_t v = *s, a = v ^ (k1 | (i < 2 ? 0 : 64));
            if (a < 63 && a != (32 ^ 63)) *s = v ^ bit;
        }
    }
    // inserts x (not present); false when no slot was found.  Every step is one
    // exchange: what it displaces goes to the bucket's other slot, what that
    // displaces to its own other bucket.  (At most 45% full, a wave needs 2-5
    // steps of 9 instructions; compare-and-swap probes of the four slots took
    // 70 instructions a round, 3 rounds a wave.)
    DEV bool insert(int32_t x, int code) const {
        const uint32_t h = (uint32_t)x * mul;
        uint32_t bk = h >> sh, v = (h << b) | (uint32_t)(code ^ 63);
        for (int it = 0; it < 256; it++) {
            v = __hip_atomic_exchange(t + 2 * bk + (it & 1), v, __ATOMIC_RELAXED, kScope);
            if (v == kEmpty) return true;
            if (it & 1) {
                bk ^= v >> sh;
                v ^= 64;
            }
        }
        return false;
    }
    static constexpr int kScope = LDS ? __HIP_MEMORY_SCOPE_WAVEFRONT : __HIP_MEMORY_SCOPE_AGENT;
    DEV static void sync() {
        if constexpr (LDS) lsync();
        else wsync();
    }
    // U of the leaf: the parent's list (masks pm, nullptr: all 1) with the
    // order rule x > c, then nc[0, q), whose new elements get mask newc
    template <int W>
    DEV bool build(const Grp<W> &g, glb_i32 *puid, glb_u8 *pupm, int pnu, int32_t c, glb_i32 *nc, int q,
                   int newc) const {
        using V4 = uint32_t __attribute__((ext_vector_type(4)));
        using P128 = std::conditional_t<LDS, __attribute__((address_space(3))) V4 *, __attribute__((address_space(1))) V4 *>;
        for (int j = g.gl; j < (1 << (b - 1)); j += W) ((P128)t)[j] = V4{kEmpty, kEmpty, kEmpty, kEmpty};
        sync();
        bool ok = true;
        for (int j = g.gl; j < pnu; j += W) {
            const int32_t x = puid[j];
            const int pm = pupm ? pupm[j] : 0x81;
            ok &= insert(x, (pm & 0x80) && x > c ? pm & 0x7f : 32);
        }
        sync();
        for (int j0 = 0; j0 < q; j0 += W) {
            const int j = j0 + g.gl;
            bool add = false;
            int32_t x = 0;
            if (j < q) {
                x = nc[j];
                add = pnu == 0 || find(x) == 0;
                if (!add) mark(x, (uint32_t)newc);
            }
            sync();
            if (add) ok &= insert(x, newc);
            sync();
        }
        return g.ballot(!ok) == 0;
    }
};

// Position of the first entry of a[0, n) not below x (ascending), by all the
// worker's lanes: each step narrows the range W-fold.
template <int W>
DEV int wave_lower_bound(const Grp<W> &g, glb_i32 *a, int n, int32_t x) {
    int lo = 0;
    while (n > 0) {
        const int st = (n + W - 1) / W;  // lane i looks at the end of piece i
        const int i = (g.gl + 1) * st - 1;
        const bool below = i < n && a[lo + i] < x;
        const int full = __popcll(g.ballot(below)) * st;  // pieces wholly below x
        if (st == 1) return lo + full;
        lo += full;
        n = n - full < st - 1 ? n - full : st - 1;
    }
    return lo;
}

// Entries of the ascending list a[0, n) below x: three probes a round, whose
// loads overlap, so half the dependent rounds of a binary search in the motif
// leaf (Barabasi-Albert 100K k = 4 4.88 -> 4.63 ms, Chung-Lu 18K k = 4 1.22 -> 1.20;
// keeping the counts of a parent's elements for all its leaves instead cost
// more than the searches: 5.03 and 1.25).
DEV int below4(glb_i32 *a, int n, int32_t x) {
    int lo = 0;
    while (n > 3) {
        const int s = n >> 2;
        const int32_t p = a[lo + s], q = a[lo + 2 * s], r = a[lo + 3 * s];
        const int c = (p < x ? 1 : 0) + (q < x ? 1 : 0) + (r < x ? 1 : 0);
        const int hi = c < 3 ? lo + (c + 1) * s : lo + n;
        lo = c ? lo + c * s + 1 : lo;
        n = hi - lo;
    }
    if (n > 0) {
        const int last = lo + n - 1;
        const int32_t p = a[lo], q = a[lo + 1 < last ? lo + 1 : last], r = a[last];
        lo += (p < x ? 1 : 0) + (n > 1 && q < x ? 1 : 0) + (n > 2 && r < x ? 1 : 0);
    }
    return lo;
}

// The lanes' lists (len entries at `list`) laid end to end, f(entry, tag of its
// list) called for every entry, W consecutive ones at a time, U of those steps'
// loads in flight (f(none, 0) past the lists' end).  recs: list address and
// tag, by list; bits: a set bit where a list starts, so the list of an entry is
// a popcount.  VALU-bound once the loads overlap: about 35 instructions a step
// with the table test, against 104 with generic pointers, 64-bit index
// arithmetic and a bounds check per step (with the insertions by exchange:
// Chung-Lu 18K k = 4 1.44 -> 1.26 ms, Barabasi-Albert 12K k = 5 38.8 -> 33.3 ms,
// triangles of R-MAT s18 1.63 -> 1.32 ms).  U = 4 in the motif leaf, whose
// registers allow no more, 8 in the clique kernel at 3 waves per SIMD
// (triangles of R-MAT s18 of edge factor 8 1.05 -> 1.00 ms).
template <int U, int W, class F>
DEV void stream_lists(const Grp<W> &g, lds_u64 *recs, lds_u64 *bits, glb_i32 *list, int len, int tag, int32_t none,
                      F f) {
    const uint64_t mx = g.ballot(len > 0);
    const int sc = g.iscan(len), pre = sc - len;
    const int T = g.bcast(sc, W - 1);
    // addresses have 48 bits (the first `pre` entries before a list may lie
    // outside the array: they are not read)
    if (len > 0) recs[g.below(mx)] = ((uint64_t)(list - pre) & 0xffffffffffffull) | ((uint64_t)tag << 56);
    for (int p0 = 0; p0 < T; p0 += kLeafCap) {
        const int pe = T - p0 < kLeafCap ? T : p0 + kLeafCap;
        for (int w = g.gl; w < kLeafCap / 64 + U; w += W) bits[w] = 0;
        lsync();
        if (len > 0 && pre >= p0 && pre < pe) lor(bits + ((pre - p0) >> 6), 1ull << ((pre - p0) & 63));
        // lists that started before this chunk
        int own0 = __popcll(g.ballot(len > 0 && pre < p0)) - 1;
        lsync();
        // U * W positions from t0; the last ones (full = false) may end early
        auto step = [&](int t0, auto full) {
            uint64_t rec[U], seg[U];
            int32_t ys[U];
            int tg[U];
#pragma unroll
            for (int u = 0; u < U; u++) seg[u] = bits[(t0 + u * W - p0) >> 6];
#pragma unroll
            for (int u = 0; u < U; u++) {
                if constexpr (W == 64) seg[u] = unil<W>(seg[u]);
                else seg[u] = (seg[u] >> ((t0 + u * W - p0) & 63)) & ((1ull << W) - 1);
                rec[u] = recs[own0 + __popcll(seg[u] & ((2ull << g.gl) - 1))];
                own0 += __popcll(seg[u]);
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int t = t0 + u * W + g.gl;
                tg[u] = (int)(rec[u] >> 56);
                glb_i32 *const a = (glb_i32 *)(rec[u] & 0xffffffffffffull) + t;
                if constexpr (full) {
                    ys[u] = *a;
                } else {
                    ys[u] = none;
                    if (t < pe) ys[u] = *a;
                    else tg[u] = 0;
                }
            }
#pragma unroll
            for (int u = 0; u < U; u++)
                if (full || t0 + u * W < pe) f(ys[u], tg[u]);
        };
        int t0 = p0;
        for (; t0 + U * W <= pe; t0 += U * W) step(t0, std::true_type{});
        if (t0 < pe) step(t0, std::false_type{});
        lsync();
    }
}

// The edges that a leaf node has counted so far in 32 bits (e at LDS address
// e_at, all copies) go to the class counters, whose sums wrap at 64 bits like the
// final ones: its part of the adjacent pairs, taken from the others and from the
// pairs with a new neighbour.  ind: the prefix's bits of the class table's index.
// Returns this lane's share of the leaves.
template <int W>
DEV unsigned long long leaf_flush(const Grp<W> &g, glb_u16 *lut, lds_u64 *shist, lds_u32 *e, uint64_t ind, int K) {
    const int npm = 1 << (K - 2), lw = K - 2, o2 = quick_off(K - 1);
    const bool sq = K <= 6;
    const int ne = sq ? npm * npm : npm * (npm + 1) / 2, copies = leaf_copies(K);
    unsigned long long leaves = 0;
    auto child = [&](int i) -> uint64_t { return K == 3 ? 0 : ind + ((uint64_t)i << quick_off(K - 2)); };
    for (int t = g.gl; t < ne; t += W) {
        uint64_t ee = 0;
        for (int k = 0; k < copies; k++) {
            ee += e[k * ne + t];
            e[k * ne + t] = 0;
        }
        if (!ee) continue;
        int i = t >> lw, j = t & (npm - 1);
        if (!sq) {
            for (i = 0; (i + 1) * (i + 2) / 2 <= t;) i++;
            j = t - i * (i + 1) / 2;
        }
        if (i < j) j = i, i = t & (npm - 1);
        if (!i) continue;
        if (j) {
            badd(shist + lut[child(i) + ((uint64_t)(j | npm) << o2)], ee);
            badd(shist + lut[child(i) + ((uint64_t)j << o2)], 0 - ee);
            badd(shist + lut[child(j) + ((uint64_t)npm << o2)], 0 - ee);
            leaves -= ee;
        }
        badd(shist + lut[child(i) + ((uint64_t)npm << o2)], 0 - ee);
        leaves -= ee;
    }
    lsync();
    return leaves;
}

// The counts of one leaf node, added to the class counters at LDS address shist_at.  (c, pmc):
// the child of the parent's list (puid, pupm, pnu) that makes the node, its
// mask; K = 3: the root alone, c = id[0], whose elements [lo, hi) are taken
// as children.  lds_at: motif_leaf_fixed bytes of LDS, then `space` bytes for the table;
// gtab: a table of 2^space slots in memory instead.  WIDE: such a node of many
// elements, whose edge counts are flushed now and then; a function of its own, as
// flushing in the one function cost the k = 5 kernel 3% (Barabasi-Albert 12K 33.1
// -> 34.0 ms), a call from there 20%.  Not inlined: the node's
// registers are then its own, not shared with the search around it.
template <int W, bool WIDE>
__device__ __attribute__((noinline)) LeafSum motif_leaf(const int64_t *off_, const int32_t *adj_, const int64_t *ostart_,
                                                        const uint16_t *lut_, const int32_t *puid_,
                                                        const uint8_t *pupm_, uint32_t shist_at, uint32_t lds_at,
                                                        uint32_t *gtab, uint64_t pind, int32_t v0, int K, int32_t c,
                                                        int pmc, int pnu, int psdeg, int lo, int hi, int space) {
    glb_i64 *const off = (glb_i64 *)unil<W>(off_), *const ostart = (glb_i64 *)unil<W>(ostart_);
    glb_i32 *const adj = (glb_i32 *)unil<W>(adj_), *const puid = (glb_i32 *)unil<W>(puid_);
    glb_u16 *const lut = (glb_u16 *)unil<W>(lut_);
    glb_u8 *const pupm = (glb_u8 *)unil<W>(pupm_);
    gtab = unil<W>(gtab), pind = unil<W>(pind);
    v0 = uni<W>(v0), K = uni<W>(K), c = uni<W>(c), pmc = uni<W>(pmc), pnu = uni<W>(pnu), psdeg = uni<W>(psdeg);
    lo = uni<W>(lo), hi = uni<W>(hi), space = uni<W>(space);
    lds_u64 *const lds = (lds_u64 *)(uintptr_t)(uint32_t)uni<W>((int)lds_at);
    lds_u64 *const shist = (lds_u64 *)(uintptr_t)(uint32_t)uni<W>((int)shist_at);
    Grp<W> g;
    const bool root = K == 3;
    const int npm = 1 << (K - 2), newc = npm >> 1;  // newc: mask of an element only N(c) holds
    const int64_t cb = unil<W>(off[c]), ce = unil<W>(off[c + 1]);
    const int sdeg = psdeg + (int)(ce - cb);
    const int64_t cs = root ? unil<W>(ostart[c]) : cb + wave_lower_bound(g, adj + cb, (int)(ce - cb), v0 + 1);
    glb_i32 *const nc = adj + cs;  // N(c) above id[0]
    const int q = (int)(ce - cs);
    const int tot = pnu + q;  // elements of U, common ones twice
    LeafSum r{0, 0, 0};

    lds_u64 *recs = lds;
    lds_u64 *bits = recs + W;
    lds_u64 *qs = bits + kLeafCap / 64 + 4;
    lds_u32 *nm = (lds_u32 *)(qs + npm);
    lds_u32 *e = nm + npm;
    // counters of a pair: npm x npm, several copies, up to k = 6; triangular at 7
    const bool sq = K <= 6;
    const int ne = sq ? npm * npm : npm * (npm + 1) / 2, copies = leaf_copies(K);
    LeafTab<true> tl;
    LeafTab<false> tg;
    if (!WIDE && !gtab) {
        // at most 45% full while the space allows it
        int b = 7;
        while ((16 << b) <= space && 9 * (2 << b) < 20 * tot) b++;
        tl.t = (lds_u32 *)(lds + motif_leaf_fixed(W, K) / 8);
        tl.b = b, tl.sh = 32 - b;
        tl.mul = 0x9E3779B1u;
        // up to 6/7 full; a failed insertion is rare from there on down
        if ((8 << b) > space || 7 * tot > 6 * (2 << b) || !tl.build(g, puid, pupm, pnu, c, nc, q, newc)) {
            r.big = leaf_table_bits(tot);
            return r;
        }
    } else {
        tg.t = (glb_u32 *)gtab;
        tg.b = space - 1, tg.sh = 33 - space;
        tg.mul = 0x9E3779B1u;
        for (int tries = 0; !tg.build(g, puid, pupm, pnu, c, nc, q, newc); tries++) {
            if (tries == 7) {
                r.big = -1;
                return r;
            }
            tg.mul = tg.mul * 0x2545F491u + 2;  // another odd multiplier
        }
    }
    for (int j = g.gl; j < ne * copies / 2; j += W) ((lds_u64 *)e)[j] = 0;
    for (int j = g.gl; j < npm; j += W) nm[j] = 0, qs[j] = 0;
    lsync();

    // elements of U, W at a time: n_i and q_i, then their out-lists (v0, in
    // place of an entry past their end, is never in U)
    uint32_t nnew = 0, enew = 0;  // class newc / (newc, newc), counted in registers
    const int lw = K - 2;
    unsigned long long qnew = 0, by = 0, leaves = 0, rpairs = 0;
    lds_u32 *const ecopy = e + (g.gl & (copies - 1)) * ne;
    const uint64_t ind = root ? 0 : pind + (K - 3 >= 2 ? (uint64_t)pmc << quick_off(K - 3) : 0);
    auto scan = [&](const auto &tab) {
        for (int j0 = 0; j0 < tot; j0 += W) {
        if (WIDE && j0 && j0 % kLeafFlush == 0) {
            if (enew) ladd(e + (sq ? (newc << lw) + newc : newc * (newc + 1) / 2 + newc), enew);
            enew = 0;
            lsync();
            leaves += leaf_flush(g, lut, shist, e, ind, K);
        }
        if (WIDE && root && (j0 + W <= lo || j0 >= hi)) continue;
        const int j = j0 + g.gl;
        int32_t x = 0;
        int code = 0;
        if (j < tot) {
            x = j < pnu ? puid[j] : nc[j - pnu];
            code = tab.find(x);
            // a neighbour of c that an earlier list holds too is visited in
            // the parent's list
            if (j >= pnu && code != newc) code = 0;
            if (root && (j < lo || j >= hi)) code = 0;
        }
        const int cx = code & 31;
        int len = 0;
        int64_t os = 0;
        if (code) {
            const int64_t b = off[x], en = off[x + 1];
            os = ostart[x];
            len = (int)(en - os);
            if (cx) {
                const int up = (int)(en - b) - below4(adj + b, (int)(os - b), v0 + 1);
                by += (unsigned long long)(sdeg + (int)(en - b));
                if (cx == newc) {
                    nnew++;
                    qnew += (unsigned long long)up;
                } else {
                    ladd(nm + cx, 1u);
                    ladd(qs + cx, (uint64_t)up);
                }
                if (root) rpairs += (unsigned long long)(tot - 1 - j);
            }
        }
        stream_lists<4>(g, recs, bits, adj + os, len, cx, v0, [&](int32_t y, int mx) {
            const int cd = tab.find(y);
            const bool nn = mx == newc && cd == newc;
            enew += nn ? 1u : 0u;
            if (cd && !nn) {
                const int cy = cd & 31;
                if (sq) {
                    ladd(ecopy + ((mx << lw) + cy), 1u);
                } else {
                    const int a = mx > cy ? mx : cy, z = mx > cy ? cy : mx;
                    ladd(ecopy + (__umul24(a, a + 1) >> 1) + z, 1u);
                }
            }
        });
        }
    };
    if (WIDE || gtab) scan(tg);
    else scan(tl);
    if (nnew) ladd(nm + newc, nnew);
    if (qnew) ladd(qs + newc, (uint64_t)qnew);
    if (enew) ladd(e + (sq ? (newc << lw) + newc : newc * (newc + 1) / 2 + newc), enew);
    lsync();
    if (copies > 1) {
        for (int t = g.gl; t < ne; t += W) {
            uint32_t sum = 0;
            for (int k = 0; k < copies; k++) sum += e[k * ne + t];
            e[t] = sum;
        }
        lsync();
    }
    // edges between masks i >= j (0: U \ E); the lut index of the prefix
    // id[0..K-3] and its child's mask i
    auto edges = [&](int i, int j) -> uint64_t {
        if (!sq) return e[i * (i + 1) / 2 + j];
        return i == j ? (uint64_t)e[(i << lw) + i] : (uint64_t)e[(i << lw) + j] + e[(j << lw) + i];
    };
    auto child = [&](int i) -> uint64_t { return root ? 0 : ind + ((uint64_t)i << quick_off(K - 2)); };
    const int o2 = quick_off(K - 1);
    if (root) rpairs = g.lsum(rpairs);
    auto pair = [&](int i, int j) {
        const uint64_t ni = nm[i], nj = nm[j];
        const uint64_t pr = root ? rpairs : i == j ? ni * (ni - 1) / 2 : ni * nj;
        if (pr == 0) return;
        const uint64_t ee = edges(i, j);
        if (ee) badd(shist + lut[child(i) + ((uint64_t)(j | npm) << o2)], ee);
        if (pr != ee) badd(shist + lut[child(i) + ((uint64_t)j << o2)], pr - ee);
        leaves += pr;
    };
    if (W < 64 && npm > W) {
        // few lanes for many masks, most of them without elements (Chung-Lu 1,000
        // of 1,500 edges, k = 7: 8 lanes 27.2 -> 19.5 ms, 16 lanes 12.4 -> 9.2)
        uint32_t some = 0;
        for (int k = 0; k < npm; k += W) some |= (uint32_t)g.ballot(nm[k + g.gl] != 0) << k;
        for (; some; some &= some - 1) {
            const int i = __builtin_ctz(some);
            for (int j = 1 + g.gl; j <= i; j += W) pair(i, j);
        }
    } else {
        for (int t = g.gl; t < npm * npm; t += W) {
            const int i = t >> (K - 2), j = t & (npm - 1);
            if (j != 0 && i >= j) pair(i, j);
        }
    }
    for (int i = 1 + g.gl; i < npm; i += W) {
        uint64_t nw = qs[i];
        if (!nm[i]) continue;
        for (int j = 0; j < npm; j++) nw -= i == j ? 2 * edges(i, i) : i > j ? edges(i, j) : edges(j, i);
        if (nw) badd(shist + lut[child(i) + ((uint64_t)npm << o2)], nw);
        leaves += nw;
    }
    lsync();
    r.cnt = leaves;
    // the node's own bytes (at k = 3 the root's are counted by the caller)
    r.bytes = 4ull * by + 4ull * (K - 1) * leaves + (!root && g.gl == 0 ? 4ull * (unsigned long long)sdeg : 0ull);
    return r;
}

// Triangles of root v0 (k = 3): the edges {u, y} inside N+(v0), u one of its
// children [lo, hi), found from the out-lists N+(u) laid end to end over the
// lanes and tested against a table of N+(v0), as in the motif leaf.  first:
// the call that builds the table (the root's later calls find it in place).
// Bound by the table reads (R-MAT s18 of edge factor 16: 659 M tests a call,
// 83 M triangles; one child at a time, each entry searched in the longer list:
// 5.19 -> 1.81 ms).  lds_at: recs u64[W] | bits u64[kLeafCap / 64 + 8] | table.
constexpr int kTriFixed = 64 * 8 + kLeafCap / 8 + 64;
// (the triangles' own: at 8 lanes the table fits the default slice of 1,456 B only
// so; R-MAT s15 of edge factor 8, k = 3, 1.34 -> 0.20 ms)
constexpr int tri_fixed(int W) { return kTriFixed - (64 - W) * 8; }
struct TriSum {
    unsigned long long cnt, by;  // this lane's share; by: out-degrees of the children
};
template <int W>
__device__ __attribute__((noinline)) TriSum triangles(const int64_t *off_, const int32_t *adj_,
                                                      const int64_t *ostart_, uint32_t at, int b, int32_t v0, int lo, int hi, bool first,
                                                      bool &ok) {
    glb_i64 *const off = (glb_i64 *)unil<W>(off_), *const ostart = (glb_i64 *)unil<W>(ostart_);
    glb_i32 *const adj = (glb_i32 *)unil<W>(adj_);
    b = uni<W>(b), v0 = uni<W>(v0), lo = uni<W>(lo), hi = uni<W>(hi);
    const Grp<W> g;
    lds_u64 *const recs = (lds_u64 *)(uintptr_t)(uint32_t)uni<W>((int)at);
    lds_u64 *const bits = recs + W;
    LeafTab<true> tab;
    tab.t = (lds_u32 *)(recs + tri_fixed(W) / 8);
    tab.b = b, tab.sh = 32 - b, tab.mul = 0x9E3779B1u;
    const int64_t ls = unil<W>(ostart[v0]);
    glb_i32 *const L = adj + ls;
    TriSum r{0, 0};
    ok = true;
    if (first) {
        const int d = (int)(unil<W>(off[v0 + 1]) - ls);
        ok = tab.build(g, L, (glb_u8 *)nullptr, 0, v0, L, d, 1);
        if (!ok) return r;
    }
    for (int j0 = lo; j0 < hi; j0 += W) {
        const int j = j0 + g.gl;
        int len = 0;
        int64_t os = 0;
        if (j < hi) {
            const int32_t u = L[j];
            os = ostart[u];
            len = (int)(off[u + 1] - os);
            r.by += (unsigned long long)len;
        }
        uint32_t found = 0;
        stream_lists<8>(g, recs, bits, adj + os, len, 0, v0, [&](int32_t y, int) { found += tab.find(y) ? 1 : 0; });
        r.cnt += found;
    }
    return r;
}

// ---------------------------------------------------------------------------
// Cliques of a batch of second-level pairs of a root's local bitmap (rows[i *
// NW + w] bit b: L[64w+b] in N+(L[i]), L = N+(root)): pairs 0..P-1, pair t
// belonging to child cur + a with pre[a] <= t < pre[a+1] and being its
// (t - pre[a])-th candidate.  The loops visit exactly the DFS children of
// every node above the last level, so the algorithmic bytes (sum of
// out-degrees of the children of nodes with 1..k-2 vertices) are summed in the
// same loops from dp[] = out-degrees.
//
// K <= 5: a lane per pair (i, j) takes S2 = row i & row j and, at K = 5, counts
// the edges of S2 bit by bit.  K >= 6: candidate sets are expanded breadth
// first, sw at a time, level by level: a stage holds up to sw sets and the
// prefix sums of their sizes; the lanes stride over the elements of a stage's
// sets, one level finer than a lane per set, whose cost (|S| x |S & row|)
// varies too much across a wave.  Stage K-4's elements are counted directly
// (the edges of set & row); earlier stages fill the next one and are resumed
// when it is done.  Bound by LDS reads of rows and by divergence in the bit
// loops.  (K = 7 on an 8,192-vertex R-MAT: list intersection, one child at a
// time, 174 ms; stages 1.44 ms.  R-MAT s17 K = 5 1.52 -> 1.24 ms from reading
// the rows with LDS instructions instead of generic ones.)
struct PairSum {
    unsigned long long cnt, by;  // this lane's share
};
// Rows lo..d-1 of the bitmap of root v0's out-neighbourhood L (two or more
// words a row, d <= 64 NW): the out-lists N+(L[i]) laid end to end over the
// lanes, each entry looked up in a table of L, whose slots' positions are a
// byte array.  False when the table could not be filled.  Latency-bound: three
// dependent loads a child batch, then a list step's loads; eight of those are in
// flight.  (R-MAT s17 of edge factor 8, a root of 100 children with its pairs
// at k = 5: 155 -> 98 us against build_rows' linear probes through generic
// pointers.)
// at: recs u64[W] | bits u64[kLeafCap / 64 + 8] | table | positions.
constexpr int rows_bits(int NW) { return NW == 4 ? 8 : 7; }
constexpr int rows_scratch(int NW) { return kTriFixed + 10 * (1 << rows_bits(NW)); }
template <int W, int NW>
__device__ __attribute__((noinline)) bool root_rows(const int64_t *off_, const int32_t *adj_, const int64_t *ostart_,
                                                    uint32_t at, uint32_t rows_at, uint32_t dp_at, int32_t v0, int lo,
                                                    int d) {
    glb_i64 *const off = (glb_i64 *)unil<W>(off_), *const ostart = (glb_i64 *)unil<W>(ostart_);
    glb_i32 *const adj = (glb_i32 *)unil<W>(adj_);
    v0 = uni<W>(v0), lo = uni<W>(lo), d = uni<W>(d);
    const Grp<W> g;
    lds_u64 *const recs = (lds_u64 *)(uintptr_t)(uint32_t)uni<W>((int)at);
    lds_u64 *const bits = recs + 64;
    lds_u64 *const rows = (lds_u64 *)(uintptr_t)(uint32_t)uni<W>((int)rows_at);
    lds_u32 *const dp = (lds_u32 *)(uintptr_t)(uint32_t)uni<W>((int)dp_at);
    constexpr int b = rows_bits(NW);
    LeafTab<true> tab;
    tab.t = (lds_u32 *)(recs + kTriFixed / 8);
    tab.b = b, tab.sh = 32 - b, tab.mul = 0x9E3779B1u;
    lds_u8 *const val = (lds_u8 *)(tab.t + (2 << b));
    glb_i32 *const L = adj + unil<W>(ostart[v0]);
    for (int t = g.gl; t < (2 << b); t += W) tab.t[t] = kEmpty;
    for (int t = lo * NW + g.gl; t < d * NW; t += W) rows[t] = 0;
    lsync();
    // only children above lo can be set in rows lo.. (lists are sorted)
    bool ok = true;
    for (int j = lo + 1 + g.gl; j < d; j += W) ok &= tab.insert(L[j], 1);
    lsync();
    if (g.ballot(!ok)) return false;
    for (int j = lo + 1 + g.gl; j < d; j += W) val[tab.slot(L[j])] = (uint8_t)j;
    lsync();
    for (int j0 = lo; j0 < d; j0 += W) {
        const int j = j0 + g.gl;
        int len = 0;
        int64_t os = 0;
        if (j < d) {
            const int32_t u = L[j];
            os = ostart[u];
            len = (int)(off[u + 1] - os);
            dp[j] = (uint32_t)len;
            if (j == d - 1) len = 0;  // no child above the last
        }
        stream_lists<8>(g, recs, bits, adj + os, len, g.gl, v0, [&](int32_t y, int i) {
            const int s = tab.slot(y);
            if (s >= 0) {
                const int k = val[s];
                lor(rows + (j0 + i) * NW + (k >> 6), 1ull << (k & 63));
            }
        });
    }
    return true;
}

// One bitmap over the out-neighbourhoods of several light roots (lane's root v
// with d children, sum of the d's T <= W): child i of the r-th root is position
// pre_r + i, and a row holds positions of its own root only, so the cliques in
// it are those of all the roots.  Rows and out-degrees as for one root; an
// out-list's entries are searched among their root's children above it.
// A root of 8 children leaves most lanes idle and waits for the same chain of
// loads as a full one; together they share it.  The search in LDS (1 to 5
// steps) costs 10-25 instructions an entry, about as much as a table's probe,
// and needs no table.  (Barabasi-Albert 100K k = 4 0.41 -> 0.12 ms, Chung-Lu 50K
// k = 4 0.27 -> 0.12, uniform random of 2 M edges k = 3 0.39 -> 0.22, R-MAT s18
// of edge factor 8 k = 4 1.47 -> 0.82.)
// at: recs u64[W] | bits u64[kLeafCap / 64 + 8] | children i32[W] | spans u32[W].
constexpr int kLightScratch = kTriFixed + 2 * 64 * 4;
template <int W>
__device__ __attribute__((noinline)) void light_rows(const int64_t *off_, const int32_t *adj_, const int64_t *ostart_,
                                                     uint32_t at, uint32_t rows_at, uint32_t dp_at, int32_t v, int d,
                                                     int lo) {
    glb_i64 *const off = (glb_i64 *)unil<W>(off_), *const ostart = (glb_i64 *)unil<W>(ostart_);
    glb_i32 *const adj = (glb_i32 *)unil<W>(adj_);
    const Grp<W> g;
    lds_u64 *const recs = (lds_u64 *)(uintptr_t)(uint32_t)uni<W>((int)at);
    lds_u64 *const bits = recs + 64;
    lds_u32 *const kid = (lds_u32 *)(recs + kTriFixed / 8), *const span = kid + 64;
    lds_u64 *const rows = (lds_u64 *)(uintptr_t)(uint32_t)uni<W>((int)rows_at);
    lds_u32 *const dp = (lds_u32 *)(uintptr_t)(uint32_t)uni<W>((int)dp_at);
    const int sc = g.iscan(d), T = g.bcast(sc, W - 1);
    // the lane's position: its root's first and one past its last
    span[g.gl] = 0;
    lsync();
    if (d > 0) span[sc - d] = (uint32_t)g.gl + 1;
    lsync();
    const uint64_t first = g.ballot(span[g.gl] != 0), upto = (2ull << g.gl) - 1;
    const int s = 63 - __builtin_clzll((first & upto) | 1);
    const int e = first & ~upto ? __builtin_ctzll(first & ~upto) : T;
    const int r = (int)span[s] - 1;
    const int64_t ls = __shfl(d > 0 ? (long long)ostart[v] : 0ll, r < 0 ? 0 : r, W);
    int most = d;
    for (int o = W / 2; o; o >>= 1) {
        const int x = __shfl_xor(most, o, W);
        most = x > most ? x : most;
    }
    most = uni<W>(most);
    int32_t u = 0x7fffffff;
    int len = 0;
    int64_t os = 0;
    if (g.gl < T) {
        u = adj[ls + g.gl - s];
        os = ostart[u];
        len = (int)(off[u + 1] - os);
        dp[g.gl] = (uint32_t)len;
        rows[g.gl] = 0;
        if (g.gl < lo || g.gl + 1 == e) len = 0;  // no child above the last
    }
    lsync();
    kid[g.gl] = (uint32_t)u;
    span[g.gl] = (uint32_t)e;
    lsync();
    const int top = most > 1 ? 1 << (31 - __builtin_clz(most - 1)) : 0;
    stream_lists<8>(g, recs, bits, adj + os, len, g.gl, -1, [&](int32_t y, int i) {
        // the last child <= y of (i, e)
        const int e = (int)span[i];
        int a = i;
        for (int o = top; o; o >>= 1) {
            const int32_t x = (int32_t)kid[a + o];  // past the children: in span
            a += a + o < e && x <= y ? o : 0;
        }
        if (a > i && (int32_t)kid[a] == y) lor(rows + i, 1ull << a);
    });
}

// A root's rows [lo, d) and out-degrees to (publish) or from (fetch) a buffer
// that workers of other compute units read: device-scope words, several loads
// in flight.  Rows of nw words at rows_at, out-degrees at dp_at, both in LDS.
template <int W, bool OUT>
__device__ __attribute__((noinline)) void copy_rows(uint64_t *buf_, uint32_t rows_at, uint32_t dp_at, int nw, int lo,
                                                    int d) {
    using glb_w64 = __attribute__((address_space(1))) uint64_t;
    glb_w64 *const buf = (glb_w64 *)unil<W>((uint64_t)buf_);
    lds_u64 *const rows = (lds_u64 *)(uintptr_t)(uint32_t)uni<W>((int)rows_at);
    lds_u32 *const dp = (lds_u32 *)(uintptr_t)(uint32_t)uni<W>((int)dp_at);
    nw = uni<W>(nw), lo = uni<W>(lo), d = uni<W>(d);
    const Grp<W> g;
    const int n = d * nw;
    // words [0, n): rows; then two out-degrees a word
    const int end = n + (d + 1) / 2;
    if constexpr (OUT) {
        for (int t = lo * nw + g.gl; t < end; t += W) {
            const int i = 2 * (t - n);
            const uint64_t x = t < n ? rows[t] : (uint64_t)dp[i] | (i + 1 < d ? (uint64_t)dp[i + 1] << 32 : 0);
            __hip_atomic_store(buf + t, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        stores_done();
    } else {
        for (int t0 = lo * nw; t0 < end; t0 += 4 * W) {
            uint64_t x[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int t = t0 + u * W + g.gl;
                x[u] = __hip_atomic_load(buf + (t < end ? t : end - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int t = t0 + u * W + g.gl, i = 2 * (t - n);
                if (t < n) rows[t] = x[u];
                else if (t < end) {
                    dp[i] = (uint32_t)x[u];
                    if (i + 1 < d) dp[i + 1] = (uint32_t)(x[u] >> 32);
                }
            }
        }
    }
}

// bytes of one stage of sw sets: sets u64[sw * NW] | prefix u32[sw + 1], size,
// cursor
__host__ __device__ constexpr int stage_bytes(int sw, int NW) { return sw * NW * 8 + ((sw + 4) & ~1) * 4; }
// a child's own bitmap: rows u64[64], the set of all its elements, dp i32[64],
// columns u64[64]
constexpr int kChildBytes = 65 * 8 + 64 * 4 + 64 * 8;
// a light batch: rows, out-degrees and the larger of its scratch and its prefix
constexpr int kLightRoots = 64 * 8 + 64 * 4 + kLightScratch;

// position of the r-th set bit (0-based) of m; m has more than r bits
DEV int select64(uint64_t m, int r) {
    int pos = 0;
#pragma unroll
    for (int sh = 32; sh >= 1; sh >>= 1) {
        const int c = __popcll(m & ((1ull << sh) - 1));
        if (r >= c) {
            r -= c;
            m >>= sh;
            pos += sh;
        }
    }
    return pos;
}
// the r-th set bit of an NW-word set
template <int NW, class P64>
DEV int set_select(P64 s, int r) {
    int w = 0;
    uint64_t m = s[0];
#pragma unroll
    for (int k = 1; k < NW; k++) {
        const int c = __popcll(m);
        if (w == k - 1 && r >= c) {
            r -= c;
            w = k;
            m = s[k];
        }
    }
    return w * 64 + select64(m, r);
}

// L: everything is in LDS, at the given LDS addresses (else generic pointers)
template <int W, int NW, bool L>
__device__ __attribute__((noinline)) PairSum clique_pairs(uint64_t rows_at, uint64_t dp_at, uint64_t pre_at,
                                                          uint64_t st_at, int K, int cur, int P, int sw) {
    using P64 = std::conditional_t<L, lds_u64 *, uint64_t *>;
    using P32 = std::conditional_t<L, lds_u32 *, uint32_t *>;
    const P64 rows = (P64)(uintptr_t)unil<W>(rows_at);
    const P32 dp = (P32)(uintptr_t)unil<W>(dp_at), pre = (P32)(uintptr_t)unil<W>(pre_at);
    const P64 st = (P64)(uintptr_t)unil<W>(st_at);
    K = uni<W>(K), cur = uni<W>(cur), P = uni<W>(P), sw = uni<W>(sw);
    auto sync = [&]() {
        if constexpr (L) lsync();
        else wsync();
    };
    const Grp<W> g;
    PairSum r{0, 0};
    // edges inside s above each element; their lower ends' out-degrees to by
    // (a set's sum fits 32 bits: with ids in degree order an out-degree is at
    // most sqrt(2E))
    auto edges = [&](const uint64_t (&s)[NW]) {
        int pc = 0;
        uint32_t by = 0;
        // a row's bits lie above its own: half a word at a time, the words from
        // there on
#pragma unroll
        for (int h = 0; h < 2 * NW; h++) {
            for (uint32_t m = (uint32_t)(s[h >> 1] >> (h & 1) * 32); m; m &= m - 1) {
                const int x = h * 32 + __builtin_ctz(m);
                by += dp[x];
                const P32 row = (P32)(rows + x * NW);
#pragma unroll
                for (int w = h; w < 2 * NW; w++) pc += __popc((uint32_t)(s[w >> 1] >> (w & 1) * 32) & row[w]);
            }
        }
        r.by += by;
        return pc;
    };
    int a = 0;
    if (K <= 5) {
        for (int t = g.gl; t < P; t += W) {
            while ((int)pre[a + 1] <= t) a++;
            const int i = cur + a, j = set_select<NW>(rows + i * NW, t - (int)pre[a]);
            r.by += (unsigned long long)dp[j];
            uint64_t s[NW];
            int pc = 0;
#pragma unroll
            for (int w = 0; w < NW; w++) {
                s[w] = rows[i * NW + w] & rows[j * NW + w];
                if (K == 4) pc += __popcll(s[w]);
            }
            if (K == 5) pc = edges(s);
            r.cnt += (unsigned long long)pc;
        }
        return r;
    }
    const int sb = stage_bytes(sw, NW) / 8;  // words of a stage
    // lane gl's set (gl < sw, else empty) becomes element gl of stage q
    auto fill = [&](int q, const uint64_t (&s)[NW]) {
        int n = 0;
#pragma unroll
        for (int w = 0; w < NW; w++) {
            if (g.gl < sw) st[q * sb + g.gl * NW + w] = s[w];
            n += __popcll(s[w]);
        }
        const int ps = g.iscan(n);
        const P32 pp = (P32)(st + q * sb + sw * NW);
        if (g.gl < sw) pp[g.gl + 1] = ps;
        if (g.gl == 0) pp[0] = 0;
        const int T = g.bcast(ps, W - 1);
        if (g.gl == 0) pp[sw + 1] = T, pp[sw + 2] = 0;
        sync();
        return T;
    };
    const int last = K - 6;  // stage whose elements are counted
    for (int p0 = 0; p0 < P; p0 += sw) {
        uint64_t s[NW];
#pragma unroll
        for (int w = 0; w < NW; w++) s[w] = 0;
        const int t = p0 + g.gl;
        if (g.gl < sw && t < P) {
            while ((int)pre[a + 1] <= t) a++;
            const int i = cur + a, j = set_select<NW>(rows + i * NW, t - (int)pre[a]);
            r.by += (unsigned long long)dp[j];
#pragma unroll
            for (int w = 0; w < NW; w++) s[w] = rows[i * NW + w] & rows[j * NW + w];
        }
        int T = fill(0, s), c = 0, q = 0;
        while (q >= 0) {
            const P64 sets = st + q * sb;
            const P32 pp = (P32)(sets + sw * NW);
            if (q == last) {
                int pa = 0;
                for (int u = g.gl; u < T; u += W) {
                    while ((int)pp[pa + 1] <= u) pa++;
                    const P64 S = sets + pa * NW;
                    const int x = set_select<NW>(S, u - (int)pp[pa]);
                    r.by += (unsigned long long)dp[x];
                    uint64_t n[NW];
#pragma unroll
                    for (int w = 0; w < NW; w++) n[w] = S[w] & rows[x * NW + w];
                    r.cnt += (unsigned long long)edges(n);
                }
                c = T;
            }
            if (c >= T) {
                q--;
                if (q >= 0) {
                    sync();
                    const P32 up = (P32)(st + q * sb + sw * NW);
                    T = uni<W>((int)up[sw + 1]);
                    c = uni<W>((int)up[sw + 2]);
                }
                continue;
            }
            // the next sw elements of this stage fill the next one
#pragma unroll
            for (int w = 0; w < NW; w++) s[w] = 0;
            const int u = c + g.gl;
            if (g.gl < sw && u < T) {
                int lo = 0, hi = sw - 1;  // last set whose prefix is <= u
                while (lo < hi) {
                    const int mid = (lo + hi + 1) >> 1;
                    if ((int)pp[mid] <= u) lo = mid;
                    else hi = mid - 1;
                }
                const P64 S = sets + lo * NW;
                const int x = set_select<NW>(S, u - (int)pp[lo]);
                r.by += (unsigned long long)dp[x];
#pragma unroll
                for (int w = 0; w < NW; w++) s[w] = S[w] & rows[x * NW + w];
            }
            c += sw;
            if (g.gl == 0) pp[sw + 2] = (uint32_t)c;
            q++;
            T = fill(q, s);
            c = 0;
        }
        sync();
    }
    return r;
}
// k = 6 below a child with a bitmap of its own: its elements [cur, cur + P) as
// the third vertex x; the second, j, runs over x's predecessors (col), the
// fourth and fifth are counted in the common successors.  Taken by x, not by j,
// lanes side by side have sets of like size: by j they fall from |N(j)| to
// nothing along one j's elements.  VALU-bound in the inner loop, 13 instructions
// a bit of the lower half and 9 of the upper.  (6-cliques of R-MAT s17 of edge
// factor 8, learned queues: 2.23 ms by j, 2.02 by x, 1.93 with the halves
// apart.)  pp: u32[65].
template <int W>
__device__ __attribute__((noinline)) PairSum child_quads(uint32_t rows_at, uint32_t cols_at, uint32_t dp_at,
                                                         uint32_t pp_at, int cur, int P) {
    lds_u64 *const rows = (lds_u64 *)(uintptr_t)(uint32_t)uni<W>((int)rows_at);
    lds_u64 *const cols = (lds_u64 *)(uintptr_t)(uint32_t)uni<W>((int)cols_at);
    lds_u32 *const dp = (lds_u32 *)(uintptr_t)(uint32_t)uni<W>((int)dp_at);
    lds_u32 *const pp = (lds_u32 *)(uintptr_t)(uint32_t)uni<W>((int)pp_at);
    cur = uni<W>(cur), P = uni<W>(P);
    const Grp<W> g;
    PairSum r{0, 0};
    int n = 0;
    if (g.gl < P) {
        const int x = cur + g.gl, d = (int)dp[x];
        const int p = __popcll(cols[x]);
        r.by += (unsigned long long)d * (unsigned)(p + 1);
        n = rows[x] ? p : 0;
    }
    const int sc = g.iscan(n);
    const int T = g.bcast(sc, W - 1);
    pp[g.gl] = (uint32_t)(sc - n);
    if (g.gl == 0) pp[W] = (uint32_t)T;
    lsync();
    int pa = 0;
    for (int u = g.gl; u < T; u += W) {
        while ((int)pp[pa + 1] <= u) pa++;
        const int x = cur + pa;
        const int j = select64(cols[x], u - (int)pp[pa]);
        const uint64_t s = rows[x] & rows[j];
        uint32_t by = 0, pc = 0;
        // a row's bits lie above its own: the upper half needs its upper words only
        const uint32_t s0 = (uint32_t)s, s1 = (uint32_t)(s >> 32);
        for (uint32_t m = s0; m; m &= m - 1) {
            const int y = __builtin_ctz(m);
            const uint64_t row = rows[y];
            by += dp[y];
            pc += (uint32_t)__popc(s0 & (uint32_t)row) + (uint32_t)__popc(s1 & (uint32_t)(row >> 32));
        }
        const lds_u32 *const up = (lds_u32 *)(rows + 32) + 1;
        for (uint32_t m = s1; m; m &= m - 1) {
            const int y = __builtin_ctz(m);
            by += dp[32 + y];
            pc += (uint32_t)__popc(s1 & up[2 * y]);
        }
        r.cnt += pc;
        r.by += by;
    }
    lsync();
    return r;
}

// Lists past the bitmaps (roots of more than 256 out-neighbours, or bitmaps off),
// in functions of their own: inlined, their loops ran on the registers that the
// bitmap paths left and on spilled ones.  Latency-bound: a chain of loads a child,
// then one a search step.  (R-MAT s15 of edge factor 8, bitmaps off, k = 5: 32.4 ms
// inlined, 29.4 so, 20.9 with fewer looks at the mailbox; R-MAT s18 of edge factor
// 16, k = 5: 670, 637, 588.)

// Whether x is in the ascending list a[0, n), n > 0.
template <class P>
DEV bool list_has(P a, int n, int32_t x) {
    int lo = 0;
    for (int len = n; len > 1;) {
        const int half = len >> 1;
        lo += a[lo + half - 1] < x ? half : 0;
        len -= half;
    }
    return a[lo] == x;
}
// Intersection of two ascending lists into out (sorted): the shorter one is
// strided, the longer searched.
template <int W>
__device__ __attribute__((noinline)) int list_intersect(const int32_t *A, int na, const int32_t *B, int nb,
                                                        int32_t *out) {
    A = unil<W>(A), B = unil<W>(B), out = unil<W>(out), na = uni<W>(na), nb = uni<W>(nb);
    const Grp<W> g;
    const int32_t *S = na > nb ? B : A, *L = na > nb ? A : B;
    const int ns = na > nb ? nb : na, nl = na > nb ? na : nb;
    if (ns == 0 || S[ns - 1] < L[0] || L[nl - 1] < S[0]) return 0;
    int w = 0;
    for (int base = 0; base < ns; base += W) {
        const int t = base + g.gl;
        const int32_t x = t < ns ? S[t] : -1;
        const bool found = t < ns && list_has(L, nl, x);
        const uint64_t m = g.ballot(found);
        if (found) out[w + g.below(m)] = x;
        w += __popcll(m);
    }
    return w;
}
// Common elements of the last level's candidates uid[i + 1, nu) and N+(uid[i]), for
// children i from lo up to hi, as many as start before `until` (one at least,
// kListRun at most): this lane's count, the children's out-degrees (all lanes the
// same) and the next child.
constexpr int kListRun = 64;
struct ListSum {
    unsigned long long cnt, by;
    int next;
};
template <int W>
__device__ __attribute__((noinline)) ListSum list_leaf(const int64_t *off_, const int32_t *adj_, const int64_t *ostart_,
                                                       const int32_t *uid, int nu, int lo, int hi, uint64_t until) {
    glb_i64 *const off = (glb_i64 *)unil<W>(off_), *const ostart = (glb_i64 *)unil<W>(ostart_);
    glb_i32 *const adj = (glb_i32 *)unil<W>(adj_);
    uid = unil<W>(uid), nu = uni<W>(nu), lo = uni<W>(lo), hi = uni<W>(hi), until = unil<W>(until);
    const Grp<W> g;
    ListSum r{0, 0, lo};
    if (hi - lo > kListRun) hi = lo + kListRun;
    do {
        const int i = r.next;
        const int32_t c = uni<W>(uid[i]);
        const int64_t os = unil<W>(ostart[c]);
        const int na = (int)(unil<W>(off[c + 1]) - os), nb = nu - i - 1;
        glb_i32 *const A = adj + os;
        const int32_t *const B = uid + i + 1;
        r.by += (unsigned long long)na;
        r.next = i + 1;
        if (na == 0 || nb == 0 || A[na - 1] < B[0] || B[nb - 1] < A[0]) continue;
        // (one loop: narrow workers of a wave then share it, R-MAT s15 k = 3 with
        // lists, 8 lanes, 1.74 -> 1.30 ms)
        const int32_t *const G = (const int32_t *)A, *const S = na <= nb ? G : B, *const L = na <= nb ? B : G;
        const int ns = na <= nb ? na : nb, nl = na <= nb ? nb : na;
        for (int t = g.gl; t < ns; t += W) r.cnt += list_has(L, nl, S[t]) ? 1 : 0;
    } while (r.next < hi && now_ticks() < until);
    return r;
}

// A job's head, in registers; its prefix ids go to the worker's LDS record (jid).
struct JobHead {
    int lvl, lo, hi, q;
    int range_end;  // > 0: a static range job over roots [jid[0], range_end)
    bool donated;
    bool shared;    // one of hi jobs that claim the root's children from its shared cursor
};

// Shared by the workers of a block.
struct BlockLDS {
    int32_t busy;      // workers that have a job or static jobs left
    uint32_t pending;  // finished jobs not yet subtracted from the launch's count
    int32_t pad[2];
};

template <int W, int MODE>
struct Worker {
    Grp<W> g;
    const EnumParams &p;
    WorkerLDS ws;
    unsigned long long *shist;  // class counters the leaf phase adds to
    const uint16_t *lut;
    int qid;
    int32_t qword;  // the current job's query word (query index | donation threshold)
    int job_sm;     // the current job's donation threshold
    bool qmotif;
    uint32_t epoch;
    char *lds_lo, *lds_top;
    char *g_lo, *g_top;
    int K;
    int32_t v0;
    int job_lvl;
    int steps;
    unsigned long long cnt;    // per-lane partial count of the current job
    unsigned long long bytes;  // per-lane partial algorithmic bytes
    int range_hi;  // end of the current range job's roots (v0 + 1 otherwise)
    uint64_t t_start;
    uint64_t last_poll;  // wall clock of the last request check
    int poll_shift;      // the check period doubles when nobody asked
    int pub;          // words a row | lo << 4 | d << 16 of the running bitmap root
                      // (0: its rows cannot be published)
    uint32_t pub_no;  // publications so far << 1 | this root's rows are published
    int from;         // worker + 1 that published a job's rows (0: nobody)
    BlockLDS *blk;
    // static queue: jobs [own_cur, own_end) of queue records own_base.. are
    // this worker's; a queue shared by a group still has to be claimed
    int64_t own_base;
    int own_cur, own_end;
    int own_queue;       // the queue's cursor slot, -1 once it is exhausted
    bool abort;
    DEV Worker(const EnumParams &p_, WorkerLDS ws_, unsigned long long *sh_, char *lds_slice, BlockLDS *blk_, int wid)
        : p(p_), ws(ws_), shist(sh_), blk(blk_) {
        lds_lo = lds_top = lds_slice;
        g_lo = g_top = p.arena + (int64_t)wid * p.arena_per_worker;
        K = 0;
        qid = -1;
        qword = 0;
        job_sm = p.steal_min;
        qmotif = MODE == 1;
        lut = nullptr;
        epoch = (uint32_t)*p.epoch;
        steps = 0;
        cnt = bytes = 0;
        range_hi = 0;
        abort = false;
        t_start = now_ticks();
        last_poll = t_start;
        poll_shift = 0;
        pub = from = 0;
        pub_no = 0;
    }
    // The word that says which of a worker's publications its arena holds.
    DEV unsigned long long *pub_word(int w) const {
        const int wpb = (int)blockDim.x / W;
        return mailbox(w / wpb) + kMailPub + w % wpb;
    }
    DEV unsigned long long pub_tag(uint32_t no) const { return ((unsigned long long)epoch << 32) | no; }
    DEV int me() const { return (int)blockIdx.x * ((int)blockDim.x / W) + uni<W>((int)threadIdx.x / W); }
    DEV void set_pub_word(unsigned long long tag) {
        if (g.gl == 0) __hip_atomic_store(pub_word(me()), tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        stores_done();
    }
    // Out-degrees follow a root's rows, which are first in the worker's slice.
    DEV char *dp_of(int nw, int d) const { return lds_lo + ((d * nw * 8 + 15) & ~15); }
    // The running root's rows to the start of this worker's arena, which holds
    // nothing else while they are in LDS.  A job on some of the root's children
    // then starts with a copy (3-8 KB, one round of loads) instead of building
    // the rows again, which took longer than most pieces: 5-cliques of R-MAT
    // s17 of edge factor 8 0.79 -> 0.73 ms, 6-cliques (plain queues) 3.14 -> 2.79,
    // 7-cliques of s13 0.97 -> 0.77.  The word says which root the arena holds:
    // it is taken back before the arena is used for anything else, and read
    // after the copy, so a copy that a later root may have overwritten is known
    // and the rows are built after all.
    DEV void publish() {
        if (!pub || (pub_no & 1)) return;
        const int nw = pub & 15, lo = pub >> 4 & 0xfff, d = pub >> 16;
        copy_rows<W, true>((uint64_t *)g_lo, lds_at(lds_lo), lds_at(dp_of(nw, d)), nw, lo, d);
        pub_no += 3;  // the next number, live
        set_pub_word(pub_tag(pub_no));
    }
    // The arena is about to be used for something else.
    DEV void unpublish() {
        pub = 0;
        if (!(pub_no & 1)) return;
        pub_no--;
        set_pub_word(0);
    }
    // Rows from where the job's giver published them; false when it has moved on.
    DEV bool fetch_rows(int nw, int lo, int d) {
        if (from <= 0 || from > p.nworkers) return false;
        copy_rows<W, false>((uint64_t *)(p.arena + (int64_t)(from - 1) * p.arena_per_worker), lds_at(lds_lo),
                            lds_at(dp_of(nw, d)), nw, lo, d);
        stores_done();
        unsigned long long tag = 0;
        if (g.gl == 0) tag = __hip_atomic_load(pub_word(from - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return g.bcast64(tag, 0) == pub_tag((uint32_t)uni<W>(ws.jid()[kJobPub - 3]));
    }

    // ---- helpers -----------------------------------------------------------
    DEV int deg(int32_t v) const { return (int)(p.off[v + 1] - p.off[v]); }
    DEV const int32_t *nbr(int32_t v) const { return p.adj + p.off[v]; }

    DEV void fail(int code) {
        if (g.gl == 0) atomicCAS(&p.sc->error, 0, code);
        abort = true;
    }

    DEV char *alloc(int64_t bytes_) {
        int64_t b = (bytes_ + 15) & ~(int64_t)15;
        if (lds_top + b <= lds_lo + p.lds_per_worker) {
            char *r = lds_top;
            lds_top += b;
            return r;
        }
        if (g_top + b <= g_lo + p.arena_per_worker) {
            char *r = g_top;
            g_top += b;
            return r;
        }
        fail(2);
        return nullptr;
    }
    DEV char *alloc_glb(int64_t bytes_) {
        int64_t b = (bytes_ + 15) & ~(int64_t)15;
        if (g_top + b <= g_lo + p.arena_per_worker) {
            char *r = g_top;
            g_top += b;
            return r;
        }
        fail(2);
        return nullptr;
    }

    DEV bool watchdog_expired() {
        return p.watchdog_ticks && (now_ticks() - t_start > p.watchdog_ticks);
    }

    DEV bool check_abort() {
        if ((++steps & 255) == 0) {
            int e = __hip_atomic_load(&p.sc->error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (e || watchdog_expired()) {
                if (!e) fail(1);
                abort = true;
            }
        }
        return abort;
    }

    // ---- donation --------------------------------------------------------------
    // An idle worker asks: it writes its request into the mailbox of a random
    // block (one line per block, kMailSlots requests) and waits for the job in
    // its own slot (one line per worker).  A busy worker looks at its own
    // block's mailbox now and then and divides what it has left between itself
    // and the askers.  No line is shared by more than a block and the few
    // workers asking it; the only word that every block updates is the launch's
    // count of unfinished jobs, when its last worker runs out of work.
    // (Device-scope accesses to one line serialise at about 8 ns.  With one
    // ticket word, one count and one static-work counter polled by every idle
    // worker, a busy worker's own accesses waited behind the polls: a 3,301-vertex
    // sparse graph's k = 5 motifs took 13 worker-seconds with 6,144 workers, 0.8
    // with 1,024; the mailboxes take it from 1.75 to 0.58 ms, ER 5K k = 4 from
    // 0.91 to 0.37, Chung-Lu 18K k = 4 from 2.12 to 1.45, a mixed batch from 31
    // to 13-17 ms.)
    //
    // A job is published without fences: each of its 16 words is one 64-bit
    // agent-scope atomic store with the request's tag in the high half; the
    // reader accepts the slot, a refusal too, once all 16 tags match.

    // Boundary j (0 <= j <= parts) when the children [cur, end) of level l are
    // cut into `parts` pieces of equal estimated work.  A clique child i of a
    // list of n candidates roots about (n - i)^e subtrees, e = K - 3 - l; motif
    // children and the leaf level count as equal.  Every piece keeps at least
    // one child (end - cur >= parts).
    DEV int split_at(int l, int cur, int end, int j, int parts) const {
        if (j <= 0) return cur;
        if (j >= parts) return end;
        const int e = K - 3 - l;
        int m;
        if (MODE == 1 || e < 1) {
            m = cur + (int)(((int64_t)(end - cur) * j) / parts);
        } else {
            const float n = (float)ws.lv()[l].nu;
            const float ep = (float)(e + 1);
            const float a = powf(n - (float)cur, ep);
            const float b = powf(n - (float)end, ep);
            const float fr = (float)j / (float)parts;
            m = (int)(n - powf(a - fr * (a - b), 1.0f / ep));
        }
        if (m < cur + j) m = cur + j;
        if (m > end - (parts - j)) m = end - (parts - j);
        return m;
    }

    DEV unsigned long long *mailbox(int b) const { return p.mail + (size_t)b * kMailStride; }

    // Requests waiting in this block's mailbox, looked for at most once per
    // period, which doubles after a look that found none: their number;
    // rq: lane i's own (i < kMailSlots; 0: none).
    DEV uint64_t period() const { return p.poll_ticks << poll_shift; }
    DEV int requests(unsigned long long &rq) {
        const uint64_t now = now_ticks();
        if (now - last_poll < period()) return 0;
        last_poll = now;
        rq = 0;
        if (g.gl < kMailSlots) {
            unsigned long long *const m = mailbox(blockIdx.x) + g.gl;
            rq = __hip_atomic_load(m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            // (two workers' changes of state can pass each other)
            if (rq == kMailIdle) rq = 0, (void)atomicCAS(m, kMailIdle, 0ull);
        }
        const int n = __popcll(g.ballot(rq != 0));
        if (n == 0) poll_shift = 1;
        return n;
    }

    // Takes up to `most` of the requests out of the mailbox (not those that
    // another worker of the block took first or whose asker gave up): their
    // number; the others' lanes get rq = 0.  fresh: the answers are new jobs,
    // counted as outstanding before they become visible, so that the count
    // cannot reach zero while they wait (finished jobs not yet subtracted
    // stand in for some of them).
    DEV int accept(unsigned long long &rq, int most, bool fresh) {
        if (g.below(g.ballot(rq != 0)) >= most) rq = 0;
        if (rq != 0 && atomicCAS(mailbox(blockIdx.x) + g.gl, rq, 0ull) != rq) rq = 0;
        const int n = __popcll(g.ballot(rq != 0));
        if (fresh && n && g.gl == 0) {
            uint32_t have = blk->pending, use = 0;
            do {
                use = have < (uint32_t)n ? have : (uint32_t)n;
            } while (use && !__hip_atomic_compare_exchange_strong(&blk->pending, &have, have - use, __ATOMIC_RELAXED,
                                                                  __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
            if (use < (uint32_t)n) {
                unsigned long long old = atomicAdd(&p.sc->outstanding, (unsigned long long)(n - use));
                landed(old);
            }
        }
        return n;
    }

    // Writes answer r = 0.. to the slot of the r-th accepted asker: words
    // f(r, 0..15).
    template <class F>
    DEV void answer(unsigned long long rq, F f) {
        uint64_t left = g.ballot(rq != 0);
        for (int r = 0; left; r++) {
            const unsigned long long q = g.bcast64(rq, __builtin_ctzll(left));
            left &= left - 1;
            uint64_t *const dst = p.q[(uint32_t)q - 1].w;
            for (int j = g.gl; j < kJobWords; j += W)
                __hip_atomic_store(dst + j, slot_word((uint32_t)(q >> 32), f(r, j)), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
    }

    // record j of a static queue (strided partition: computed)
    DEV void static_record(int64_t base, int j, int32_t (&t)[4]) const {
        if (p.sq_jobs) {
            const int32_t *s = p.sq_jobs + 4 * (base + j);
            t[0] = s[0], t[1] = s[1], t[2] = s[2], t[3] = s[3];
        } else {
            t[0] = p.n - 1 - (int)(base + (int64_t)j * p.nworkers);
            t[1] = -1;
            t[2] = t[0] + 1;
            t[3] = 0;
        }
    }

    // Claims up to `n` jobs of a queue shared by a group as this worker's.
    DEV void claim_shared(int n) {
        int j = 0;
        const int len = (int)(p.sq_off[own_queue / p.q_group + 1] - own_base);
        if (g.gl == 0) j = atomicAdd(&p.sq_cur[own_queue], n);
        j = g.bcast(j, 0);
        own_cur = j < len ? j : len;
        own_end = j + n < len ? j + n : len;
        if (own_end >= len) own_queue = -1;
    }

    // Answers waiting requests with equal shares of what this worker has left:
    // of its static jobs (they need no prefix, and the worker is busy with
    // another job), else of a range job's untouched roots, else of the children
    // of the shallowest level of the job (below `top`) that has enough of them.
    // min_first > 0: the job's own level may be cut down to pieces of that
    // many children (heavy children, where steal_min would leave too much);
    // min_pairs > 0: the same for the pairs of a bitmap root's child (level 1).
    // lists: the worker is on the list path, whose children are short beside a
    // look at the mailbox; while its looks find askers and nothing to give, the
    // period doubles, 16-fold at most.  (R-MAT s15 of edge factor 8, bitmaps off,
    // k = 6 181 -> 127 ms; with the same on the bitmap paths k = 7 of R-MAT s13 of
    // edge factor 16 3.6 -> 4.2.)
    DEV void maybe_donate(int top, int min_first = 0, int min_pairs = 0, bool lists = false) {
        unsigned long long rq = 0;
        int n = requests(rq);
        if (n == 0) return;
        const int shift = poll_shift;
        poll_shift = 0;
        if (own_cur >= own_end && own_queue >= 0) claim_shared(n);
        if (own_cur < own_end) {
            const int cur = own_cur, len = own_end - cur;
            n = accept(rq, len, false);
            if (n == 0) return;
            // this worker keeps the first share (it may be empty)
            auto cut = [&](int j) { return cur + (int)((int64_t)len * j / (n + 1)); };
            answer(rq, [&](int r, int j) {
                return j == 0   ? kStaticJobs
                       : j == 1 ? cut(r + 1)
                       : j == 2 ? cut(r + 2)
                       : j == 4 ? (int)(uint32_t)own_base
                       : j == 5 ? (int)(uint32_t)(own_base >> 32)
                                : 0;
            });
            own_end = cut(1);
            return;
        }
        if (p.steal && range_hi - v0 - 1 >= 2) {
            const int lo = v0 + 1, len = range_hi - lo;
            n = accept(rq, len - 1, true);
            if (n == 0) return;
            auto cut = [&](int j) { return lo + (int)((int64_t)len * j / (n + 1)); };
            answer(rq, [&](int r, int j) {
                return j == 0 ? 0 : j == 1 ? -1 : j == 2 ? cut(r + 2) : j == 3 ? qword : j == 4 ? cut(r + 1) : -1;
            });
            range_hi = cut(1);
            if (g.gl == 0) ws.st()[kStDonated] += (unsigned long long)n;
            return;
        }
        // a clique's last level has cheap children: split it only in bigger pieces
        const int leaf_min = 4 * job_sm;
        for (int l = p.steal ? job_lvl : top; l < top; l++) {
            const int cur = ws.lv()[l].cur, end = ws.lv()[l].end;
            const int minc = min_pairs > 0 && l == 1                ? min_pairs
                             : min_first > 0 && l == job_lvl ? min_first
                             : l == K - 3                    ? leaf_min
                                                             : job_sm;
            if (end - cur < minc) continue;
            int most = (end - cur) / minc - 1;
            most = most < 1 ? 1 : most > end - cur - 1 ? end - cur - 1 : most;
            if (most < 1) break;
            n = accept(rq, most, true);
            if (n == 0) return;
            publish();
            answer(rq, [&](int r, int j) {
                return j == 0   ? l
                       : j == kJobPub && l <= 1     ? (pub_no & 1 ? me() + 1 : 0)
                       : j == kJobPub + 1 && l <= 1 ? (int)pub_no
                       : j == 1 ? split_at(l, cur, end, r + 1, n + 1)
                       : j == 2 ? split_at(l, cur, end, r + 2, n + 1)
                       : j == 3 ? qword
                       : j - 4 <= l ? ws.lv()[j - 4].vtx
                                    : -1;
            });
            ws.lv()[l].end = split_at(l, cur, end, 1, n + 1);
            if (g.gl == 0) ws.st()[kStDonated] += (unsigned long long)n;
            return;
        }
        // nothing to give: the askers go elsewhere
        if (lists) poll_shift = shift < 4 ? shift + 1 : 4;
    }

    // ---- motif levels ----------------------------------------------------------
    DEV void motif_root_level(int32_t v) {
        Lvl &L = ws.lv()[0];
        const int32_t *a = p.adj + p.ostart[v];
        int n = (int)(p.off[v + 1] - p.ostart[v]);
        L.uid = const_cast<int32_t *>(a);
        L.upm = nullptr;
        L.eid = const_cast<int32_t *>(a);
        L.epm = nullptr;
        L.nu = n;
        L.ne = n;
        L.vtx = v;
        L.ind = 0;
        L.sdeg = deg(v);
        L.mark_lds = lds_top;
        L.mark_glb = g_top;
    }

    DEV uint8_t upm_at(const Lvl &L, int j) const { return L.upm ? L.upm[j] : (uint8_t)0x81; }
    DEV int epm_at(const Lvl &L, int j) const { return L.epm ? (int)L.epm[j] : 1; }

    // U_{l+1}, E_{l+1} from level l and child c (pmc = c's mask in U_l).
    DEV void motif_forward(int l, int32_t c, int pmc) {
        Lvl &P = ws.lv()[l];
        Lvl &N = ws.lv()[l + 1];
        const int l1 = l + 1;
        const int64_t cb = unil<W>(p.off[c]);
        const int32_t *nc = p.adj + cb;
        const int dc = (int)(unil<W>(p.off[c + 1]) - cb);
        const int s0 = uni<W>(lower_bound(nc, dc, v0 + 1));
        const int q = dc - s0;
        const int pnu = uni<W>(P.nu);
        const int32_t *const puid = unil<W>(P.uid);
        const uint8_t *const pupm = unil<W>(P.upm);
        N.mark_lds = lds_top;
        N.mark_glb = g_top;
        const int cap = pnu + q;
        int32_t *uid = (int32_t *)alloc((int64_t)cap * 4);
        uint8_t *upm = (uint8_t *)alloc(cap);
        int32_t *eid = (int32_t *)alloc((int64_t)cap * 4);
        uint8_t *epm = (uint8_t *)alloc(cap);
        char *tmark_l = lds_top, *tmark_g = g_top;
        int32_t *nw = (int32_t *)alloc((int64_t)(q > 0 ? q : 1) * 4);
        uint8_t *hit = (uint8_t *)alloc(pnu > 0 ? pnu : 1);
        if (abort) return;
        for (int j = g.gl; j < pnu; j += W) hit[j] = 0;
        wsync();
        // scan N(c) above v0: mark hits in U_l, collect new vertices (sorted)
        int nnew = 0;
        for (int base = 0; base < q; base += W) {
            int t = base + g.gl;
            bool in = t < q;
            int32_t x = in ? nc[s0 + t] : 0;
            bool found = false;
            if (in) {
                int pos = lower_bound(puid, pnu, x);
                found = pos < pnu && puid[pos] == x;
                if (found) hit[pos] = 1;
            }
            uint64_t m = g.ballot(in && !found);
            if (in && !found) nw[nnew + g.below(m)] = x;
            nnew += __popcll(m);
        }
        wsync();
        // merge by ranks: old elements and new ones interleave in id order
        const uint8_t bit = (uint8_t)(1u << l1);
        for (int j = g.gl; j < pnu; j += W) {
            int32_t x = puid[j];
            int o = j + lower_bound(nw, nnew, x);
            uint8_t pm = pupm ? pupm[j] : (uint8_t)0x81;
            if (hit[j]) pm |= bit;
            bool valid = (pm & 0x80) && x > c;
            uid[o] = x;
            upm[o] = (uint8_t)((pm & 0x7f) | (valid ? 0x80 : 0));
        }
        for (int t = g.gl; t < nnew; t += W) {
            int32_t x = nw[t];
            int o = t + lower_bound(puid, pnu, x);
            uid[o] = x;
            upm[o] = (uint8_t)(bit | 0x80);
        }
        const int nu = pnu + nnew;
        wsync();
        int ne = 0;
        for (int base = 0; base < nu; base += W) {
            int j = base + g.gl;
            bool in = j < nu;
            uint8_t pm = in ? upm[j] : 0;
            bool v = in && (pm & 0x80);
            uint64_t m = g.ballot(v);
            if (v) {
                int o = ne + g.below(m);
                eid[o] = uid[j];
                epm[o] = (uint8_t)(pm & 0x7f);
            }
            ne += __popcll(m);
        }
        wsync();
        // release the temporaries
        lds_top = tmark_l;
        g_top = tmark_g;
        N.uid = uid;
        N.upm = upm;
        N.eid = eid;
        N.epm = epm;
        N.nu = nu;
        N.ne = ne;
        N.vtx = c;
        N.sdeg = P.sdeg + dc;
        N.ind = (l1 >= 2) ? P.ind + ((uint64_t)pmc << quick_off(l1)) : 0;
    }

    // ---- motif leaf ------------------------------------------------------------
    // k = 3: children of the root to a chunk (each builds the root's table again)
    static constexpr int kMotif3Chunk = 512;
    DEV static int motif3_chunk(int children) { return children <= 8 * kMotif3Chunk ? kMotif3Chunk : (children + 7) / 8; }
    // Leaf node of child i0 of level pl = K-4 (k >= 4), or the root itself at
    // k = 3 (pl = -1) with the elements [lo, hi) of its list as children.
    DEV void motif_leaf_node(int pl, int i0, int lo, int hi) {
        if (check_abort()) return;
        const Lvl &P = ws.lv()[pl < 0 ? 0 : pl];
        const int32_t c = pl < 0 ? v0 : P.eid[i0];
        const int pmc = pl < 0 ? 0 : epm_at(P, i0), pnu = pl < 0 ? 0 : P.nu, sd = pl < 0 ? 0 : P.sdeg;
        auto run = [&](auto wide, uint32_t *gtab, int space) {
            return motif_leaf<W, decltype(wide)::value>(p.off, p.adj, p.ostart, lut, P.uid, P.upm, lds_at(shist),
                                                        lds_at(lds_lo), gtab, P.ind, v0, K, c, pmc, pnu, sd, lo, hi, space);
        };
        LeafSum r = run(std::false_type{}, nullptr, p.lds_per_worker - motif_leaf_fixed(W, K));
        if (r.big) {
            // U does not fit the LDS table: one in the arena
            char *const mg = g_top;
            const int b = r.big;
            uint32_t *const gtab = (uint32_t *)alloc_glb((int64_t)4 << b);
            if (abort) return;
            r = b >= kLeafWideBits ? run(std::true_type{}, gtab, b) : run(std::false_type{}, gtab, b);
            g_top = mg;
            if (r.big) fail(2);
        }
        cnt += r.cnt;
        bytes += r.bytes;
    }

    // ---- clique levels ----------------------------------------------------------
    DEV void clique_root_level(int32_t v) {
        Lvl &L = ws.lv()[0];
        L.uid = const_cast<int32_t *>(p.adj + p.ostart[v]);
        L.nu = (int)(p.off[v + 1] - p.ostart[v]);
        L.vtx = v;
        L.mark_lds = lds_top;
        L.mark_glb = g_top;
    }

    DEV const int32_t *onbr(int32_t v) const { return p.adj + p.ostart[v]; }
    DEV int odeg(int32_t v) const { return (int)(p.off[v + 1] - p.ostart[v]); }

    DEV void clique_forward(int l, int i) {
        Lvl &P = ws.lv()[l];
        Lvl &N = ws.lv()[l + 1];
        const int32_t c = P.uid[i];
        const int32_t *B = P.uid + i + 1;
        const int nb = P.nu - i - 1;
        const int na = odeg(c);
        N.mark_lds = lds_top;
        N.mark_glb = g_top;
        const int cap = na < nb ? na : nb;
        int32_t *out = (int32_t *)alloc((int64_t)(cap > 0 ? cap : 1) * 4);
        if (abort) return;
        const int w = list_intersect<W>(onbr(c), na, B, nb, out);
        wsync();
        N.uid = out;
        N.nu = w;
        N.vtx = c;
    }

    DEV void clique_leaf_phase(int l, int lo, int hi) {
        Lvl &P = ws.lv()[l];
        while (lo < hi) {
            if (check_abort()) return;
            // donation of this level's tail happens through lv[l].cur/end
            P.cur = lo;
            maybe_donate(l + 1, 0, 0, true);
            hi = uni<W>(P.end);
            if (lo >= hi) break;
            const ListSum r = list_leaf<W>(p.off, p.adj, p.ostart, P.uid, P.nu, lo, hi,
                                           last_poll + period());
            cnt += r.cnt;
            if (g.gl == 0) bytes += 4ull * r.by;
            lo = uni<W>(r.next);
        }
    }

    // k = 3: the root's children [lo, hi), a wave of them per donation check;
    // false when N+(v) does not fit an LDS table
    DEV bool triangle_root(int lo, int hi) {
        Lvl &R = ws.lv()[0];
        const int d = R.nu;
        int b = 7;
        while (9 * (2 << b) < 20 * d) b++;  // at most 45% full
        while (b > 7 && tri_fixed(W) + (8 << b) > p.lds_per_worker && 7 * d <= 6 * (1 << b)) b--;
        if (tri_fixed(W) + (8 << b) > p.lds_per_worker) return false;
        R.cur = lo;
        R.end = hi < d ? hi : d;
        for (bool first = true;; first = false) {
            if (check_abort()) return true;
            maybe_donate(1);
            const int cur = uni<W>(R.cur), end = uni<W>(R.end);
            if (cur >= end) return true;
            const int to = end - cur < W ? end : cur + W;
            R.cur = to;
            bool ok;
            const TriSum r = triangles<W>(p.off, p.adj, p.ostart, lds_at(lds_lo), b, v0, cur, to, first, ok);
            if (!ok) {
                R.cur = cur;
                return false;
            }
            cnt += r.cnt;
            bytes += 4ull * r.by;
        }
    }

    // ---- clique, local bitmap of the root's out-neighbourhood -------------
    template <int NW>
    DEV void clique_bitmap_root(int32_t v, int lvl, int lo, int hi, bool first_piece, bool shared) {
        const int d = uni<W>(odeg(v));
        const int32_t *L = onbr(v);
        Lvl &R = ws.lv()[0];
        R.uid = const_cast<int32_t *>(L);
        R.nu = d;
        R.vtx = v;
        R.mark_lds = lds_top;
        R.mark_glb = g_top;
        const int jobs_on_root = hi;  // shared: the root's job count
        if (shared) {
            lo = 0;
            hi = d;
        }
        // level 1: pairs [lo, hi) of one child, at `child`
        const int p0 = lo, p1 = hi, child = lvl ? uni<W>(lower_bound(L, d, ws.jid()[1])) : 0;
        if (lvl) lo = child, hi = child + 1;
        if (hi > d) hi = d;
        if (lo >= hi) return;
        // pair-phase data first, so that it gets the LDS
        uint64_t *rows = (uint64_t *)alloc((int64_t)d * NW * 8);
        int32_t *dp = (int32_t *)alloc((int64_t)d * 4);
        int32_t *pre = nullptr;
        if (abort) return;
        // a root whose bitmap the launch prebuilt (a heavy root cut into
        // many pieces): copy its rows instead of building them
        int slot = -1;
        const bool in_lds = (char *)dp >= lds_lo && (char *)dp < lds_top && (char *)rows >= lds_lo && (char *)rows < lds_top;
        if (p.npre > 0) {
            int a = 0, b = p.npre;
            while (a < b) {
                const int mid = (a + b) >> 1;
                if (p.pre_roots[mid] < v) a = mid + 1;
                else b = mid;
            }
            if (a < p.npre && p.pre_roots[a] == v) slot = a;
        }
        if (slot >= 0) {
            const uint64_t *gr = (const uint64_t *)(p.pre + p.pre_offs[slot]);
            const int32_t *gd = (const int32_t *)(gr + (int64_t)d * NW);
            for (int t = lo * NW + g.gl; t < d * NW; t += W) rows[t] = gr[t];
            for (int i = g.gl; i < d; i += W) dp[i] = gd[i];
            wsync();
        } else if (shared) {
            fail(3);  // the host gives a shared cursor only to prebuilt roots
            return;
        } else if (!(in_lds && from && fetch_rows(NW, lo, d)) && !stream_rows<NW>(v, lo, d, rows, dp)) {
            pre = (int32_t *)alloc((int64_t)(d + 1) * 4);
            if (abort) return;
            build_rows<NW>(v, lo, d, L, rows, dp, pre);
            if (abort) return;
        }
        if (!pre) pre = (int32_t *)alloc((int64_t)(d + 1) * 4);
        if (abort) return;
        wsync();
        // K >= 6: the stages, allocated after the build so that the build's
        // hash gets the LDS first; as wide as the LDS left allows
        int sw = W;
        char *st = nullptr, *cu = nullptr;
        if ((K == 6 || (K > 6 && NW > 1)) && lds_top + kChildBytes <= lds_lo + p.lds_per_worker) cu = alloc(kChildBytes);
        if (K >= 6) {
            while (sw > 8 && lds_top + (K - 5) * stage_bytes(sw, NW) > lds_lo + p.lds_per_worker) sw >>= 1;
            st = alloc((int64_t)(K - 5) * stage_bytes(sw, NW));
            if (abort) return;
        }
        if (in_lds && slot < 0 && g_top == g_lo && (int)blockDim.x / W <= kMailPubs &&
            p.arena_per_worker >= (int64_t)d * (NW * 8 + 4) + 8)
            pub = NW | lo << 4 | d << 16;
        if (lvl) {
            R.cur = R.end = hi;
            pairs_of_child<NW>(R, rows, dp, pre, st, sw, cu, child, p0, p1);
        } else if (shared) {
            // guided self-scheduling with the root's other jobs: each claim
            // takes about 1 / (2 x jobs on the root) of the children left, at
            // least one, so the root's last children are spread thinly
            // whatever their weights; the claim that starts at child 0 counts
            // the root's bytes.  (Claims sized by estimated work, pop^(k-3)
            // per child with a compare-and-swap cursor, balanced better but
            // their extra claims cost more: R-MAT k = 6 4.78 -> 5.0 ms.)
            int32_t *cursor = p.pre_cursor + slot;
            const int share = 2 * (jobs_on_root > 1 ? jobs_on_root : 1);
            while (!abort) {
                int a = 0, n = 1;
                if (g.gl == 0) {
                    const int cur = __hip_atomic_load(cursor, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    n = d > cur ? (d - cur + share - 1) / share : 1;
                    a = atomicAdd(cursor, n);
                }
                a = g.bcast(a, 0);
                n = g.bcast(n, 0);
                if (a >= d) break;
                if (a == 0 && g.gl == 0) bytes += 4ull * (unsigned long long)d;
                pair_phase<NW>(R, rows, dp, pre, st, sw, cu, a, a + n < d ? a + n : d);
            }
        } else {
            if (first_piece && g.gl == 0) bytes += 4ull * (unsigned long long)d;
            pair_phase<NW>(R, rows, dp, pre, st, sw, cu, lo, hi);
        }
        lds_top = R.mark_lds;
        g_top = R.mark_glb;
    }

    // Rows lo..d-1 of root v's bitmap by root_rows / light_rows; false when
    // they or the scratch are not in LDS
    template <int NW>
    DEV bool stream_rows(int32_t v, int lo, int d, uint64_t *rows, int32_t *dp) {
        char *const at = lds_top;
        if ((char *)rows < lds_lo || (char *)rows >= at || (char *)dp < lds_lo || (char *)dp >= at) return false;
        char *const end = lds_lo + p.lds_per_worker;
        if (d <= W) {
            if (at + kLightScratch > end) return false;
            light_rows<W>(p.off, p.adj, p.ostart, lds_at(at), lds_at(rows), lds_at(dp), v, g.gl == 0 ? d : 0, lo);
            wsync();
            return true;
        }
        if constexpr (NW > 1) {
            if (at + rows_scratch(NW) > end) return false;
            const bool ok = root_rows<W, NW>(p.off, p.adj, p.ostart, lds_at(at), lds_at(rows), lds_at(dp), v, lo, d);
            wsync();
            return ok;
        }
        return false;
    }

    // Several light roots at once (lane's root v with d children, sum <= W):
    // one bitmap, enumerated as one root's; pieces of it are not given away.
    DEV void light_roots(int32_t v, int d) {
        job_lvl = 2;
        unpublish();
        lds_top = lds_lo;
        g_top = g_lo;
        cnt = 0;
        const int T = uni<W>(g.bcast(g.iscan(d), W - 1));
        uint64_t *rows = (uint64_t *)alloc(64 * 8);
        int32_t *dp = (int32_t *)alloc(64 * 4);
        light_rows<W>(p.off, p.adj, p.ostart, lds_at(lds_top), lds_at(rows), lds_at(dp), v, d, 0);
        wsync();
        bytes += 4ull * (unsigned long long)d;
        if (K == 3) {
            // (larger sizes look in pair_phase)
            if (check_abort()) return;
            maybe_donate(0);
            if (g.gl < T) {
                cnt += (unsigned long long)__popcll(rows[g.gl]);
                bytes += 4ull * (unsigned long long)dp[g.gl];
            }
            return;
        }
        int32_t *pre = (int32_t *)alloc((int64_t)(T + 1) * 4);
        int sw = W;
        char *st = nullptr;
        if (K >= 6) {
            while (sw > 8 && lds_top + (K - 5) * stage_bytes(sw, 1) > lds_lo + p.lds_per_worker) sw >>= 1;
            st = alloc((int64_t)(K - 5) * stage_bytes(sw, 1));
        }
        if (abort) return;
        Lvl &R = ws.lv()[0];
        R.uid = (int32_t *)dp;  // ids are only read for jobs given away
        R.nu = T;
        R.vtx = v0;
        pair_phase<1>(R, rows, dp, pre, st, sw, nullptr, 0, T);
    }

    // Rows lo..d-1 of the local bitmap of root v (L = N+(v), d = |L|): row i
    // bit j set when L[j] is in N+(L[i]); dp[i] = out-degree of L[i].
    template <int NW>
    DEV void build_rows(int32_t v, int lo, int d, const int32_t *L, uint64_t *rows, int32_t *dp, int32_t *pre) {
        (void)v;
        // build scratch, released after the build: a hash of N+(v) (id ->
        // position, load factor <= 1/2) and each child's list start
        char *const build_lds = lds_top;
        char *const build_glb = g_top;
        constexpr int HB = NW == 1 ? 7 : (NW == 2 ? 8 : 9);
        constexpr int HS = 1 << HB;
        int32_t *hkey = (int32_t *)alloc(HS * 4);
        uint8_t *hval = (uint8_t *)alloc(HS);
        int64_t *rst = (int64_t *)alloc((int64_t)d * 8);
        if (abort) return;
        for (int t = g.gl; t < HS; t += W) hkey[t] = -1;
        for (int i = g.gl; i < d; i += W) {
            const int32_t u = L[i];
            const int64_t os = p.ostart[u];
            rst[i] = os;
            dp[i] = (int)(p.off[u + 1] - os);
        }
        for (int t = lo * NW + g.gl; t < d * NW; t += W) rows[t] = 0;
        wsync();
        // only children above lo can be set in rows lo.. (lists are sorted)
        for (int j = lo + g.gl; j < d; j += W) {
            const int32_t key = L[j];
            uint32_t h = ((uint32_t)key * 2654435761u) >> (32 - HB);
            while (true) {
                if (atomicCAS(&hkey[h], -1, key) == -1) {
                    hval[h] = (uint8_t)j;
                    break;
                }
                h = (h + 1) & (HS - 1);
            }
        }
        // flatten (i, x in N+(L[i])) for i in [lo, d) and set the bits
        int carry = 0;
        for (int base = lo; base < d; base += W) {
            const int i = base + g.gl;
            const int x = i < d ? dp[i] : 0;
            const int sc = g.iscan(x);
            if (i < d) pre[i - lo + 1] = carry + sc;
            carry += g.bcast(sc, W - 1);
        }
        if (g.gl == 0) pre[0] = 0;
        wsync();
        const int T = carry;
        int a = 0;  // row of this lane's element; t only grows
        constexpr int U = 4;
        for (int t0 = 0; t0 < T; t0 += U * W) {
            int32_t xs[U];
            int ra[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int t = t0 + u * W + g.gl;
                ra[u] = -1;
                xs[u] = 0;
                if (t < T) {
                    while (pre[a + 1] <= t) a++;
                    ra[u] = a;
                    xs[u] = p.adj[rst[lo + a] + (t - pre[a])];
                }
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (ra[u] < 0) continue;
                const int32_t x = xs[u];
                uint32_t h = ((uint32_t)x * 2654435761u) >> (32 - HB);
                int k;
                while ((k = hkey[h]) != x && k != -1) h = (h + 1) & (HS - 1);
                if (k == x) {
                    const int j = hval[h];
                    atomicOr(&rows[(lo + ra[u]) * NW + (j >> 6)], 1ull << (j & 63));
                }
            }
        }
        wsync();
        lds_top = build_lds;
        g_top = build_glb;
    }

    // first-level children [lo, hi) in batches of W; each batch is
    // flattened into its (i, j) pairs, which the lanes stride over
    // (st, sw: the stages of K >= 6; cu: room for a child's own bitmap)
    // a batch of the pairs described by pre, from child cur on
    template <int NW>
    DEV PairSum pairs(const uint64_t *rows, const int32_t *dp, const int32_t *pre, const char *st, int sw, int cur,
                      int P) {
        auto lds = [&](const void *a) { return (const char *)a >= lds_lo && (const char *)a < lds_lo + p.lds_per_worker; };
        if (lds(rows) && lds(dp) && lds(pre) && (K < 6 || lds(st)))
            return clique_pairs<W, NW, true>(lds_at(rows), lds_at(dp), lds_at(pre), lds_at(st), K, cur, P, sw);
        return clique_pairs<W, NW, false>((uintptr_t)rows, (uintptr_t)dp, (uintptr_t)pre, (uintptr_t)st, K, cur, P, sw);
    }

    // k >= 6: the pairs [lo, hi) of child i alone, a chunk at a time, so that a
    // heavy child's pairs are given away too: its work grows with the square
    // (k = 6) of its pairs or faster, and one worker's share of a dense root
    // would otherwise be the launch (8,192-vertex R-MAT k = 7: 1.90 ms with whole
    // children, 1.28 ms with their pairs divided, 0.95 ms with batches of W / 2
    // pairs instead of 2 W as well)
    template <int NW>
    DEV void pairs_of_child(Lvl &R, const uint64_t *rows, const int32_t *dp, int32_t *pre, char *st, int sw, char *cu,
                            int i, int lo, int hi) {
        Lvl &C = ws.lv()[1];
        int n = 0;
#pragma unroll
        for (int w = 0; w < NW; w++) n += __popcll(rows[i * NW + w]);
        n = uni<W>(n);
        C.vtx = R.uid[i];
        C.nu = n;
        C.cur = lo;
        C.end = hi < n ? hi : n;
        const int chunk = K >= 7 ? W / 4 : W;
        // a child with at most 64 pairs gets a bitmap of its own, over its own
        // elements: one word a row, where the root's has NW.  (The inner loop
        // takes 21 instructions a bit instead of 44, and almost all of k = 6's
        // bits lie under such children of wide roots: R-MAT s17 of edge factor
        // 8, 2.97 -> 2.45 ms.  Below `alone` pairs a child is better off in a
        // batch of several: 16 / 24 / 40 measured 2.54 / 2.45 / 2.79 ms, and
        // with child_quads 16 / 24 / 32 2.11 / 2.04 / 2.04.)  At k = 6 a full
        // wave then takes child_quads, whose order keeps its lanes level; for
        // that a one-word root's children get bitmaps too (6-cliques of R-MAT
        // s14 0.41 -> 0.34 ms, s13 0.27 -> 0.22; from 32 pairs on 0.35 and 0.23).
        const bool own = cu && n <= 64;
        uint64_t *const crow = (uint64_t *)cu;
        int32_t *const cdp = (int32_t *)(crow + 65);
        uint64_t *const ccol = (uint64_t *)(cdp + 64);
        // (the quads' prefix takes the stage's place, which a narrow one is too
        // small for)
        const bool quads = W == 64 && K == 6 && own && st >= lds_lo && st < lds_lo + p.lds_per_worker &&
                           stage_bytes(sw, NW) >= 4 * (W + 1);
        int sw1 = sw;
        if (own) {
            while (sw1 < W && stage_bytes(2 * sw1, 1) <= stage_bytes(sw, NW)) sw1 *= 2;
            for (int x = g.gl; x < n; x += W) {
                const int at = set_select<NW>(rows + i * NW, x);
                uint64_t out = 0, col = 0;
                int e = 0;
#pragma unroll
                for (int w = 0; w < NW; w++) {
                    const uint64_t in = rows[at * NW + w];
                    uint64_t m = unil<W>(rows[i * NW + w]);
                    while (m) {
                        const int b = __builtin_ctzll(m);
                        m &= m - 1;
                        const uint64_t bit = (in >> b) & 1;
                        out |= bit << e;
                        if constexpr (W == 64) {
                            const uint64_t pred = __ballot(bit != 0);
                            if (e == g.gl) col = pred;
                        }
                        e++;
                    }
                }
                ccol[x] = col;
                crow[x] = out;
                cdp[x] = dp[at];
            }
            if (g.gl == 0) crow[64] = n < 64 ? (1ull << n) - 1 : ~0ull;
        }
        while (true) {
            if (check_abort()) return;
            maybe_donate(2, 2, K >= 7 ? 4 : 32);
            const int cur = uni<W>(C.cur), end = uni<W>(C.end);
            if (cur >= end) return;
            const int P = end - cur < chunk ? end - cur : chunk;
            C.cur = cur + P;
            if (g.gl == 0) pre[0] = -cur, pre[1] = P;
            wsync();
            const PairSum r = quads ? child_quads<W>(lds_at(crow), lds_at(ccol), lds_at(cdp), lds_at(st), cur, P)
                              : own ? pairs<1>(crow, cdp, pre, st, sw1, 64, P) : pairs<NW>(rows, dp, pre, st, sw, i, P);
            cnt += r.cnt;
            bytes += 4ull * r.by;
            wsync();
        }
    }

    template <int NW>
    DEV void pair_phase(Lvl &R, const uint64_t *rows, const int32_t *dp, int32_t *pre, char *st, int sw, char *cu,
                        int lo, int hi) {
        // a front child with this many pairs is heavy enough to travel alone,
        // with twice as many its pairs are divided too
        const int heavy = K >= 7 ? 4 : W / 2, alone = K >= 7 ? 8 : 24;
        R.cur = lo;
        R.end = hi;
        unsigned long long by = 0;
        while (true) {
            if (check_abort()) break;
            int front = 0;
            if (K >= 6 && g.gl == 0 && R.cur < R.end) {
#pragma unroll
                for (int w = 0; w < NW; w++) front += __popcll(rows[R.cur * NW + w]);
            }
            front = g.bcast(front, 0);
            maybe_donate(1, front >= heavy ? 2 : 0);
            if (front >= (cu ? alone : 2 * heavy) && R.cur < R.end) {
                const int i = R.cur;
                R.cur = i + 1;
                if (g.gl == 0) by += (unsigned long long)dp[i];
                pairs_of_child<NW>(R, rows, dp, pre, st, sw, cu, i, 0, 0x7fffffff);
                continue;
            }
            const int cur = R.cur, end = R.end;
            if (cur >= end) break;
            // a batch holds children until it has about `target` pairs (at
            // least one child), so heavy roots reach a donation point often
            const int avail = end - cur < W ? end - cur : W;
            int np = 0;
            if (g.gl < avail) {
#pragma unroll
                for (int w = 0; w < NW; w++) np += __popcll(rows[(cur + g.gl) * NW + w]);
            }
            const int sc = g.iscan(np);
            const int target = K == 4 ? 16 * W : K >= 7 ? W / 2 : 2 * W;
            int take = __popcll(g.ballot(g.gl < avail && sc - np < target));
            take = take < 1 ? 1 : take;
            R.cur = cur + take;
            if (g.gl < take) {
                by += (unsigned long long)dp[cur + g.gl];
                pre[g.gl + 1] = sc;
            }
            if (g.gl == 0) pre[0] = 0;
            const int P = g.bcast(sc, take - 1);
            wsync();
            const PairSum r = pairs<NW>(rows, dp, pre, st, sw, cur, P);
            cnt += r.cnt;
            by += r.by;
            wsync();
        }
        bytes += 4ull * by;
    }

    // ---- one job ------------------------------------------------------------
    // children [lo, hi) of the node whose prefix ws.jid()[0..lvl] is in LDS;
    // first_piece: a static job that starts at the root's first child (the
    // root node's own bytes are counted once, by that job); shared: one of
    // `hi` jobs on a prebuilt bitmap root that claim its children from the
    // root's shared cursor
    // Light roots that can be run together from `root` on (each with at most
    // half the lanes' children, a quarter at k >= 7, where one lane's share of a
    // dense one could outlast the launch): of a range job, then
    // of the worker's own queue.  False when there is only one; else lane's
    // root v with d children (d = 0 past the last), the job's root and the
    // queue moved on to the last of them, `merged` the queue's jobs taken.
    DEV bool collect_light(const JobHead &jh, int &root, int &merged, int32_t &v, int &d) {
        const int most = K <= 6 ? W / 2 : W / 4;
        if (K < 3 || (K > 3 && !p.bitmap) || p.root_cost || p.root_count || p.lds_per_worker < kLightRoots) return false;
        if (jh.lvl || jh.shared || jh.donated || (!jh.range_end && (jh.lo != 0 || jh.hi != 0x7fffffff))) return false;
        if (odeg(root) > most) return false;
        const int m = range_hi - root;
        // a queue shared by a group: light roots are claimed many at a time
        if (m == 1 && own_cur >= own_end && own_queue >= 0) claim_shared(W / 8);
        v = root + g.gl;
        bool ok = g.gl < m;
        if (!ok && own_cur + g.gl - m < own_end) {
            int32_t t[4];
            static_record(own_base, own_cur + g.gl - m, t);
            v = t[0];
            ok = t[3] == jh.q && (t[1] == -1 ? t[2] == v + 1 : t[1] == 0 && t[2] == 0x7fffffff);
        }
        d = ok ? odeg(v) : W + 1;
        const bool light = d <= most;
        const int sc = g.iscan(light ? d : W + 1);
        const uint64_t no = g.ballot(!light || sc > W);
        const int n = no ? __builtin_ctzll(no) : W;
        if (n < 2) return false;
        if (g.gl >= n) d = 0;
        root += (n < m ? n : m) - 1;
        const int taken = n > m ? n - m : 0;
        own_cur += taken;
        merged += taken;
        v0 = root;
        return true;
    }

    DEV void run_job(int lvl, int lo, int hi, bool first_piece, bool shared) {
        v0 = uni<W>(ws.jid()[0]);
        if constexpr (MODE == 0) unpublish();
        job_lvl = lvl;
        lds_top = lds_lo;
        g_top = g_lo;
        cnt = 0;
        constexpr bool motif = MODE == 1;
        // a motif worker's slice is its leaf scratch; its lists are in the arena
        if (motif) lds_top = lds_lo + p.lds_per_worker;
        if (!motif && K == 2) {
            if (g.gl == 0) {
                int d = odeg(v0);
                cnt += (unsigned long long)d;
                bytes += 4ull * (unsigned long long)d;
            }
            return;
        }
        if (!motif && p.bitmap && K >= 4 && (lvl == 0 || (lvl == 1 && K >= 6))) {
            const int d = odeg(v0);
            if (d <= 64) {
                clique_bitmap_root<1>(v0, lvl, lo, hi, first_piece, shared);
                return;
            }
            if (d <= 128) {
                clique_bitmap_root<2>(v0, lvl, lo, hi, first_piece, shared);
                return;
            }
            if (d <= 256) {
                clique_bitmap_root<4>(v0, lvl, lo, hi, first_piece, shared);
                return;
            }
        }
        if (shared) {  // only prebuilt bitmap roots have a shared cursor
            fail(3);
            return;
        }
        // rebuild the prefix levels 0..lvl
        if (motif) motif_root_level(v0);
        else clique_root_level(v0);
        if (first_piece && g.gl == 0)
            bytes += 4ull * (unsigned long long)(motif ? deg(v0) : odeg(v0));
        for (int l = 1; l <= lvl && !abort; l++) {
            const int32_t c = ws.jid()[l];
            Lvl &P = ws.lv()[l - 1];
            int pos = lower_bound(P.uid, P.nu, c);
            if (pos >= P.nu || P.uid[pos] != c) {
                fail(3);
                return;
            }
            if (motif) motif_forward(l - 1, c, upm_at(P, pos) & 0x7f);
            else clique_forward(l - 1, pos);
        }
        if (abort) return;
        {
            Lvl &L = ws.lv()[lvl];
            int ne = motif ? L.ne : L.nu;
            L.cur = lo < ne ? lo : ne;
            L.end = hi < ne ? hi : ne;
        }
        int k = lvl;
        while (k >= lvl) {
            if (check_abort()) return;
            Lvl &L = ws.lv()[k];
            if (!motif && K == 3 && triangle_root(L.cur, L.end)) return;
            if (!motif && k == K - 3) {
                clique_leaf_phase(k, L.cur, L.end);
                if (abort) return;
                lds_top = L.mark_lds;
                g_top = L.mark_glb;
                k--;
                continue;
            }
            maybe_donate(k + 1, 0, 0, !motif);
            const int i = uni<W>(L.cur);
            if (i < uni<W>(L.end)) {
                if (motif && k >= K - 4) {
                    // a child makes a leaf node; at k = 3 the root is one, its
                    // children taken a chunk per donation check
                    const bool root = K == 3;
                    const int left = uni<W>(L.end) - i, chunk = motif3_chunk(uni<W>(L.ne));
                    const int to = root ? i + (left < chunk ? left : chunk) : i + 1;
                    L.cur = to;
                    motif_leaf_node(root ? -1 : k, i, root ? i : 0, root ? to : 0x7fffffff);
                    if (abort) return;
                    continue;
                }
                L.cur = i + 1;
                if (motif) {
                    const int32_t c = uni<W>(L.eid[i]);
                    const int pmc = uni<W>(epm_at(L, i));
                    motif_forward(k, c, pmc);
                    if (abort) return;
                    Lvl &N = ws.lv()[k + 1];
                    if (g.gl == 0) bytes += 4ull * (unsigned long long)N.sdeg;
                    N.cur = 0;
                    N.end = N.ne;
                } else {
                    if (g.gl == 0) bytes += 4ull * (unsigned long long)odeg(L.uid[i]);
                    clique_forward(k, i);
                    if (abort) return;
                    Lvl &N = ws.lv()[k + 1];
                    N.cur = 0;
                    N.end = N.nu;
                }
                k++;
            } else {
                lds_top = L.mark_lds;
                g_top = L.mark_glb;
                k--;
            }
        }
    }
};

// ---------------------------------------------------------------------------
// work acquisition

// static queues: one per q_group workers (one per worker when q_group <= 1)
DEV int num_queues(const EnumParams &p) {
    const int gq = p.q_group > 1 ? p.q_group : 1;
    return (p.nworkers + gq - 1) / gq;
}
// jobs of queue w, and where its records start (strided partition, no job
// arrays, one queue per worker: worker w holds roots n-1-w, n-1-w-nworkers, ...)
DEV int queue_jobs(const EnumParams &p, int w, int64_t &base) {
    if (p.sq_jobs == nullptr) {
        base = w;
        return w < p.n ? (int)((p.n - 1 - w) / p.nworkers) + 1 : 0;
    }
    base = p.sq_off[w];
    return (int)(p.sq_off[w + 1] - base);
}

// A static record (root, lo, hi, q) as a job head.
template <int W>
DEV void static_head(const Grp<W> &g, const WorkerLDS &ws, int r, int lo, int hi, int q, JobHead &jh) {
    jh.lvl = 0;
    jh.donated = false;
    jh.shared = lo == -2;  // (root, -2, jobs on the root, q): children from the shared cursor
    jh.range_end = lo == -1 ? hi : 0;
    jh.lo = lo < 0 ? 0 : lo;
    jh.hi = lo == -1 ? 0x7fffffff : hi;
    jh.q = q;
    if (g.gl == 0) ws.jid()[0] = r;
    wsync();
}

// The worker's own queue: all of it is the worker's from the start, taken
// with one atomic (a queue whose block starts late may have lost jobs to
// probe_queues by then); a queue shared by a group is claimed job by job.
template <int W, int MODE>
DEV void open_own_queue(Worker<W, MODE> &wk, int wid) {
    const EnumParams &p = wk.p;
    const bool shared = p.q_group > 1;
    const int w = shared ? wid / p.q_group : wid;
    const int len = queue_jobs(p, w, wk.own_base);
    wk.own_cur = wk.own_end = 0;
    wk.own_queue = shared && len > 0 ? w * p.q_group : -1;
    if (!shared && len > 0) {
        int j = 0;
        if (wk.g.gl == 0) j = atomicAdd(&p.sq_cur[w], len);
        j = wk.g.bcast(j, 0);
        wk.own_cur = j < len ? j : len;
        wk.own_end = len;
    }
}

template <int W, int MODE>
DEV bool take_own(Worker<W, MODE> &wk, JobHead &jh) {
    if (wk.own_cur >= wk.own_end && wk.own_queue >= 0) wk.claim_shared(1);
    if (wk.own_cur >= wk.own_end) return false;
    int32_t t[4];
    wk.static_record(wk.own_base, wk.own_cur++, t);
    static_head<W>(wk.g, wk.ws, uni<W>(t[0]), uni<W>(t[1]), uni<W>(t[2]), uni<W>(t[3]), jh);
    return true;
}

// While blocks of the launch have yet to start (the grid is larger than what
// is resident), nobody hands out their queues: an idle worker looks for a job
// among a random run of queues.
template <int W, int MODE>
DEV bool probe_queues(Worker<W, MODE> &wk, uint32_t &seed, JobHead &jh) {
    const EnumParams &p = wk.p;
    const Grp<W> &g = wk.g;
    const int nq = num_queues(p);
    seed = seed * 1664525u + 1013904223u;
    int w = (int)((seed >> 8) % (uint32_t)nq) + g.gl;
    if (w >= nq) w -= nq;
    int64_t base = 0;
    int len = 0, cur = 0;
    int32_t *const cursor = &p.sq_cur[p.q_group > 1 ? (w < nq ? w : 0) * p.q_group : (w < nq ? w : 0)];
    if (w < nq) {
        len = queue_jobs(p, w, base);
        cur = __hip_atomic_load(cursor, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const uint64_t some = g.ballot(w < nq && cur < len);
    if (!some) return false;
    const int l = __builtin_ctzll(some);
    int32_t t[4] = {0, 0, 0, 0};
    int got = 0;
    if (g.gl == l) {
        const int j = atomicAdd(cursor, 1);
        if (j < len) {
            got = 1;
            wk.static_record(base, j, t);
        }
    }
    if (!g.bcast(got, l)) return false;
    static_head<W>(g, wk.ws, g.bcast(t[0], l), g.bcast(t[1], l), g.bcast(t[2], l), g.bcast(t[3], l), jh);
    return true;
}

// Reads a worker's own slot: 1 with the job its request was answered with, 2
// with static jobs that are now its own queue, 3 when the request was turned
// down, 0 while nothing has come.
template <int W, int MODE>
DEV int poll_slot(Worker<W, MODE> &wk, int wid, uint32_t tag, JobHead &jh) {
    const Grp<W> &g = wk.g;
    const uint64_t *src = wk.p.q[wid].w;
    int v[(kJobWords + W - 1) / W];
    bool mine_ok = true;
#pragma unroll
    for (int r = 0; r < (kJobWords + W - 1) / W; r++) {
        const int j = g.gl + r * W;
        v[r] = 0;
        if (j < kJobWords) {
            uint64_t x = __hip_atomic_load(src + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (!slot_word_of(x, tag)) mine_ok = false;
            v[r] = (int32_t)(uint32_t)x;
        }
    }
    if (g.ballot(!mine_ok) != 0) return 0;
    const int w0 = g.bcast(v[0], 0), w1 = g.bcast(v[0], 1), w2 = g.bcast(v[0], 2), w3 = g.bcast(v[0], 3);
    if (w0 == kNoJob) return 3;
    if (w0 == kStaticJobs) {
        wk.own_base = (int64_t)(((uint64_t)(uint32_t)g.bcast(v[0], 5) << 32) | (uint32_t)g.bcast(v[0], 4));
        wk.own_cur = w1;
        wk.own_end = w2;
        return 2;
    }
#pragma unroll
    for (int r = 0; r < (kJobWords + W - 1) / W; r++) {
        const int j = g.gl + r * W;
        if (j >= 4 && j < kJobWords) wk.ws.jid()[j - 4] = v[r];
    }
    jh.lvl = w0;
    jh.lo = w1;
    jh.hi = w2;
    jh.q = w3;
    jh.range_end = 0;
    jh.donated = true;
    jh.shared = false;
    if (jh.lo < 0) {  // the rest of a range job: roots [jid[0], hi)
        jh.range_end = jh.hi;
        jh.lo = 0;
        jh.hi = 0x7fffffff;
    }
    wsync();
    return 1;
}

// A worker has run out of work.  The last worker of a block closes its mailbox
// and subtracts the block's finished jobs; true when no job of the launch is
// left.
template <int W>
DEV bool go_idle(const EnumParams &p, const Grp<W> &g, BlockLDS *blk) {
    int last = 0;
    if (g.gl == 0) last = atomicSub(&blk->busy, 1) == 1;
    if (!g.bcast(last, 0)) return false;
    if (g.gl < kMailSlots) {
        const unsigned long long rq = atomicExch(p.mail + (size_t)blockIdx.x * kMailStride + g.gl, kMailIdle);
        if (rq != 0 && rq != kMailIdle) {
            uint64_t *const dst = p.q[(uint32_t)rq - 1].w;
            for (int j = 0; j < kRefusalWords; j++)
                __hip_atomic_store(dst + j, slot_word((uint32_t)(rq >> 32), refusal_value(j)), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    int end = 0;
    if (g.gl == 0) {
        const unsigned long long done = atomicExch(&blk->pending, 0u);
        end = done && atomicSub(&p.sc->outstanding, done) == done;
    }
    return g.bcast(end, 0) != 0;
}

// An idle worker has work again.
template <int W>
DEV void go_busy(const EnumParams &p, const Grp<W> &g, BlockLDS *blk) {
    int first = 0;
    if (g.gl == 0) first = atomicAdd(&blk->busy, 1) == 0;
    if (g.bcast(first, 0) && g.gl < kMailSlots)
        (void)atomicCAS(p.mail + (size_t)blockIdx.x * kMailStride + g.gl, kMailIdle, 0ull);
}

// Adds a worker's counts for query `q` to the query's result: the clique count
// (one lane's total) and, in batch launches, the worker's class counters.
template <int W>
DEV void flush_query(const EnumParams &p, const Grp<W> &g, int q, unsigned long long count,
                     unsigned long long *whist, unsigned long long last_ticks) {
    if (q < 0) return;
    const QueryDesc &Q = p.qd[q];
    if (g.gl == 0 && count && !Q.motif) atomicAdd(&Q.out[0], count);
    if (g.gl == 0 && Q.done_ticks && last_ticks) atomicMax(Q.done_ticks, last_ticks);
    if (p.nq > 1 && Q.motif) {
        for (int i = g.gl; i < Q.ncls; i += W) {
            unsigned long long v = whist[i];
            if (v) {
                atomicAdd(&Q.out[i], v);
                whist[i] = 0;
            }
        }
        wsync();
    }
}

// MODE 0: cliques, 1: motifs; WAVES: the waves per SIMD the registers are
// budgeted for.
template <int W, int MODE, int WAVES = min_waves<W, MODE>()>
__global__ __launch_bounds__(kThreads, WAVES) void enum_kernel(EnumParams p) {
    extern __shared__ __align__(16) char smem[];
    Grp<W> g;
    const int nthr = (int)blockDim.x;  // 64, 128 or 256
    const int wpb = nthr / W;
    const int wib = uni<W>(threadIdx.x / W);
    const int wid = blockIdx.x * wpb + wib;
    // LDS: block record | single-query class counters of the block | per-worker records |
    // per-worker class counters (batch) | per-worker stack slices
    const bool single = p.nq == 1;
    const int bslots = single && p.qd[0].motif ? (p.qd[0].ncls + 1) & ~1 : 0;
    const int wslots = single ? 0 : (p.hist_slots + 1) & ~1;
    const size_t wsb = worker_lds_bytes(p.kmax);
    BlockLDS *const blk = (BlockLDS *)smem;
    unsigned long long *bhist = (unsigned long long *)(smem + sizeof(BlockLDS));
    char *base = smem + sizeof(BlockLDS) + (size_t)bslots * 8;
    const WorkerLDS ws = worker_lds(base + wib * wsb, p.kmax);
    base += wpb * wsb;
    unsigned long long *whist = (unsigned long long *)base + (size_t)wib * wslots;
    base += (size_t)wpb * wslots * 8;
    char *slice = base + (int64_t)wib * p.lds_per_worker;
    for (int i = threadIdx.x; i < bslots; i += nthr) bhist[i] = 0;
    for (int i = threadIdx.x; i < wpb * wslots; i += nthr) ((unsigned long long *)(smem + sizeof(BlockLDS) + (size_t)bslots * 8 + wpb * wsb))[i] = 0;
    if (threadIdx.x == 0) {
        const unsigned long long t = wall_clock64();
        atomicAdd(&p.sc->started, 1);
        const int left = p.nworkers - (int)blockIdx.x * wpb;
        blk->busy = left < wpb ? left : wpb;
        blk->pending = 0;
        for (int i = 0; i < kMailSlots; i++)
            __hip_atomic_store(p.mail + (size_t)blockIdx.x * kMailStride + i, 0ull, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        atomicMin(&p.sc->st[blockIdx.x % kStatCopies].t_start, t);
        if (p.start_ticks) atomicMin(p.start_ticks, t);
    }
    __syncthreads();

    unsigned long long bytes = 0;
    if (wid < p.nworkers) {
        if (g.gl == 0)
            for (int i = 0; i < kStats; i++) ws.st()[i] = 0;
        wsync();
        Worker<W, MODE> wk(p, ws, single ? bhist : whist, slice, blk, wid);
        uint32_t seed = 0x9E3779B9u * (uint32_t)(wid + 1);
        bool idle = false, all_started = false;
        uint32_t seq = 0;  // requests of this launch
        int asked = -1;    // mailbox word that holds this worker's request
        int waited = 0;    // time since it was written, in sleeps
        // sleeps of the next round, the most of a round now, rounds at that many
        int backoff = 1, most = 4, dry = 0;
        uint32_t spins = 0;
        const bool can_ask = (uint32_t)wid < p.q_cap;
        open_own_queue(wk, wid);
        while (true) {
            JobHead jh;
            bool got = take_own(wk, jh);
            if (!got) {
                if (!idle) {
                    idle = true;
                    if (g.gl == 0 && !ws.st()[kStStatic]) ws.st()[kStStatic] = wall_clock64();
                    if (go_idle<W>(p, g, blk)) {
                        // the last job is done: tell every block
                        for (unsigned b = g.gl; b < gridDim.x; b += W)
                            __hip_atomic_store(wk.mailbox(b) + kMailOver, (unsigned long long)wk.epoch,
                                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        break;
                    }
                }
                const uint32_t tag = request_tag(wk.epoch, seq);
                if (asked >= 0) {
                    const int r = poll_slot(wk, wid, tag, jh);
                    if (r) {
                        asked = -1;
                        seq++;
                    }
                    got = r == 1;
                    if (r == 2) got = take_own(wk, jh);
                    // no answer for long: ask elsewhere (unless it is coming)
                    waited += backoff;
                    if (r == 0 && waited >= 96) {
                        int back = 0;
                        const unsigned long long rq = ((unsigned long long)tag << 32) | (uint32_t)(wid + 1);
                        if (g.gl == 0) back = atomicCAS(p.mail + asked, rq, 0ull) == rq;
                        waited = 0;
                        if (g.bcast(back, 0)) asked = -1;
                    }
                } else if (can_ask) {
                    // a random word of a random block's mailbox; a block without
                    // work, or another request there, says so at once
                    const unsigned long long rq = ((unsigned long long)tag << 32) | (uint32_t)(wid + 1);
                    for (int a = 0; a < (W > 16 ? W / 16 : 1) && asked < 0; a++) {
                        seed = seed * 1664525u + 1013904223u;
                        const int b = (int)((seed >> 8) % gridDim.x) * kMailStride + (int)(seed >> 29);
                        int in = 0;
                        if (g.gl == 0) in = atomicCAS(p.mail + b, 0ull, rq) == 0ull;
                        if (g.bcast(in, 0)) {
                            asked = b;
                            waited = 0;
                            backoff = 1;
                        }
                    }
                }
            }
            if (!got) {
                ++spins;
                // the end of the launch; rarely: another worker's failure,
                // blocks that have yet to start
                unsigned long long over = 0;
                int err = 0;
                if (g.gl == 0) {
                    over = __hip_atomic_load(wk.mailbox(blockIdx.x) + kMailOver, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if ((spins & 63) == 0)
                        err = __hip_atomic_load(&p.sc->error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                if (g.bcast64(over, 0) == wk.epoch || g.bcast(err, 0)) break;
                if (!all_started && (spins & 15) == 0) {
                    int st = 0;
                    if (g.gl == 0) st = __hip_atomic_load(&p.sc->started, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    all_started = g.bcast(st, 0) >= (int)gridDim.x;
                    if (!all_started) got = probe_queues(wk, seed, jh);
                }
            }
            if (!got) {
                if (p.watchdog_ticks && now_ticks() - wk.t_start > p.watchdog_ticks) {
                    if (g.gl == 0) atomicCAS(&p.sc->error, 0, 1);
                    break;
                }
                // sleep only when no lane of this wave has work: s_sleep
                // stalls the whole wave, including busy narrower workers.  The
                // longer nothing comes the longer: the polls and requests of
                // thousands of idle waves slow the few busy ones' loads (with
                // sleeps of 4 x 512 cycles at most R-MAT s15 k = 5 with bitmaps
                // and stealing off 129 ms, 73 so; Chung-Lu 1,000 k = 6 without
                // stealing 14.6 -> 11.6).  A step every 64 rounds, so sleeps stay
                // a few percent of the time idle (every 16: R-MAT s17 k = 6 2.53
                // -> 2.72 ms; every 64 2.56).  Narrow workers sleep longer and ask
                // fewer at a time, as there are more of them to a wave (R-MAT s15
                // k = 3 with lists, 8 lanes, 2.4 -> 1.7 ms; k = 5, 16 lanes, 2.01 ->
                // 1.84).
                if (__ballot(1) == ~0ull) {
                    for (int b = 0; b < backoff * (64 / W); b++) __builtin_amdgcn_s_sleep(8);
                    if (backoff < most) {
                        backoff *= 2;
                    } else if (++dry >= 64 && most < 256) {
                        dry = 0;
                        most *= 2;
                    }
                }
                continue;
            }
            if (idle) {
                idle = false;
                go_busy<W>(p, g, blk);
            }
            backoff = 1, most = 4, dry = 0;
            const int jq = job_query(jh.q);
            bool ok = jh.q >= 0 && jq < p.nq;
            int merged = 0;  // further jobs done with this one
            // the job's own donation threshold travels with its query word
            // to every piece it gives away
            wk.qword = jh.q;
            wk.from = jh.donated && jh.lvl <= 1 && !jh.range_end ? uni<W>(ws.jid()[kJobPub - 4]) : 0;
            wk.job_sm = job_steal_min(jh.q) >= 2 ? job_steal_min(jh.q) : p.steal_min;
            if (ok && jq != wk.qid) {
                if (!single) flush_query<W>(p, g, wk.qid, ws.st()[kStQCount], whist, ws.st()[kStLast]);
                if (g.gl == 0) ws.st()[kStQCount] = 0;
                const QueryDesc &Q = p.qd[jq];
                wk.qid = jq;
                wk.K = uni<W>(Q.K);
                wk.qmotif = uni<W>(Q.motif) != 0;
                wk.lut = unil<W>(Q.lut);
                ok = (MODE == 1) == wk.qmotif && Q.K >= 2 && Q.K <= p.kmax;
            }
            const int lvl_max = wk.K == 2 ? 0 : wk.K - 3;
            const int r0 = uni<W>(ws.jid()[0]);
            const int r1 = jh.range_end > 0 ? jh.range_end : r0 + 1;
            if (!ok || jh.lvl < 0 || jh.lvl > lvl_max || r0 < 0 || r1 > p.n || r0 >= r1) {
                wk.fail(3);
            } else {
                wk.range_hi = r1;
                for (int root = r0; root < wk.range_hi && !wk.abort; root++) {
                    if (jh.range_end > 0) {
                        // range jobs skip roots without a neighbour above them;
                        // a motif root still counts its own node's bytes
                        if (p.off[root + 1] - p.ostart[root] <= 0) {
                            if (wk.qmotif && g.gl == 0)
                                wk.bytes += 4ull * (unsigned long long)(p.off[root + 1] - p.off[root]);
                            continue;
                        }
                        ws.jid()[0] = root;
                        wsync();
                    }
                    int32_t lv = 0;
                    int ld = 0;
                    bool light = false;
                    if constexpr (MODE == 0) {
                        light = wk.collect_light(jh, root, merged, lv, ld);
                    }
                    // the job's start time goes through LDS: nothing of the
                    // bookkeeping stays live in registers across the DFS
                    if (g.gl == 0) {
                        if (!ws.st()[kStFirst]) ws.st()[kStFirst] = wall_clock64();
                        ws.st()[kStT0] = __builtin_amdgcn_s_memtime();
                    }
                    if (light) wk.light_roots(lv, ld);
                    else wk.run_job(jh.lvl, jh.lo, jh.hi,
                               !jh.shared && (jh.range_end > 0 || (!jh.donated && jh.lvl == 0 && jh.lo == 0)),
                               jh.shared);
                    unsigned long long jc = g.lsum(wk.cnt);
                    if (g.gl == 0) {
                        const unsigned long long dt = __builtin_amdgcn_s_memtime() - ws.st()[kStT0];
                        ws.st()[kStQCount] += jc;
                        ws.st()[kStBusy] += dt;
                        if (dt > ws.st()[kStJobMax]) ws.st()[kStJobMax] = dt;
                        ws.st()[kStLast] = wall_clock64();
                        if (p.root_cost) atomicAdd(&p.root_cost[root], dt);
                        if (p.root_count && jc) atomicAdd(&p.root_count[root], jc);
                    }
                }
            }
            if (g.gl == 0) {
                ws.st()[kStJobs] += 1 + merged;
                atomicAdd(&blk->pending, 1u + (unsigned)merged);
            }
            if (wk.abort) break;
        }
        wsync();
        if (!single) flush_query<W>(p, g, wk.qid, ws.st()[kStQCount], whist, ws.st()[kStLast]);
        bytes = g.lsum(wk.bytes);
    }
    __syncthreads();
    // a single query's results: one of res_copies copies per block, so that
    // the blocks do not all queue up for the same words
    unsigned long long *const out = p.qd[0].out + (size_t)(blockIdx.x % (unsigned)p.res_copies) * p.res_stride;
    if (single && bslots) {
        for (int i = threadIdx.x; i < p.qd[0].ncls; i += nthr)
            if (bhist[i]) atomicAdd(&out[i], bhist[i]);
    }
    // Per-worker statistics (held by lane 0 of each worker) reduced over the
    // block, so that each block, not each worker, adds to the shared words.
    // The reduction reuses the start of the block's dynamic LDS (at least the
    // worker records, > 88 B per wave): a static array would count towards
    // the LDS that decides how many blocks share a CU.  Fields 0-4 and 10 are
    // sums, the others maxima.
    constexpr int NF = 11;
    unsigned long long (*red)[NF] = (unsigned long long (*)[NF])smem;
    const bool holder = wid < p.nworkers && g.gl == 0;
    const unsigned long long *st = ws.st();
    unsigned long long f[NF] = {holder ? bytes : 0ull,          holder ? st[kStJobs] : 0ull,
                                holder ? st[kStBusy] : 0ull,    holder ? st[kStDonated] : 0ull,
                                holder && single ? st[kStQCount] : 0ull,
                                holder ? st[kStBusy] : 0ull,    holder ? st[kStFirst] : 0ull,
                                holder ? st[kStStatic] : 0ull,  holder ? st[kStLast] : 0ull,
                                holder ? st[kStJobMax] : 0ull,
                                holder && st[kStJobs] ? 1ull : 0ull};
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
#pragma unroll
        for (int i = 0; i < NF; i++) {
            const unsigned long long y = __shfl_xor(f[i], o, 64);
            f[i] = i < 5 || i == 10 ? f[i] + y : (y > f[i] ? y : f[i]);
        }
    }
    // every wave has read its records (and the class counters were flushed)
    // before the reduction overwrites them
    __syncthreads();
    if (__lane_id() == 0) {
#pragma unroll
        for (int i = 0; i < NF; i++) red[threadIdx.x / 64][i] = f[i];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < nthr / 64; w++) {
            for (int i = 0; i < NF; i++)
                f[i] = i < 5 || i == 10 ? f[i] + red[w][i] : (red[w][i] > f[i] ? red[w][i] : f[i]);
        }
        SchedStats &st = p.sc->st[blockIdx.x % kStatCopies];
        if (f[0]) atomicAdd(&st.alg_bytes, f[0]);
        if (f[1]) atomicAdd(&st.jobs, f[1]);
        if (f[2]) atomicAdd(&st.busy_sum, f[2]);
        if (f[3]) atomicAdd(&st.donations, f[3]);
        if (f[4] && single && !p.qd[0].motif) atomicAdd(&out[0], f[4]);
        atomicMax(&st.busy_max, f[5]);
        atomicMax(&st.t_first_job, f[6]);
        atomicMax(&st.t_static_done, f[7]);
        atomicMax(&st.t_last_job, f[8]);
        atomicMax(&st.job_max, f[9]);
        if (f[10]) atomicAdd(&st.active_workers, f[10]);
        atomicMax(&st.t_exit, (unsigned long long)wall_clock64());
    }
}

// Local bitmaps of the launch's prebuilt roots, one block per root, in the
// layout clique_bitmap_root reads: rows (d x NW uint64, row i bit j set when
// L[j] is in N+(L[i]), L = N+(v)) then the out-degrees of L (d int32).  The
// host lists only roots with out-degree <= 256.
// threads per block of the bitmap pre-pass: the largest bitmaps (256 rows of
// up to a few hundred entries) finish sooner with more waves on their rows
// (R-MAT s17, 1,830 roots: 256 threads 94 us, 512 81 us, 1024 89 us)
constexpr int kPrebuildThreads = 512;
__global__ __launch_bounds__(kPrebuildThreads) void prebuild_kernel(EnumParams p) {
    __shared__ int32_t hkey[512];
    __shared__ uint8_t hval[512];
    __shared__ int64_t rst[256];
    __shared__ int32_t spre[257];
    __shared__ int32_t wsum[kPrebuildThreads / 64];
    __shared__ unsigned long long srows[256 * 4];
    // the roots are ascending by degree rank: the largest bitmaps (last) are
    // built by the first blocks, so they do not start last and set the tail
    const int b = p.npre - 1 - (int)blockIdx.x, tid = threadIdx.x;
    if (b < 0) return;
    const int32_t v = p.pre_roots[b];
    const int d = (int)(p.off[v + 1] - p.ostart[v]);
    if (d > 256) return;
    const int NW = d <= 64 ? 1 : d <= 128 ? 2 : 4;
    const int HB = NW == 1 ? 7 : NW == 2 ? 8 : 9;
    const int HS = 1 << HB;
    const int32_t *L = p.adj + p.ostart[v];
    uint64_t *rows = (uint64_t *)const_cast<char *>(p.pre + p.pre_offs[b]);
    int32_t *gdp = (int32_t *)(rows + (int64_t)d * NW);
    for (int t = tid; t < HS; t += blockDim.x) hkey[t] = -1;
    // one child per thread (d <= 256 <= blockDim.x): its list start, its
    // out-degree and the block-wide exclusive prefix of the out-degrees
    int od = 0;
    if (tid < d) {
        const int32_t u = L[tid];
        const int64_t os = p.ostart[u];
        rst[tid] = os;
        od = (int)(p.off[u + 1] - os);
        gdp[tid] = od;
    }
    int incl = od;  // inclusive scan within the wave
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(incl, o, 64);
        if ((tid & 63) >= o) incl += y;
    }
    if ((tid & 63) == 63) wsum[tid >> 6] = incl;
    for (int t = tid; t < d * NW; t += blockDim.x) srows[t] = 0;
    __syncthreads();
    int wbase = 0;
    for (int w = 0; w < (tid >> 6); w++) wbase += wsum[w];
    if (tid < d) spre[tid + 1] = wbase + incl;
    if (tid == 0) spre[0] = 0;
    for (int j = tid; j < d; j += blockDim.x) {
        const int32_t key = L[j];
        uint32_t h = ((uint32_t)key * 2654435761u) >> (32 - HB);
        while (atomicCAS(&hkey[h], -1, key) != -1) h = (h + 1) & (HS - 1);
        hval[h] = (uint8_t)j;
    }
    __syncthreads();
    // each wave takes whole rows (child a's out-list, every 4th row) and its
    // lanes stride the list, U loads in flight per lane: coalesced reads and
    // no search for the row of an element; bits go into the LDS rows
    const int wv = tid >> 6, ln = tid & 63;
    constexpr int U = 4;
    for (int a = wv; a < d; a += kPrebuildThreads / 64) {
        const int64_t base = rst[a];
        const int len = spre[a + 1] - spre[a];
        for (int e0 = 0; e0 < len; e0 += U * 64) {
            int32_t xs[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int e = e0 + u * 64 + ln;
                xs[u] = e < len ? p.adj[base + e] : -1;
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int32_t x = xs[u];
                if (x < 0) continue;
                uint32_t h = ((uint32_t)x * 2654435761u) >> (32 - HB);
                int k;
                while ((k = hkey[h]) != x && k != -1) h = (h + 1) & (HS - 1);
                if (k == x) {
                    const int j = hval[h];
                    atomicOr(&srows[a * NW + (j >> 6)], 1ull << (j & 63));
                }
            }
        }
    }
    __syncthreads();
    for (int t = tid; t < d * NW; t += blockDim.x) rows[t] = srows[t];
}

int prebuild_launch(const EnumParams &p, void *stream) {
    if (p.npre <= 0) return DM_OK;
    hipLaunchKernelGGL(prebuild_kernel, dim3(p.npre), dim3(kPrebuildThreads), 0, (hipStream_t)stream, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(DM_ERR_HIP, "prebuild launch: %s", hipGetErrorString(e));
    return DM_OK;
}

__global__ void fill_u32_kernel(uint32_t *ptr, uint32_t value, size_t count) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < count; i += stride) ptr[i] = value;
}

// Resets the scheduler state of a launch; graph-capturable (no memset or
// host copies).  Clears the job slots, so that nothing an earlier launch left
// there matches a request, whatever the epoch (16 bytes a thread: 0.8 MB for
// 6,144 workers).
__global__ void enum_init_kernel(SchedCounters *sc, unsigned long long njobs, int32_t *epoch, int32_t *sq_cur,
                                 int nworkers, unsigned long long *results, size_t nresults,
                                 unsigned long long *done_ticks, int nq, unsigned long long *start_ticks,
                                 unsigned long long *mail, int blocks, Job *q, int slots) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    if (i == 0) {
        sc->outstanding = njobs;
        sc->started = 0;
        sc->error = 0;
        *epoch = *epoch + 1;
        if (start_ticks) *start_ticks = ~0ull;
    }
    for (size_t t = i; t < kStatCopies; t += stride) {
        SchedStats z{};
        z.t_start = ~0ull;
        sc->st[t] = z;
    }
    // no block takes requests before it has begun; the launch is not over
    for (size_t t = i; t < (size_t)blocks * kMailStride; t += stride)
        mail[t] = t % kMailStride < kMailSlots ? kMailIdle : 0;
    for (size_t t = i; t < (size_t)nworkers; t += stride) sq_cur[t] = 0;
    for (size_t t = i; t < (size_t)slots * sizeof(Job) / 16; t += stride) ((ulong2 *)q)[t] = ulong2{0, 0};
    for (size_t t = i; t < nresults; t += stride) results[t] = 0;
    if (done_ticks)
        for (size_t t = i; t < (size_t)nq; t += stride) done_ticks[t] = 0;
}

// ---------------------------------------------------------------------------
size_t enum_lds_bytes(int vwave, int threads, int kmax, int ncls_single, int hist_slots, int lds_per_worker) {
    int wpb = threads / vwave;
    size_t b = sizeof(BlockLDS) + (size_t)((ncls_single + 1) & ~1) * 8;
    b += (size_t)wpb * worker_lds_bytes(kmax);
    b += (size_t)wpb * (size_t)((hist_slots + 1) & ~1) * 8;
    b += (size_t)wpb * lds_per_worker;
    return b;
}

// launch modes: 0 cliques, 1 motifs, 2 motifs of sizes 5 and 6 (the
// full-wave motif kernel at kDeepMotifWaves; narrower widths keep mode 1's)
template <int W>
static const void *kernel_mode(int mode) {
    switch (mode) {
        case 0: return (const void *)enum_kernel<W, 0>;
        case 1: return (const void *)enum_kernel<W, 1>;
        case 2:
            if constexpr (W == 64) return (const void *)enum_kernel<W, 1, kDeepMotifWaves>;
            else return (const void *)enum_kernel<W, 1>;
        default: return nullptr;
    }
}

static const void *kernel_for(int vwave, int mode) {
    switch (vwave) {
        case 8: return kernel_mode<8>(mode);
        case 16: return kernel_mode<16>(mode);
        case 32: return kernel_mode<32>(mode);
        case 64: return kernel_mode<64>(mode);
        default: return nullptr;
    }
}

static bool threads_ok(int threads) { return threads == 64 || threads == 128 || threads == 256; }

int enum_occupancy(int vwave, int mode, int threads, size_t lds, int *blocks_per_cu) {
    const void *k = kernel_for(vwave, mode);
    if (!k || !threads_ok(threads) || threads < vwave) return set_error(DM_ERR_ARG, "unsupported launch shape");
    if (lds > 160 * 1024) return set_error(DM_ERR_ARG, "LDS request %zu exceeds 160 KiB", lds);
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return set_error(DM_ERR_HIP, "hipFuncSetAttribute: %s", hipGetErrorString(e));
    }
    int nb = 0;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k, threads, lds);
    if (e != hipSuccess) return set_error(DM_ERR_HIP, "occupancy query: %s", hipGetErrorString(e));
    // The query divides the CU's 160 KiB by the dynamic size alone.  gfx950
    // allocates a block's LDS, static and dynamic together, in 1280-byte
    // units (measured: 53,760 B per block keeps 3 blocks on a CU, 53,761 B
    // leaves 2), so a persistent launch sized by the query alone would hold
    // blocks that only become resident once others have exited.
    constexpr size_t kLdsGranule = 1280;
    static std::atomic<int> static_lds[4][4] = {};  // + 1: 0 = not read yet
    const int vi = vwave == 8 ? 0 : vwave == 16 ? 1 : vwave == 32 ? 2 : 3;
    int sl = static_lds[vi][mode].load(std::memory_order_relaxed) - 1;
    if (sl < 0) {
        hipFuncAttributes fa{};
        e = hipFuncGetAttributes(&fa, k);
        if (e != hipSuccess) return set_error(DM_ERR_HIP, "hipFuncGetAttributes: %s", hipGetErrorString(e));
        sl = (int)fa.sharedSizeBytes;
        static_lds[vi][mode].store(sl + 1, std::memory_order_relaxed);
    }
    const size_t per_block = (lds + (size_t)sl + kLdsGranule - 1) / kLdsGranule * kLdsGranule;
    const int fit = (int)((size_t)160 * 1024 / per_block);
    *blocks_per_cu = nb < fit ? nb : fit;
    return DM_OK;
}

int enum_launch(const EnumParams &p, int mode, int vwave, int blocks, int threads, size_t lds, void *stream) {
    const void *k = kernel_for(vwave, mode);
    if (!k || !threads_ok(threads) || threads < vwave) return set_error(DM_ERR_ARG, "unsupported launch shape");
    EnumParams copy = p;
    void *args[] = {&copy};
    hipError_t e = hipLaunchKernel(k, dim3(blocks), dim3(threads), args, lds, (hipStream_t)stream);
    if (e != hipSuccess) return set_error(DM_ERR_HIP, "enum launch: %s", hipGetErrorString(e));
    return DM_OK;
}

int enum_init_launch(const EnumParams &p, unsigned long long njobs, int32_t *epoch, unsigned long long *results,
                     size_t nresults, unsigned long long *done_ticks, int nq, int launch_blocks, void *stream) {
    const int slots = (int)std::min<int64_t>(p.nworkers, p.q_cap);
    size_t work = std::max<size_t>({(size_t)slots * sizeof(Job) / 16, (size_t)p.nworkers, nresults, (size_t)nq, (size_t)1});
    int blocks = (int)std::min<size_t>((work + 255) / 256, 1024);
    hipLaunchKernelGGL(enum_init_kernel, dim3(blocks), dim3(256), 0, (hipStream_t)stream, p.sc, njobs, epoch, p.sq_cur,
                       p.nworkers, results, nresults, done_ticks, nq, p.start_ticks, p.mail, launch_blocks, p.q,
                       slots);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(DM_ERR_HIP, "init launch: %s", hipGetErrorString(e));
    return DM_OK;
}

SchedStats sched_totals(const SchedCounters &c) {
    SchedStats t = c.st[0];
    for (int i = 1; i < kStatCopies; i++) {
        const SchedStats &s = c.st[i];
        t.donations += s.donations;
        t.jobs += s.jobs;
        t.alg_bytes += s.alg_bytes;
        t.busy_sum += s.busy_sum;
        t.active_workers += s.active_workers;
        t.busy_max = std::max(t.busy_max, s.busy_max);
        t.job_max = std::max(t.job_max, s.job_max);
        t.t_start = std::min(t.t_start, s.t_start);
        t.t_first_job = std::max(t.t_first_job, s.t_first_job);
        t.t_static_done = std::max(t.t_static_done, s.t_static_done);
        t.t_last_job = std::max(t.t_last_job, s.t_last_job);
        t.t_exit = std::max(t.t_exit, s.t_exit);
    }
    return t;
}

int fill_u32_launch(void *ptr, uint32_t value, size_t count, void *stream) {
    if (count == 0) return DM_OK;
    int blocks = (int)((count + 255) / 256);
    if (blocks > 1024) blocks = 1024;
    hipLaunchKernelGGL(fill_u32_kernel, dim3(blocks), dim3(256), 0, (hipStream_t)stream,
                       (uint32_t *)ptr, value, count);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(DM_ERR_HIP, "fill launch: %s", hipGetErrorString(e));
    return DM_OK;
}

}  // namespace dm
