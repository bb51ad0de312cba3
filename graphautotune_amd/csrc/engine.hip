// MI355X (gfx950) subgraph pattern-matching engine.
//
// One persistent launch runs every pattern of a plan. Each wavefront (64
// lanes) takes a chunk of directed edges from a global work queue; an edge
// (v0 -> v1) fixes the first two pattern vertices, and the wave walks the
// plan's trie depth-first from there:
//   * non-leaf levels take one candidate at a time; their prefix sets are
//     intersections computed by all 64 lanes (stream one sorted list,
//     binary-search the other, compact with ballot + mbcnt) into LDS;
//   * leaf levels count every candidate at once: the (candidate, element)
//     pairs of all candidates form one flattened index space that the lanes
//     sweep 64 at a time, finding their owner candidate with ds_bpermute and
//     crediting hits with ballot + popcount, so lane utilisation does not
//     depend on set sizes. The IEP tail is then combined per candidate.
// Counts are exact uint64 (modular arithmetic for the signed IEP terms).
// A task whose intersection could outgrow its LDS buffer is abandoned and
// queued for a second launch that keeps the same buffers in HBM.
//
// Replaces the six-kernel host-recursive executor of the reference
// (include/engine/engine.cuh:232-428, include/engine/engine_kernel.cuh).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdio>
#include <cstring>
#include <numeric>
#include <set>
#include <type_traits>
#include <vector>

#include "handles.hpp"
#include "kept.h"
#include "plan_dev.h"

namespace gatk {

constexpr int W = 64;
constexpr int kSplitLevels = 3;  // LDS subtask levels (see KArgs)
constexpr int kLevelsHbm = kSplitLevels + 1;  // timeline id of the HBM launch (its subtasks: + 1)

// A split subtask: candidates [lo, hi) of the loop of node `node` (at depth
// `depth` >= 2) below root edge `edge` (directed edge index: v0 = its row,
// v1 = its entry), with the candidates of depths 2 .. depth-1 taken from
// loop positions pos[2 ..]. lo >= hi marks an empty or cancelled entry. With
// pos[0] = k + 1 the range is not one of the loop but of the father of the
// node's KEEP_SUM op k (leaf_sum).
struct SplitTask {
    long long edge;
    int node, depth, lo, hi;
    int pos[GATP_MAX_DEPTH];
};

struct KArgs {
    const long long *off;
    const int *adj;
    const int *split;  // split[v] = number of neighbours of v below v
    int n;
    long long m;
    long long e_lo, e_hi;        // root edges of this count: [e_lo, e_hi)
    const GatPlanDev *plan;
    unsigned long long *counts;  // kCountCopies copies of [GATP_MAX_TERMS]
    unsigned long long *queue;   // heads of the launches' queues (see queue_next)
    unsigned int *drained;       // [queue] set once a wave has found the queue empty
    long long *ovf;              // overflow task starts
    unsigned long long *ovf_n;   // overflow task count
    long long ovf_cap;
    int *gstore;                 // HBM set buffers (overflow launch)
    unsigned long long *bytes;   // W_alg accumulator
    unsigned int *err;           // device error flags
    int cap;                     // entries per buffer of an intersection
    int stage_cap;               // entries per buffer of a staged neighbour list
    long long store_off[GATP_MAX_STORE];  // first entry of each set buffer
    int state_bytes;             // LDS of a wave before its set buffers
    int chunk;
    int lin_thr;
    int gallop_ratio;
    int strategy;
    int account;
    // Dense neighbourhood bitmaps of high-degree vertices ("hubs"): row h
    // holds bit x set iff x is a neighbour of hub h. hub_map == nullptr means
    // the graph is degree-ordered and the hubs are vertices [0, n_hubs); else
    // it gives a vertex's row, or -1, and rows from n_hubs on are not used.
    const unsigned *hub_bits;
    const int *hub_map;
    long long hub_words;  // words per row: (n + 31) / 32
    int n_hubs;
    // Splitting: a task that has run longer than split_ticks of the wall
    // clock while the queue it came from is drained hands the rest of its
    // shallowest unfinished loop at depth >= 2 to subs[out_base ..] (count in
    // *out_n, at most out_cap used). The main launch makes level-1 subtasks;
    // the launch of level k (sub_mode k, LDS buffers) runs them and may split
    // into level k + 1, up to level kSplitLevels, which does not split.
    // Subtasks that outgrow LDS are copied to the HBM list
    // (subs[sovf_base ..], count *sovf_n), which also takes the splits of the
    // HBM launch; a last subtask launch with HBM buffers (sub_mode
    // kSplitLevels + 1) runs it.
    int sub_mode;
    SplitTask *subs;
    unsigned long long *in_n, *out_n, *sovf_n;
    long long in_base, out_base, sovf_base;
    long long in_cap, out_cap, sovf_cap;
    long long split_ticks;  // <= 0: no splitting
    // Kept COUNT values (GATP_KEEP_*), null without. A leaf's |N(c) ∩ father|
    // is the same for every path that ends in c while the father stays, and
    // there are many (R-MAT s13's C5: 1.3e9 paths over 6.7e7 pairs of vertices).
    // edge_tab[k][e] is the value of directed edge e with truncation k, or -1.
    // Pool i holds tables of tab_size entries from pool + i pool_tables
    // tab_size on; key x uses table x % pool_tables, whose entry c holds the tag
    // x + 1, the value and the epoch for the key that wrote it last. Every count has its
    // own epoch, so nothing of an earlier one is taken. One pool for all waves:
    // with a table per wave the subtasks of one root each filled their own (before
    // the pair sweep C5 108 ms instead of 56, house on Chung-Lu 65,536 46 instead of 36).
    KeptEdge *edge_tab[4];
    KeptEntry *pool;
    unsigned pool_tables;
    int tab_size;
    unsigned epoch;
    int keep;  // this count uses the tables
    // Timeline (GAT_FLAG_TIMELINE): one record of kTlFields int64 per wave
    // at tl + kTlFields * (tl_base + wave), or none when tl is null.
    long long *tl;
    int tl_base;
};

// Timeline record: launch id, unit (wave or workgroup), wall-clock start and
// end, shader cycles spent building rows and counting (clique store), items
// taken from the queue, and pairs counted (clique store).
constexpr int kTlFields = 8;
__device__ __forceinline__ void tl_write(long long *tl, int idx, int launch, int unit, long long t0, long long t1,
                                         long long build, long long count, long long items, long long pairs) {
    long long *r = tl + (long long)kTlFields * idx;
    r[0] = launch;
    r[1] = unit;
    r[2] = t0;
    r[3] = t1;
    r[4] = build;
    r[5] = count;
    r[6] = items;
    r[7] = pairs;
}

// Subtask blocks a task may hand on between commits. A batched plan's trie
// starts a loop for every child node of a candidate, and once a task is due
// to split each such loop goes to the next split launch with one record.
constexpr int kMaxDonations = 64;

struct WaveState {
    unsigned long long task_acc[GATP_MAX_TERMS];
    unsigned long long wave_acc[GATP_MAX_TERMS];
    long long sbeg[GATP_MAX_SLOTS];
    int slen[GATP_MAX_SLOTS];
    int staged[GATP_MAX_SLOTS];  // neighbour list copied into its LDS buffer
    int val[GATP_MAX_DEPTH + 1];
    int f_node[GATP_MAX_DEPTH + 1];
    int f_cur[GATP_MAX_DEPTH + 1];
    int f_hi[GATP_MAX_DEPTH + 1];
    unsigned long long bytes;   // committed W_alg of this wave
    unsigned long long ebytes;  // W_alg of the work not yet committed
    long long t0;               // wall clock at the start of the task
    long long f_t0[GATP_MAX_DEPTH + 1];  // and of the frames above the leaves (see rest_is_long)
    long long rb;               // first edge of the task's root v0
    long long sub_edge;         // root edge of the running subtask, or -1
    long long don_base[kMaxDonations];  // subtask blocks donated since the last commit
    int don_cnt[kMaxDonations];
    int n_don;
    int base_depth;             // frames exist from this depth on (2, or a subtask's depth)
    int base_lo;                // first position of that depth's frame
    int path_pos[GATP_MAX_DEPTH + 1];  // a subtask's positions at depths 2 .. base_depth-1
    int abort;
    int ex_in[GATP_MAX_LEAF_OPS];  // leaf: excluded levels whose vertex lies in the op's father
    int leafcnt[GATP_MAX_LEAF_OPS][W];  // last: only the plan's max_leaf_ops rows are allocated
};

__device__ __forceinline__ int lane_id() { return __lane_id(); }
__device__ __forceinline__ unsigned long long ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }
__device__ __forceinline__ int mbcnt(unsigned long long m) {
    return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}
__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ long long uni64(long long x) {
    const int lo = __builtin_amdgcn_readfirstlane((int)(unsigned)(x & 0xffffffffll));
    const int hi = __builtin_amdgcn_readfirstlane((int)(x >> 32));
    return (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ int bperm(int x, int src) { return __builtin_amdgcn_ds_bpermute(src << 2, x); }
__device__ __forceinline__ long long bperm64(long long x, int src) {
    const int lo = bperm((int)(x & 0xffffffffll), src), hi = bperm((int)(x >> 32), src);
    return (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}
// Reads of one lane's registers by the whole wave: LanePull for a lane index
// that is the same in every lane (v_readlane, no LDS crossbar), PermPull for
// a per-lane index (ds_bpermute).
struct LanePull {
    int s;
    __device__ __forceinline__ int operator()(int x) const { return __builtin_amdgcn_readlane(x, s); }
    __device__ __forceinline__ long long operator()(long long x) const {
        const int lo = __builtin_amdgcn_readlane((int)(x & 0xffffffffll), s);
        const int hi = __builtin_amdgcn_readlane((int)(x >> 32), s);
        return (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
    }
};
struct PermPull {
    int s;
    __device__ __forceinline__ int operator()(int x) const { return bperm(x, s); }
    __device__ __forceinline__ long long operator()(long long x) const { return bperm64(x, s); }
};
// Lanes own consecutive segments [off_l, off_l + len_l) of T elements, off_l
// not decreasing with l; lane j of a chunk of W elements starting at k0
// handles element k0 + j, whose owner is the last lane whose segment starts
// at or before it. The lanes with off_l <= x are a prefix of the wave, so
// one ballot gives the owner of a position that is the same in every lane:
// when the chunk's first and last elements have one owner, so do all its
// elements, and body(LanePull) reads that lane's fields with readlane;
// otherwise each lane finds its owner by binary search over the lanes and
// body(PermPull) reads them with ds_bpermute. Every lane must be active.
template <class F>
__device__ __forceinline__ void by_owner(int off, int k0, int T, F &&body) {
    const int s0 = __popcll(ballot(off <= k0)) - 1;
    const int s1 = __popcll(ballot(off <= min(k0 + W, T) - 1)) - 1;
    if (s0 == s1) {
        body(LanePull{s0});
    } else {
        const int j = k0 + lane_id();
        int s = 0;
#pragma unroll
        for (int step = 32; step >= 1; step >>= 1)
            if (bperm(off, s + step) <= j && s + step < W) s += step;
        body(PermPull{s});
    }
}
// LDS accesses of one wavefront are performed in program order; the fences
// keep the compiler from moving them across this point.
__device__ __forceinline__ void wsync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ int excl_scan(int x, int *total) {
    int v = x;
#pragma unroll
    for (int d = 1; d < W; d <<= 1) {
        const int y = __shfl_up(v, d);
        if (lane_id() >= d) v += y;
    }
    *total = __shfl(v, W - 1);
    return v - x;
}
__device__ __forceinline__ unsigned long long wave_sum64(unsigned long long x) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) x += __shfl_xor(x, d);
    return x;
}
__device__ __forceinline__ unsigned long long range_mask(int lo, int hi) {  // bits [lo,hi), 0<=lo<hi<=64
    const unsigned long long h = hi >= 64 ? ~0ull : ((1ull << hi) - 1);
    return h & ~((1ull << lo) - 1);
}

// Number of elements of sorted a[0,len) below t.
template <class P>
__device__ __forceinline__ int lbound(P a, int len, int t) {
    int lo = 0, n = len;
    while (n > 0) {
        const int h = n >> 1;
        if (a[lo + h] < t) {
            lo += h + 1;
            n -= h + 1;
        } else {
            n = h;
        }
    }
    return lo;
}
// Membership of x in sorted a[0,len): linear scan below lin_thr entries
// (the reference's set_search_type switch, array_vertex_set.cuh:145-158),
// otherwise a branch-free binary descent that never reads past len.
template <class P>
__device__ __forceinline__ bool has(P a, int len, int x, int lin_thr) {
    if (len <= 0) return false;
    if (len < lin_thr) {
        for (int i = 0; i < len; i++) {
            const int y = a[i];
            if (y >= x) return y == x;
        }
        return false;
    }
    int base = 0, n = len;
    while (n > 1) {
        const int half = n >> 1;
        base = (a[base + half] <= x) ? base + half : base;
        n -= half;
    }
    return a[base] == x;
}

// Work queues. Atomics on one address are performed one after the other, about
// 20 ns each on this chip, so one head would feed a launch at most 50 tasks per
// microsecond and hold back every wave that asks meanwhile (C4 + P4 on a random
// graph of 1.6M directed edges: 8.8 ms with 16 edges per task and 19 ms with 4;
// 3.8 and 4.3 ms with 64 heads; a launch without work: 50 and 6 us). A queue has
// kHeads heads on cache lines of their own; head q hands out the items
// (r / kRun kHeads + q) kRun + r % kRun, r = 0, 1, ..: runs of kRun neighbouring
// items, which share a root and the tables kept for it, go to the waves of one
// head, and waves 8 apart sit on one XCD. A wave whose head is empty moves on to
// the next one with items left.
constexpr int kHeads = 64, kHeadStride = 16, kRun = 8;
enum { kQueueMain = 0, kQueueOverflow = 1, kQueueSub = 1 /* + sub_mode */, kQueues = 6 };
constexpr int kQueueWords = kQueues * kHeads * kHeadStride;
__device__ __forceinline__ long long queue_item(unsigned long long r, int q) {
    return (long long)((r / kRun * kHeads + q) * kRun + r % kRun);
}
// The next of the n items of queue id, or -1; *q: this wave's head.
__device__ __forceinline__ long long queue_next(unsigned long long *queue, unsigned int *drained, int id, long long n,
                                                int *q, int ln) {
    if (n <= 0) return -1;
    unsigned long long *heads = queue + id * kHeads * kHeadStride;
    for (;;) {
        unsigned long long r = 0;
        if (ln == 0) r = atomicAdd(&heads[*q * kHeadStride], 1ull);
        const long long item = queue_item((unsigned long long)uni64((long long)__shfl(r, 0)), *q);
        if (item < n) return item;
        static_assert(kHeads == W, "one head per lane");
        const unsigned long long at = __hip_atomic_load(&heads[ln * kHeadStride], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned long long m = ballot(queue_item(at, ln) < n);
        if (!m) {
            if (ln == 0 && !__hip_atomic_load(&drained[id], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                __hip_atomic_store(&drained[id], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return -1;
        }
        const int k = (*q + 1) % kHeads;  // the next head from k on that has items
        const unsigned long long rot = k ? m >> k | m << (kHeads - k) : m;
        *q = (k + __ffsll((long long)rot) - 1) % kHeads;
    }
}

// Counters are kept in kCountCopies copies of GATP_MAX_TERMS, one per group of
// workgroups, which the host adds up: atomics on one address are performed one
// after the other, 17 ns each, and every wave of a launch ends with one per
// pattern (4,096 waves and 21 patterns: 1.5 ms on one copy).
constexpr int kCountCopies = 32;
__device__ __forceinline__ unsigned long long *count_copy(unsigned long long *counts) {
    return counts + (blockIdx.x % kCountCopies) * GATP_MAX_TERMS;
}

struct Ctx {
    const KArgs &a;
    const GatPlanDev &P;
    WaveState *S;
    int *store;
    int ln;
};

// Truncation bound of an op/vid: max over groups of min over member levels.
// Level `d` reads the per-lane candidate c.
__device__ __forceinline__ int group_bound(const WaveState *S, const uint8_t *groups, int ngroups, int d, int c) {
    if (ngroups == 0) return INT_MAX;
    int best = INT_MIN;
    for (int g = 0; g < ngroups; g++) {
        int mn = INT_MAX;
        const unsigned m = groups[g];
        for (int f = 0; f <= GATP_MAX_DEPTH; f++)
            if (m >> f & 1u) mn = min(mn, f == d ? c : S->val[f]);
        best = max(best, mn);
    }
    return best;
}
__device__ __forceinline__ int mask_bound(const WaveState *S, unsigned mask, int d, int c) {
    int mn = INT_MAX;
    for (int f = 0; f <= GATP_MAX_DEPTH; f++)
        if (mask >> f & 1u) mn = min(mn, f == d ? c : S->val[f]);
    return mn;
}
__device__ __forceinline__ bool equals_any(const WaveState *S, unsigned mask, int d, int x) {
    bool r = false;
    for (int f = 0; f < d; f++)
        if (mask >> f & 1u) r |= (S->val[f] == x);
    return r;
}

// Length of N(v) below t (split[] answers the common t == v case).
__device__ __forceinline__ int trunc_len(const KArgs &a, int v, long long beg, int deg, int t) {
    if (t == INT_MAX) return deg;
    if (t == v) return a.split[v];
    return lbound(a.adj + beg, deg, t);
}

// Hub row of vertex v, or -1.
__device__ __forceinline__ int hub_of(const KArgs &a, int v) {
    if (a.n_hubs == 0) return -1;
    const int h = a.hub_map ? a.hub_map[v] : v;
    return h < a.n_hubs ? h : -1;
}
// Membership of x in the first len entries of hub h's sorted neighbour
// list, whose last kept entry is lim: one bitmap word instead of a search.
__device__ __forceinline__ bool hub_has(const KArgs &a, int h, int x, int lim) {
    return x <= lim && ((a.hub_bits[(long long)h * a.hub_words + (x >> 5)] >> (x & 31)) & 1u);
}
// Largest kept entry of a neighbour-list prefix of length len (-1 if empty).
__device__ __forceinline__ int list_lim(const KArgs &a, long long beg, int len) {
    return len > 0 ? a.adj[beg + len - 1] : -1;
}

// Number of distinct values among ex[0,nex) that lie in the first len
// entries of N(v) (list at beg): the excluded chosen vertices a COUNT
// without a father set must subtract from len. One membership test each
// (bitmap word for hubs) instead of a sweep of the list.
__device__ __forceinline__ int excluded_in_list(const KArgs &a, int v, long long beg, int len, const int *ex,
                                                int nex) {
    if (len <= 0) return 0;
    const int h = hub_of(a, v);
    const int lim = h >= 0 ? list_lim(a, beg, len) : 0;
    int k = 0;
    for (int q = 0; q < nex; q++) {
        bool seen = false;
        for (int q2 = 0; q2 < q; q2++) seen |= ex[q2] == ex[q];
        if (seen) continue;
        if (h >= 0 ? hub_has(a, h, ex[q], lim) : has(a.adj + beg, len, ex[q], a.lin_thr)) k++;
    }
    return k;
}

// Wave-cooperative intersection of stream[0,slen) with the set tested by
// probe(x), skipping the (at most 8) excluded values; writes the sorted
// result to out when MAT.
template <bool MAT, class SP, class PR, class OP>
__device__ __forceinline__ int wave_isect(SP stream, int slen, PR probe, OP out, const int *ex, int nex, int ln) {
    int total = 0;
    for (int base = 0; base < slen; base += W) {
        const int i = base + ln;
        bool hit = false;
        int x = 0;
        if (i < slen) {
            x = stream[i];
            hit = probe(x);
            for (int k = 0; k < nex; k++) hit &= (x != ex[k]);
        }
        const unsigned long long m = ballot(hit);
        if (MAT && hit) out[total + mbcnt(m)] = x;
        total += __popcll(m);
    }
    return total;
}

// Merge-path intersection of two sorted lists A[0,na) and B[0,nb), for
// pairs of similar length. In merge order A[i] precedes B[j] iff
// A[i] <= B[j]; the 64 lanes split the na + nb merged positions into equal
// runs, find where their run starts by a binary search along its diagonal,
// and merge their run serially. A common value x = A[i] = B[j] is found
// once, when B[j] is consumed and the A element before it (A[i-1], possibly
// consumed by the previous lane) equals it. Sorted output (MAT): one pass
// counts, an exclusive scan of the lanes' counts places each run's hits,
// and a second pass writes them.
template <bool MAT, class PA, class PB, class OP>
__device__ __forceinline__ int wave_merge_isect(PA A, int na, PB B, int nb, OP out, const int *ex, int nex, int ln) {
    const int total = na + nb;
    if (na == 0 || nb == 0) return 0;
    const int run = (total + W - 1) / W;
    const int k0 = min(total, ln * run), k1 = min(total, k0 + run);
    int lo = max(0, k0 - nb), hi = min(k0, na);
    while (lo < hi) {  // i = number of A elements among the first k0 merged
        const int mid = (lo + hi) >> 1;
        if (A[mid] <= B[k0 - 1 - mid]) lo = mid + 1; else hi = mid;
    }
    const int i0 = lo, j0 = k0 - lo;
    int cnt = 0;
    for (int pass = 0; pass < (MAT ? 2 : 1); pass++) {
        int i = i0, j = j0, w = 0;
        if (pass == 1) {
            int tot = 0;
            w = excl_scan(cnt, &tot);
        }
        int prev = i > 0 ? A[i - 1] : INT_MIN;  // the A element merged last
        int a = i < na ? A[i] : INT_MAX;
        for (int k = k0; k < k1; k++) {
            if (i < na && (j >= nb || a <= B[j])) {
                prev = a;
                i++;
                a = i < na ? A[i] : INT_MAX;
            } else {
                const int x = B[j++];
                bool hit = prev == x;
                for (int q = 0; q < nex; q++) hit &= (x != ex[q]);
                if (hit) {
                    if (pass == 0) cnt++;
                    else out[w++] = x;
                }
            }
        }
    }
    int tot = 0;
    (void)excl_scan(cnt, &tot);
    return tot;
}

// Galloping intersection of a short sorted list S[0,ns) with a long one
// L[0,nl), for skewed pairs. Each lane takes a block of up to 64
// consecutive elements of S (rounds of 64 blocks), finds the first by a
// binary search of L and every further one by an exponential search from
// the previous position (steps 1, 2, 4, ... then a binary search of the
// last step), so an element costs about 2 log2 of its gap in L instead of
// log2(nl). Hits are kept as a per-lane bit mask; the exclusive scan of
// their counts places the sorted output (MAT).
template <bool MAT, class PS, class PL, class OP>
__device__ __forceinline__ int wave_gallop_isect(PS S, int ns, PL L, int nl, OP out, const int *ex, int nex, int ln) {
    int total = 0;
    for (int base = 0; base < ns; base += W * W) {
        const int blk = min(W, (ns - base + W - 1) / W);
        const int b0 = min(ns, base + ln * blk), b1 = min(ns, b0 + blk);
        unsigned long long mask = 0;
        int pos = 0;
        for (int e = b0; e < b1; e++) {
            const int x = S[e];
            int lo, hi;  // the first element >= x lies in [lo, hi]
            if (e == b0) {
                lo = 0;
                hi = nl;
            } else {
                lo = pos;
                int step = 1;
                hi = pos;
                while (hi < nl && L[hi] < x) {
                    lo = hi + 1;
                    hi = pos + step;
                    step <<= 1;
                }
                hi = min(hi, nl);
            }
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (L[mid] < x) lo = mid + 1; else hi = mid;
            }
            pos = lo;
            bool hit = pos < nl && L[pos] == x;
            for (int q = 0; q < nex; q++) hit &= (x != ex[q]);
            if (hit) mask |= 1ull << (e - b0);
        }
        int tot = 0;
        const int w = excl_scan(__popcll(mask), &tot);
        if (MAT) {
            int o = total + w;
            while (mask) {
                const int b = __ffsll((long long)mask) - 1;
                mask &= mask - 1;
                out[o++] = S[b0 + b];
            }
        }
        total += tot;
    }
    return total;
}

// Stream A (the new vertex's neighbour list) and probe the father set, or
// the reverse? A side is cheap to probe when it sits in LDS or has a hub
// bitmap; the other side is then streamed unless it is gallop_ratio times
// longer.
__device__ __forceinline__ bool stream_a(const KArgs &a, int alen, int blen, bool b_fast, bool a_fast) {
    if (a.strategy == 1) return true;
    if (a.strategy == 2) return alen <= blen;
    const long long r = a.gallop_ratio;
    if (b_fast && !a_fast) return !((long long)alen > r * (long long)blen);
    if (a_fast && !b_fast) return (long long)blen > r * (long long)alen;
    return alen <= blen;
}

// Calls f with the slot's content pointer; the two branches keep the LDS
// and global provenance apart so each access compiles to ds_* or global_*.
template <bool GS, class F>
__device__ __forceinline__ auto with_slot(const Ctx &C, int slot, F f) {
    const GatSlot &s = C.P.slots[slot];
    if (s.kind == GATP_ALIAS && (GS || !C.S->staged[slot])) return f(C.a.adj + C.S->sbeg[slot]);
    return f(C.store + C.a.store_off[s.store]);
}
// Is the slot's content in this wave's LDS buffers?
template <bool GS>
__device__ __forceinline__ bool in_lds(const Ctx &C, int slot) {
    if (GS) return false;
    const GatSlot &s = C.P.slots[slot];
    return s.kind == GATP_LIST || C.S->staged[slot];
}

// Evaluate one op for the wave-uniform candidate c at depth d.
template <bool GS>
__device__ __forceinline__ void exec_op_uniform(const Ctx &C, const GatOp &o, int d, int c, bool dup) {
    const KArgs &a = C.a;
    WaveState *S = C.S;
    const int t = uni(group_bound(S, o.groups, o.ngroups, d, c));
    const long long ab = a.off[c];
    const int deg = (int)(a.off[c + 1] - ab);
    int alen = dup ? 0 : uni(trunc_len(a, c, ab, deg, t));
    const int slot = o.slot;
    if (o.kind == GATP_ALIAS) {
        // a list that later ops search is staged into LDS when it fits
        const bool stage = !GS && o.store >= 0 && alen <= a.stage_cap;
        if (stage) {
            int *dst = C.store + a.store_off[o.store];
            for (int k = C.ln; k < alen; k += W) dst[k] = a.adj[ab + k];
        }
        if (C.ln == 0) {
            S->sbeg[slot] = ab;
            S->slen[slot] = alen;
            S->staged[slot] = stage ? 1 : 0;
        }
        return;
    }
    int ex[8];
    int nex = 0;
    if (o.kind == GATP_COUNT)
        for (int f = 0; f < d; f++)
            if (o.excl >> f & 1u) ex[nex++] = S->val[f];
    const int f = o.father;
    int blen = 0, result = 0;
    const bool has_r = f >= 0;
    bool b_lds = false;
    int hub_b = -1;
    long long bbeg = 0;
    if (has_r) {
        const GatSlot &fs = C.P.slots[f];
        b_lds = in_lds<GS>(C, f);
        const int flen = S->slen[f];
        blen = dup ? 0 : (t == INT_MAX ? flen : uni(with_slot<GS>(C, f, [&](auto B) { return lbound(B, flen, t); })));
        if (fs.kind == GATP_ALIAS) {
            bbeg = S->sbeg[f];
            if (!b_lds) hub_b = uni(hub_of(a, S->val[fs.depth]));
        }
    }
    if (o.kind == GATP_LIST) {
        const int ub = has_r ? min(alen, blen) : alen;
        if (ub > a.cap) {
            if (C.ln == 0) S->abort = 1;
            return;
        }
    }
    const int *A = a.adj + ab;
    int *out = C.store + a.store_off[o.store < 0 ? 0 : o.store];
    const int hub_a = has_r ? uni(hub_of(a, c)) : -1;
    const bool sa = !has_r || stream_a(a, alen, blen, b_lds || hub_b >= 0, hub_a >= 0);
    const int lin = a.lin_thr;
    auto run = [&](auto stream, int slen, auto probe) {
        return o.kind == GATP_LIST ? wave_isect<true>(stream, slen, probe, out, ex, nex, C.ln)
                                   : wave_isect<false>(stream, slen, probe, out, ex, nex, C.ln);
    };
    // merge path or galloping between two sorted arrays (strategies 3 and 4;
    // a hub's bitmap is not used there)
    const int sorted_pair = has_r && (a.strategy == 3 || a.strategy == 4) ? a.strategy : 0;
    auto run2 = [&](auto P, int np_, auto Q, int nq) {  // P, Q: sorted arrays
        if (sorted_pair == 3)
            return o.kind == GATP_LIST ? wave_merge_isect<true>(P, np_, Q, nq, out, ex, nex, C.ln)
                                       : wave_merge_isect<false>(P, np_, Q, nq, out, ex, nex, C.ln);
        // galloping: the shorter list is walked, the longer one searched
        if (np_ <= nq)
            return o.kind == GATP_LIST ? wave_gallop_isect<true>(P, np_, Q, nq, out, ex, nex, C.ln)
                                       : wave_gallop_isect<false>(P, np_, Q, nq, out, ex, nex, C.ln);
        return o.kind == GATP_LIST ? wave_gallop_isect<true>(Q, nq, P, np_, out, ex, nex, C.ln)
                                   : wave_gallop_isect<false>(Q, nq, P, np_, out, ex, nex, C.ln);
    };
    if (sorted_pair) {
        if (b_lds) {
            const int *B = C.store + a.store_off[C.P.slots[f].store];
            result = run2(A, alen, B, blen);
        } else {
            const int *B = C.P.slots[f].kind == GATP_ALIAS ? a.adj + bbeg
                                                           : C.store + a.store_off[C.P.slots[f].store];
            result = run2(A, alen, B, blen);
        }
    } else if (!has_r && o.kind == GATP_COUNT) {
        result = alen - uni(excluded_in_list(a, c, ab, alen, ex, nex));
    } else if (!has_r) {
        result = run(A, alen, [](int) { return true; });
    } else if (sa) {
        // stream A, probe the father: LDS buffer, hub bitmap, or HBM list
        if (b_lds) {
            const int *B = C.store + a.store_off[C.P.slots[f].store];
            result = run(A, alen, [&](int x) { return has(B, blen, x, lin); });
        } else if (hub_b >= 0) {
            const int lim = uni(list_lim(a, bbeg, blen));
            result = run(A, alen, [&](int x) { return hub_has(a, hub_b, x, lim); });
        } else {
            const int *B = C.P.slots[f].kind == GATP_ALIAS ? a.adj + bbeg
                                                           : C.store + a.store_off[C.P.slots[f].store];
            result = run(A, alen, [&](int x) { return has(B, blen, x, lin); });
        }
    } else {
        // stream the father, probe A
        auto probe_a = [&](int x) { return has(A, alen, x, lin); };
        const int lim_a = hub_a >= 0 ? uni(list_lim(a, ab, alen)) : 0;
        auto probe_hub = [&](int x) { return hub_has(a, hub_a, x, lim_a); };
        if (b_lds) {
            const int *B = C.store + a.store_off[C.P.slots[f].store];
            result = hub_a >= 0 ? run(B, blen, probe_hub) : run(B, blen, probe_a);
        } else {
            const int *B = C.P.slots[f].kind == GATP_ALIAS ? a.adj + bbeg
                                                           : C.store + a.store_off[C.P.slots[f].store];
            result = hub_a >= 0 ? run(B, blen, probe_hub) : run(B, blen, probe_a);
        }
    }
    if (C.ln == 0) {
        S->slen[slot] = result;
        if (a.account) {
            const GatSlot *fs = has_r ? &C.P.slots[f] : nullptr;
            S->ebytes += 4ull * (alen + blen) + (o.kind == GATP_LIST ? 4ull * result : 0ull) + 16ull +
                        ((fs && fs->kind == GATP_ALIAS) ? 16ull : 0ull);
        }
    }
}

// Subtask blocks handed on since the last commit are emptied when the work
// they came from is abandoned: the HBM launch re-runs that work whole.
__device__ __noinline__ void cancel_donations(const KArgs &a, WaveState *S, int ln) {
    const int nd = S->n_don;
    for (int i = 0; i < nd; i++) {
        const long long b = S->don_base[i];
        const int cnt = S->don_cnt[i];
        for (int k = ln; k < cnt; k += W) {
            a.subs[b + k].lo = 0;
            a.subs[b + k].hi = 0;
        }
    }
    wsync();
    if (ln == 0) S->n_don = 0;
    wsync();
}

// Split only in the tail: the queue the task came from has nothing left for
// idle waves (queue_drained) and the task has outrun its budget (want_split).
template <bool GS>
__device__ __forceinline__ bool queue_drained(const KArgs &a) {
    if (a.split_ticks <= 0 || a.sub_mode >= kSplitLevels) return false;
    const int id = GS ? kQueueOverflow : a.sub_mode == 0 ? kQueueMain : kQueueSub + a.sub_mode;
    return uni((int)__hip_atomic_load(&a.drained[id], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0;
}
template <bool GS>
__device__ __forceinline__ bool want_split(const KArgs &a, const WaveState *S) {
    if (a.split_ticks <= 0 || a.sub_mode >= kSplitLevels) return false;
    if (uni64(wall_clock64()) - S->t0 <= a.split_ticks) return false;
    return queue_drained<GS>(a);
}

// A loop whose first `done` candidates took `ticks`: will the other `left` take
// more than 1 / kTailShare of the split budget? In the tail such a rest does not
// wait for the budget: idle waves are there to take it, and one subtask costs 10
// to 20 us. (Counts of a few roots are tails from their start: C5 of one root of
// Chung-Lu 1M took 4.7 ms in the mean of eight while every level of subtasks
// waited for the budget, and takes 1.3.)
constexpr int kTailShare = 8;
__device__ __forceinline__ bool rest_is_long(const KArgs &a, long long ticks, int done, int left) {
    return done > 0 && ticks * left * kTailShare > a.split_ticks * done;
}
// The same for the depth-d frame, above the leaves, with candidates [cur, fh)
// left; or the task has outrun its budget (want_split).
template <bool GS>
__device__ __forceinline__ bool due_to_split(const KArgs &a, WaveState *S, int d, int cur, int fh, int ln) {
    if (a.split_ticks <= 0 || a.sub_mode >= kSplitLevels) return false;
    const long long now = uni64(wall_clock64());
    const int done = cur - (d == uni(S->base_depth) ? uni(S->base_lo) : 0);
    if (done == 0 && ln == 0) S->f_t0[d] = now;
    const bool spent = now - S->t0 > a.split_ticks;
    if (!spent && !rest_is_long(a, now - S->f_t0[d], done, fh - cur)) return false;
    return queue_drained<GS>(a);
}

// Hands candidates [lo, hi) of the depth-d frame's node to the next split
// launch, in at most 64 chunks of at least min_chunk. False, with nothing
// handed on, when the wave's record of donations or the list is full
// (reserved entries past the end of the list are left empty). Donations are
// recorded for cancellation only where the donor can still abort (LDS
// buffers); the HBM launch's tasks cannot, so their donations are unlimited.
// sum_op: the op of a KEEP_SUM's range, or -1.
__device__ __noinline__ bool donate(const Ctx C, int d, int node, int lo, int hi, int min_chunk, bool record,
                                    int sum_op = -1) {
    const KArgs &a = C.a;
    WaveState *S = C.S;
    if (record && S->n_don >= kMaxDonations) return false;
    const long long edge = S->sub_edge >= 0 ? S->sub_edge : S->rb + (S->f_cur[1] - 1);
    const int r = hi - lo;
    const int chunk = max(min_chunk, (r + W - 1) / W);
    const int parts = (r + chunk - 1) / chunk;
    unsigned long long b = 0;
    if (C.ln == 0) b = atomicAdd(a.out_n, (unsigned long long)parts);
    const long long base = uni64((long long)__shfl(b, 0));
    const long long room = a.out_cap - base;
    const int fit = room <= 0 ? 0 : (room < parts ? (int)room : parts);
    for (int k = C.ln; k < fit; k += W) {
        SplitTask *t = a.subs + a.out_base + base + k;
        t->edge = edge;
        t->node = node;
        t->depth = d;
        t->lo = fit == parts ? lo + k * chunk : 0;
        t->hi = fit == parts ? min(hi, lo + (k + 1) * chunk) : 0;
        t->pos[0] = sum_op + 1;
        for (int j = 2; j < d; j++) t->pos[j] = j < S->base_depth ? S->path_pos[j] : S->f_cur[j] - 1;
    }
    if (fit < parts) return false;
    if (record && C.ln == 0) {
        S->don_base[S->n_don] = a.out_base + base;
        S->don_cnt[S->n_don] = parts;
        S->n_don++;
    }
    wsync();
    return true;
}

constexpr int kPairChunk = 8;  // least candidates of a subtask at a pair node (pair_leaf)

// Donates the rest of the shallowest frame (depth >= base_depth, up to d)
// that has two or more candidates left; true if it did. The frame is closed
// by lowering its end to its cursor: f_cur[k] - 1 stays the position of the
// candidate being walked at depth k, which later donations from deeper
// frames record as their path.
template <bool GS>
__device__ __noinline__ bool split_shallowest(const Ctx C, int d) {
    WaveState *S = C.S;
    for (int k = uni(S->base_depth); k <= d; k++) {
        const int cur = uni(S->f_cur[k]), fh = uni(S->f_hi[k]);
        if (fh - cur < 2) continue;
        const int node = uni(S->f_node[k]);
        const int least = C.P.nodes[node].leaf ? W : C.P.nodes[node].pair ? kPairChunk : 1;
        if (!donate(C, k, node, cur, fh, least, !GS)) return false;
        if (C.ln == 0) S->f_hi[k] = cur;
        wsync();
        return true;
    }
    return false;
}

// Value of one IEP factor. Per-lane candidate c sits at depth d; leaf
// counters are read for this lane.
template <bool GS>
__device__ __forceinline__ long long vid_value(const Ctx &C, const GatVid &v, int d, int c) {
    const WaveState *S = C.S;
    const GatSlot &s = C.P.slots[v.slot];
    if (s.leaf_idx >= 0) return S->leafcnt[s.leaf_idx][C.ln];
    const int L = S->slen[v.slot];
    if (v.mode == GATP_VID_COUNT) return L;
    return with_slot<GS>(C, v.slot, [&](auto p) -> long long {
        if (v.mode == GATP_VID_LIST_REF) {
            long long r = L;
            for (int i = 0; i < v.refn; i++) r -= has(p, L, i == d ? c : S->val[i], C.a.lin_thr) ? 1 : 0;
            return r;
        }
        const int t = v.bound ? mask_bound(S, v.bound, d, c) : INT_MAX;
        long long r = t == INT_MAX ? L : lbound(p, L, t);
        for (int j = 0; j <= d; j++)
            if (v.excl >> j & 1u) {
                const int x = j == d ? c : S->val[j];
                if (x < t && has(p, L, x, C.a.lin_thr)) r--;
            }
        return r;
    });
}

template <bool GS>
__device__ __forceinline__ unsigned long long term_value(const Ctx &C, const GatTerm &T, int d, int c) {
    unsigned long long local = 0, val = 1;
    int last = -1;
    for (int g = 0; g < T.sub_count; g++) {
        const GatSub &sb = C.P.subs[T.sub_begin + g];
        const unsigned long long x = (unsigned long long)vid_value<GS>(C, C.P.vids[sb.vid], d, c);
        val = (g == last + 1) ? x : val * x;
        if (sb.flag) {
            last = g;
            local += val * (unsigned long long)(long long)sb.coef;
        }
    }
    return local;
}

// replay: rebuild the node's sets for a split subtask without adding its
// terms again (the donor counted them).
template <bool GS>
__device__ __forceinline__ bool visit(const Ctx &C, const GatNode &N, int d, int c, bool replay = false) {
    WaveState *S = C.S;
    if (C.ln == 0) S->val[d] = c;
    wsync();
    const bool dup = N.ap_levels && equals_any(S, N.ap_levels, d, c);
    for (int k = 0; k < N.op_count; k++) {
        exec_op_uniform<GS>(C, C.P.ops[N.op_begin + k], d, c, dup);
        wsync();
        if (S->abort) return false;
    }
    for (int k = 0; k < N.term_count && !replay; k++) {
        const GatTerm &T = C.P.terms[N.term_begin + k];
        const unsigned long long v = term_value<GS>(C, T, d, c);
        if (C.ln == 0) S->task_acc[T.pattern] += v;
    }
    wsync();
    return true;
}

// |N(c) ∩ father ∩ [0,t)|, father the set of slot f, without the nex values ex, for the lanes in `need`
// (0 in the others): the (candidate, element) pairs of the wave's lanes form one
// flattened index space. alen: the length of N(c) below t; *blen_out: that of
// the father.
template <bool GS>
__device__ __forceinline__ int sweep_count(const Ctx &C, int f, bool need, int c, long long ab, int alen, int t,
                                           const int *ex, int nex, int *blen_out) {
    const KArgs &a = C.a;
    WaveState *S = C.S;
    const int ln = C.ln;
    int cnt = 0;
    int blen = 0;
    // Bg: father in HBM (a neighbour list, or any set in the overflow
    // launch); Bl: father in this wave's LDS buffers. hub_b: the
    // father is a hub's neighbour list in HBM, probed by bitmap.
    const int *Bg = a.adj;
    const int *Bl = C.store;
    int hub_b = -1, lim_b = 0;
    const GatSlot &fs = C.P.slots[f];
    const bool b_lds = in_lds<GS>(C, f);
    if (b_lds) Bl = C.store + a.store_off[fs.store];
    else if (fs.kind == GATP_ALIAS) Bg = a.adj + S->sbeg[f];
    else if constexpr (GS) Bg = C.store + a.store_off[fs.store];
    const int flen = S->slen[f];
    if (need) blen = t == INT_MAX ? flen : (b_lds ? lbound(Bl, flen, t) : lbound(Bg, flen, t));
    if (!b_lds && fs.kind == GATP_ALIAS) hub_b = uni(hub_of(a, S->val[fs.depth]));
    // candidate lists with a hub bitmap are probed through it
    const int hub_a = need ? hub_of(a, c) : -1;
    const int lim_a = hub_a >= 0 ? list_lim(a, ab, alen) : 0;
    if (hub_b >= 0 && need) lim_b = blen > 0 ? Bg[blen - 1] : -1;
    const bool sa = stream_a(a, alen, blen, b_lds || hub_b >= 0, hub_a >= 0);
    const int mylen = sa ? alen : blen;
    int T = 0;
    const int myoff = excl_scan(mylen, &T);
    for (int k0 = 0; k0 < T; k0 += W) {
        const int j = k0 + ln;
        bool hit = false;
        by_owner(myoff, k0, T, [&](const auto &pull) {
            const int s_off = pull(myoff);
            const int s_sa = pull((int)sa);
            const long long s_ab = pull(ab);
            const int s_alen = pull(alen);
            const int s_blen = pull(blen);
            const int s_hub = pull(hub_a);
            const int s_lim = pull(lim_a);
            const int s_limb = pull(lim_b);
            if (j < T) {
                const int idx = j - s_off;
                int x;
                if (s_sa) {
                    x = a.adj[s_ab + idx];
                    if (b_lds) hit = has(Bl, s_blen, x, a.lin_thr);
                    else if (hub_b >= 0) hit = hub_has(a, hub_b, x, s_limb);
                    else hit = has(Bg, s_blen, x, a.lin_thr);
                } else {
                    x = b_lds ? Bl[idx] : Bg[idx];
                    hit = s_hub >= 0 ? hub_has(a, s_hub, x, s_lim) : has(a.adj + s_ab, s_alen, x, a.lin_thr);
                }
                for (int q = 0; q < nex; q++) hit &= (x != ex[q]);
            }
        });
        const unsigned long long m = ballot(hit);
        const int lo = max(myoff - k0, 0), hi2 = min(myoff + mylen - k0, W);
        if (lo < hi2) cnt += __popcll(m & range_mask(lo, hi2));
    }
    *blen_out = blen;
    return cnt;
}
// The same from the candidate alone. (Out of line, this and pair_leaf cost C5
// on R-MAT s13 a third: 19.9 against 14.7 ms.)
template <bool GS>
__device__ __forceinline__ int sweep_kept(const Ctx &C, int f, bool need, int c, int t) {
    const long long ab = need ? C.a.off[c] : 0;
    const int alen = need ? trunc_len(C.a, c, ab, (int)(C.a.off[c + 1] - ab), t) : 0;
    int blen;
    return sweep_count<GS>(C, f, need, c, ab, alen, t, nullptr, 0, &blen);
}

// The table of a KEEP_POOL op for the chosen v_0, v_1 or root edge, and the tag
// of its entries.
__device__ __forceinline__ KeptEntry *pool_table(const Ctx &C, const GatOp &o, unsigned *tag) {
    const KArgs &a = C.a;
    const WaveState *S = C.S;
    unsigned key;
    if (o.key == 3) key = (unsigned)uni((int)(S->sub_edge >= 0 ? S->sub_edge : S->rb + (S->f_cur[1] - 1)));
    else key = (unsigned)uni(S->val[o.key == 2 ? 1 : 0]);
    *tag = key + 1;
    return a.pool + ((long long)o.table * a.pool_tables + key % a.pool_tables) * a.tab_size;
}

// Is x adjacent to y, for the lanes in `need`? x, its hub row hx (hub_of) and
// so the branches on it are the same in every lane; hx is found outside, by the
// whole wave, so that no cross-lane read stands under a lane's condition.
__device__ __forceinline__ bool adjacent(const KArgs &a, int x, int hx, int y, bool need) {
    if (hx >= 0) return need && hub_has(a, hx, y, INT_MAX);
    if (!need) return false;
    const int hy = hub_of(a, y);
    if (hy >= 0) return hub_has(a, hy, x, INT_MAX);
    const long long b = a.off[x];
    return has(a.adj + b, (int)(a.off[x + 1] - b), y, a.lin_thr);
}

// Excluded levels below `upto` of a kept COUNT whose chosen vertex lies in the op's father
// set before truncation (repeated vertices once): what plan compilation does
// not know is looked up here, once per leaf frame.
__device__ __forceinline__ void leaf_exclusions(const Ctx &C, const GatNode &N, int upto) {
    const KArgs &a = C.a;
    WaveState *S = C.S;
    for (int k = 0; k < N.op_count; k++) {
        const GatOp &o = C.P.ops[N.op_begin + k];
        if (o.kind != GATP_COUNT || o.keep == GATP_KEEP_NONE || o.keep == GATP_KEEP_SUM) continue;
        int in = 0;
        for (int f = 0; f < upto; f++) {
            if (!(o.excl >> f & 1u)) continue;
            const int x = uni(S->val[f]);
            bool yes = true;
            for (int g = 0; g < f; g++) yes &= !((o.excl >> g & 1u) && S->val[g] == x);
            if (yes && !(o.ex_father >> f & 1u)) {
                // the father's set is the intersection of N(v_l) over its levels
                const int hx = uni(hub_of(a, x));
                for (int l = 0; l < GATP_MAX_DEPTH; l++)
                    if (o.levels >> l & 1u) yes = adjacent(a, x, hx, uni(S->val[l]), yes);
            }
            if (uni((int)yes)) in |= 1 << f;
        }
        if (C.ln == 0) S->ex_in[o.leaf_idx] = in;
    }
    wsync();
}

// Does every table of the leaf node hold the value of c, the ci-th candidate?
__device__ __forceinline__ bool leaf_known(const Ctx &C, const GatNode &N, int c, int ci) {
    const KArgs &a = C.a;
    bool known = true;
    for (int k = 0; k < N.op_count; k++) {
        const GatOp &o = C.P.ops[N.op_begin + k];
        if (o.kind != GATP_COUNT) continue;
        if (o.keep == GATP_KEEP_EDGE) known = known && a.edge_tab[o.table][C.S->sbeg[N.loop_slot] + ci].read() >= 0;
        if (o.keep == GATP_KEEP_POOL) {
            unsigned key = 0;  // pool_table without its cross-lane reads
            if (o.key == 3) key = (unsigned)(C.S->sub_edge >= 0 ? C.S->sub_edge : C.S->rb + (C.S->f_cur[1] - 1));
            else key = (unsigned)C.S->val[o.key == 2 ? 1 : 0];
            if (c >= a.tab_size) return false;
            const long long table = (long long)o.table * a.pool_tables + key % a.pool_tables;
            known = known && a.pool[table * a.tab_size + c].read().serves(key + 1, a.epoch);
        }
    }
    return known;
}

// The KEEP_SUM op k of leaf node N (number `node`) at depth d: its sum over all
// candidates of the frame, taken over the entries [lo, hi) of its father and
// added to the terms that use it. In the tail, a rest that one wave would sweep
// for more than 1 / kTailShare of the split budget (3 ticks an element, as in
// leaf()) goes to the next split launch in up to 64 parts. (One edge between two hubs of Chung-Lu 1M, house: 4.1 ms with the
// sum on one wave, 2.5 when the leaf that it replaces was split.)
template <bool GS>
__device__ __forceinline__ void leaf_sum(const Ctx &C, const GatNode &N, int d, int node, int k, int lo, int hi,
                                         bool can_split) {
    const KArgs &a = C.a;
    WaveState *S = C.S;
    const int ln = C.ln;
    const GatOp &o = C.P.ops[N.op_begin + k];
    const int v = uni(S->val[C.P.slots[N.loop_slot].depth]);  // v_j
    const long long vb = a.off[v];
    const int deg = (int)(a.off[v + 1] - vb), b = o.table ? v : INT_MAX;
    const int t = uni(group_bound(S, o.groups, o.ngroups, d, 0));
    KeptEdge *edge = a.edge_tab[o.table] + vb;
    unsigned long long sum = 0;
    for (int base = lo; base < hi; base += W) {
        const int i = base + ln;
        int x = INT_MAX;
        if (i < hi) x = with_slot<GS>(C, o.father, [&](auto p) { return p[i]; });
        bool use = i < hi && x < t;
        for (int f = 0; f < d; f++)
            if (o.excl >> f & 1u) use = use && x != S->val[f];
        int cnt = 0;
        const int pos = use ? lbound(a.adj + vb, deg, x) : 0;
        if (use) cnt = edge[pos].read();
        bool need = use && cnt < 0;
        if (ballot(need) && can_split && hi - base > 1 && queue_drained<GS>(a)) {
            const long long lw = need ? min((long long)deg, a.off[x + 1] - a.off[x]) : 0;
            const long long tot = uni64((long long)wave_sum64((unsigned long long)lw));
            const int kept = 3 * tot * kTailShare > a.split_ticks ? base + 1 : base + W;
            if (kept < hi && 3 * tot * kTailShare * (hi - base) > a.split_ticks * W &&
                donate(C, d, node, kept, hi, 1, !GS, k)) {
                hi = kept;
                use = use && i < hi;
                need = need && i < hi;
            }
        }
        if (ballot(need)) {
            const int fresh = sweep_kept<GS>(C, N.loop_slot, need, x, b);
            if (need) {
                cnt = fresh;
                edge[pos].write(fresh);
            }
        }
        // candidates that are skipped or empty although they lie in N(v_j)
        // below b: chosen vertices (each once)
        for (int f = 0; f < d; f++) {
            const unsigned out = N.excl | N.ap_levels;
            if (!(out >> f & 1u)) continue;
            const int y = uni(S->val[f]), hy = uni(hub_of(a, y));
            bool once = y < b;
            for (int h = 0; h < f; h++) once = once && !((out >> h & 1u) && S->val[h] == y);
            once = adjacent(a, y, hy, v, once);
            if (uni((int)once)) cnt -= adjacent(a, y, hy, x, use);
        }
        if (use) sum += (unsigned long long)(long long)cnt;
    }
    sum = wave_sum64(sum);
    if (ln == 0)
        for (int u = 0; u < N.term_count; u++) {
            const GatTerm &T = C.P.terms[N.term_begin + u];
            for (int q = 0; q < T.sub_count; q++) {
                const GatSub &sb = C.P.subs[T.sub_begin + q];
                if (C.P.vids[sb.vid].slot == o.slot) S->task_acc[T.pattern] += sum * (unsigned long long)(long long)sb.coef;
            }
        }
    wsync();
}

// All candidates of a leaf frame, flattened across lanes.
// With can_split, a wave that is due to split (want_split) hands the
// batches after the current one to the next split launch. With sum_op, the
// range is one of that op's father (see SplitTask) and nothing else is done.
template <bool GS, bool KEEP>
__device__ __forceinline__ void leaf(const Ctx &C, const GatNode &N, int d, int cur, int hi, bool can_split = false,
                                     int node = -1, int sum_op = -1) {
    const KArgs &a = C.a;
    WaveState *S = C.S;
    const int ln = C.ln;
    unsigned long long bytes = 0;
    if (KEEP && sum_op < 0) leaf_exclusions(C, N, d);
    // Parts of a frame that was split have cur > 0; a frame handed on whole is
    // left empty here. So the part with the first candidate adds the sums, and
    // an empty frame has none.
    for (int k = 0; KEEP && d >= 2 && (sum_op >= 0 || (cur == 0 && hi > 0)) && k < N.op_count; k++) {
        const GatOp &o = C.P.ops[N.op_begin + k];
        if (o.kind != GATP_COUNT || o.keep != GATP_KEEP_SUM || (sum_op >= 0 && k != sum_op)) continue;
        leaf_sum<GS>(C, N, d, node, k, sum_op >= 0 ? cur : 0, sum_op >= 0 ? hi : uni(S->slen[o.father]), can_split);
    }
    if (KEEP && sum_op >= 0) return;
    for (int cb = cur; cb < hi; cb += W) {
        const int ci = cb + ln;
        int c = 0;
        if (ci < hi) c = with_slot<GS>(C, N.loop_slot, [&](auto p) { return p[ci]; });
        // A chunk whose candidates' neighbour lists add up to more elements
        // than one wave sweeps within the split budget (about 3 ticks of the
        // 100 MHz clock per element) is not swept whole once the queue is
        // drained. First the rest of the shallowest loop above the leaf that
        // has candidates left goes to the next split launch (the most work
        // for one donation record). With none left, the leaf's candidates
        // after the first go, in about as many parts as the chunk holds
        // budgets of work (at most 64), so that whole waves sweep their lists
        // in parallel; the wave keeps the first candidate. Candidates whose values
        // are all in the tables are not swept.
        if (can_split && hi - cb > 1 && queue_drained<GS>(a)) {
            long long lw = 0;
            if (ci < hi && !(KEEP && N.kept && leaf_known(C, N, c, ci))) lw = a.off[c + 1] - a.off[c];
            const long long tot = uni64((long long)wave_sum64((unsigned long long)lw));
            if (3 * tot > a.split_ticks && !split_shallowest<GS>(C, d - 1)) {
                const long long budgets = 3 * tot / a.split_ticks + 1;
                const long long np = budgets < W ? budgets : W;
                const int r = hi - cb - 1;
                if (donate(C, d, node, cb + 1, hi, (int)((r + np - 1) / np), !GS)) hi = cb + 1;
            }
        }
        const bool valid = ci < hi;
        bool pass = valid && !equals_any(S, N.excl, d, c);
        const bool dup = pass && N.ap_levels && equals_any(S, N.ap_levels, d, c);
        long long ab = 0;
        int deg = -1;  // read when an op needs it
        for (int k = 0; k < N.op_count; k++) {
            const GatOp &o = C.P.ops[N.op_begin + k];
            const int t = group_bound(S, o.groups, o.ngroups, d, c);
            // kept values first: the lanes in `need` compute theirs
            const bool live = pass && !dup;
            bool need = live;
            int kept = 0;
            KeptEdge *edge = nullptr;
            KeptEntry *slot = nullptr;
            unsigned tag = 0;
            if (KEEP && o.keep == GATP_KEEP_SUM) {  // added by leaf_sum
                S->leafcnt[o.leaf_idx][ln] = 0;
                continue;
            }
            if (KEEP && o.keep == GATP_KEEP_EDGE) edge = a.edge_tab[o.table];
            if (KEEP && edge) {
                edge += S->sbeg[N.loop_slot] + ci;
                if (live) kept = edge->read();
                need = live && kept < 0;
            } else if (KEEP && o.keep == GATP_KEEP_POOL) {
                slot = pool_table(C, o, &tag) + c;
                if (live && c < a.tab_size) {
                    const KeptEntry::Read e = slot->read();
                    kept = e.value();
                    need = !e.serves(tag, a.epoch);
                }
            }
            const bool by_table = KEEP && (edge || slot);
            int cnt = 0;
            if (!by_table || ballot(need)) {
            if (uni(deg) < 0) {
                ab = valid ? a.off[c] : 0;
                deg = valid ? (int)(a.off[c + 1] - ab) : 0;
            }
            int alen = need ? trunc_len(a, c, ab, deg, t) : 0;
            if (o.kind == GATP_ALIAS) {
                S->leafcnt[o.leaf_idx][ln] = alen;
                continue;
            }
            // COUNT: |N(c) ∩ father ∩ [0,t)| minus excluded chosen vertices
            int ex[8];
            int nex = 0;
            for (int f = 0; f < d && !by_table; f++)  // a kept value leaves them in
                if (o.excl >> f & 1u) ex[nex++] = S->val[f];
            if (o.father < 0) {
                // |N(c) ∩ [0,t)| minus the excluded chosen vertices it holds
                S->leafcnt[o.leaf_idx][ln] = live ? alen - excluded_in_list(a, c, ab, alen, ex, nex) : 0;
                if (a.account && live) bytes += 4ull * alen + 16ull;
                continue;
            }
            int blen = 0;
            cnt = sweep_count<GS>(C, o.father, need, c, ab, alen, t, ex, nex, &blen);
            if (a.account && live)
                bytes += 4ull * (alen + blen) + 16ull + (C.P.slots[o.father].kind == GATP_ALIAS ? 16ull : 0ull);
            if (need && edge) edge->write(cnt);
            if (need && slot && c < a.tab_size) slot->write(tag, cnt, a.epoch);
            }
            if (by_table) {
                if (!need) cnt = kept;
                // the excluded vertices the set holds: in the father, below t, adjacent to c
                const int in = uni(S->ex_in[o.leaf_idx]);
                for (int f = 0; f < d; f++) {
                    if (!(in >> f & 1)) continue;
                    const int x = uni(S->val[f]);
                    const bool below = live && x < t;
                    if (o.ex_cand >> f & 1u) cnt -= below;
                    else cnt -= adjacent(a, x, uni(hub_of(a, x)), c, below);
                }
            }
            S->leafcnt[o.leaf_idx][ln] = live ? cnt : 0;
        }
        wsync();
        for (int k = 0; k < N.term_count; k++) {
            const GatTerm &Tm = C.P.terms[N.term_begin + k];
            unsigned long long v = pass ? term_value<GS>(C, Tm, d, c) : 0ull;
            v = wave_sum64(v);
            if (ln == 0) S->task_acc[Tm.pattern] += v;
        }
        wsync();
        if (can_split && hi - (cb + W) >= 2 * W && want_split<GS>(a, S) && donate(C, d, node, cb + W, hi, W, !GS))
            break;
    }
    if (a.account) {
        bytes = wave_sum64(bytes);
        if (ln == 0) S->ebytes += bytes;
    }
}

// The last two levels together (GatNode::pair): the frame's candidates v, 64 at
// a time, and below them all their candidates c in N(v), flattened over the
// lanes. A leaf frame of its own per v cost a visit, a frame and a chunk of 64
// lanes for about 40 candidates: 35 us a chunk on R-MAT s13's C5, most of it
// the chain of dependent reads from v to the table (820 ms without
// tables; of this step alone 285 to 108).
// Every c takes its value from the kept table; what is missing is computed by
// sweep_kept. Chunks of v are cut where they would hold more than kPairMax
// elements, so that the tail of a launch can still be split. Once the queue is
// drained they end at kPairTail elements, and a rest that would be long at the
// pace of the chunk just done is handed on (rest_is_long).
constexpr int kPairMax = 1 << 14, kPairTail = 1 << 11;
template <bool GS>
__device__ __forceinline__ void pair_leaf(const Ctx C, int d, int node, int cur, int hi, bool can_split) {
    const KArgs &a = C.a;
    WaveState *S = C.S;
    const int ln = C.ln;
    const GatNode &N = C.P.nodes[node], &M = C.P.nodes[N.child_begin];
    const GatOp &list = C.P.ops[N.op_begin], &o = C.P.ops[M.op_begin];
    const GatTerm &Tm = C.P.terms[M.term_begin];
    leaf_exclusions(C, M, d);
    unsigned tag;
    KeptEntry *tab = pool_table(C, o, &tag);
    const bool ex_v = o.excl >> d & 1u;
    // what the chosen vertices of the levels below d mean for every c: skip[],
    // the vertices c must differ from; less[], those to subtract where c is
    // adjacent to them (whether that is known: less_known) and they lie below t
    int skip[GATP_MAX_DEPTH], less[GATP_MAX_DEPTH], less_hub[GATP_MAX_DEPTH], n_skip = 0, n_less = 0;
    unsigned less_known = 0;
    const int in = uni(S->ex_in[o.leaf_idx]);
#pragma unroll
    for (int i = 0; i < GATP_MAX_DEPTH; i++) skip[i] = less[i] = less_hub[i] = 0;
    for (int f = 0; f < d; f++) {
        const int x = uni(S->val[f]), hx = uni(hub_of(a, x));
#pragma unroll
        for (int i = 0; i < GATP_MAX_DEPTH; i++) {  // constant indexes keep the arrays in registers
            if ((M.excl >> f & 1u) && i == n_skip) skip[i] = x;
            if ((in >> f & 1) && i == n_less) {
                less[i] = x;
                less_hub[i] = hx;
            }
        }
        if (M.excl >> f & 1u) n_skip++;
        if (in >> f & 1) {
            if (o.ex_cand >> f & 1u) less_known |= 1u << n_less;
            n_less++;
        }
    }
    unsigned levels = 0;
    for (int i = 0; i < o.ngroups; i++) levels |= o.groups[i];
    const bool t_lane = levels >> (d + 1) & 1u;  // the truncation depends on c
    const int t_all = t_lane ? 0 : uni(group_bound(S, o.groups, o.ngroups, d + 1, 0));
    unsigned long long sum = 0;
    int nl = W;
    for (int cb = cur; cb < hi; cb += nl) {
        const bool tail = can_split && queue_drained<GS>(a);
        const long long c0 = tail ? uni64(wall_clock64()) : 0;
        const int most = tail ? kPairTail : kPairMax;
        const int vi = cb + ln;
        int v = 0;
        if (vi < hi) v = with_slot<GS>(C, N.loop_slot, [&](auto p) { return p[vi]; });
        const bool use = vi < hi && !equals_any(S, N.excl, d, v);
        long long vb = 0;
        int len = 0;
        bool in_v = false;  // v is excluded from the COUNT and lies in its father
        if (use) {
            vb = a.off[v];
            const int t = min(group_bound(S, list.groups, list.ngroups, d, v), mask_bound(S, M.bound, d, v));
            len = trunc_len(a, v, vb, (int)(a.off[v + 1] - vb), t);
            in_v = ex_v;
        }
        if (ex_v && !(o.ex_father >> d & 1u))
            for (int l = 0; l < d; l++)
                if (o.levels >> l & 1u) {
                    const int x = uni(S->val[l]);
                    in_v = adjacent(a, x, uni(hub_of(a, x)), v, in_v);
                }
        int T = 0;
        int myoff = excl_scan(len, &T);
        nl = W;
        if (T > most) {
            nl = max(1, __popcll(ballot(myoff + len <= most)));  // a prefix of the lanes
            T = __shfl(myoff + len, nl - 1);
            if (ln >= nl) myoff = T;
        }
        constexpr int U = 2;  // steps in flight
        for (int k0 = 0; k0 < T; k0 += U * W) {
            int c[U], w[U], t[U];
            KeptEntry::Read e[U];
            bool live[U], wex[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int j = k0 + u * W + ln;
                c[u] = w[u] = 0;
                wex[u] = false;
                if (k0 + u * W < T)
                    by_owner(myoff, k0 + u * W, T, [&](const auto &pull) {
                        const long long s_vb = pull(vb);
                        const int s_off = pull(myoff);
                        w[u] = pull(v);
                        wex[u] = pull((int)in_v);
                        if (j < T) c[u] = a.adj[s_vb + (j - s_off)];
                    });
                live[u] = j < T;
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
#pragma unroll
                for (int i = 0; i < GATP_MAX_DEPTH; i++) {
                    if (i >= n_skip) break;
                    live[u] = live[u] && c[u] != skip[i];
                }
                live[u] = live[u] && !((M.excl >> d & 1u) && c[u] == w[u]);
                e[u] = {0, 0};  // tags start at 1
                if (live[u] && c[u] < a.tab_size) e[u] = tab[c[u]].read();
                t[u] = t_lane ? group_bound(S, o.groups, o.ngroups, d + 1, c[u]) : t_all;
            }
            int cnt[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                cnt[u] = 0;
#pragma unroll
                for (int i = 0; i < GATP_MAX_DEPTH; i++) {
                    if (i >= n_less) break;
                    const bool below = live[u] && less[i] < t[u];
                    if (less_known >> i & 1u) cnt[u] -= below;
                    else cnt[u] -= adjacent(a, less[i], less_hub[i], c[u], below);
                }
                if (live[u] && wex[u] && w[u] < t[u]) cnt[u]--;  // c lies in N(w)
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const bool need = live[u] && !e[u].serves(tag, a.epoch);
                int x = e[u].value();
                if (ballot(need)) {
                    const int fresh = sweep_kept<GS>(C, o.father, need, c[u], t[u]);
                    if (need) {
                        x = fresh;
                        if (c[u] < a.tab_size) tab[c[u]].write(tag, fresh, a.epoch);
                    }
                }
                if (live[u]) sum += (unsigned long long)(long long)(x + cnt[u]);
            }
        }
        const int left = hi - (cb + nl);
        if (!can_split || left < 2) continue;
        const bool long_rest = tail && rest_is_long(a, uni64(wall_clock64()) - c0, nl, left);
        if (long_rest && split_shallowest<GS>(C, d - 1)) continue;
        if ((long_rest || want_split<GS>(a, S)) && donate(C, d, node, cb + nl, hi, 1, !GS)) break;
    }
    sum = wave_sum64(sum);
    if (ln == 0) S->task_acc[Tm.pattern] += sum * (unsigned long long)(long long)C.P.subs[Tm.sub_begin].coef;
    wsync();
}

template <bool GS>
__device__ __forceinline__ void push_frame(const Ctx &C, int d, int node, int lo, int hi) {
    WaveState *S = C.S;
    const GatNode &N = C.P.nodes[node];
    const int ls = N.loop_slot;
    const int L = S->slen[ls];
    int hb = L;
    if (N.bound) {
        const int t = mask_bound(S, N.bound, d, 0);  // bound levels are all < d
        hb = uni(with_slot<GS>(C, ls, [&](auto p) { return lbound(p, L, t); }));
    }
    if (C.ln == 0) {
        S->f_node[d] = node;
        S->f_cur[d] = max(lo, 0);
        S->f_hi[d] = min(hi, hb);
    }
    wsync();
}

// Pending counts and W_alg of the edges finished since the last commit go
// into the wave's totals; an abandoned edge's are dropped instead.
__device__ __forceinline__ void commit_pending(WaveState *S, int np, int ln) {
    for (int i = ln; i < np; i += W) {
        S->wave_acc[i] += S->task_acc[i];
        S->task_acc[i] = 0;
    }
    if (ln == 0) {
        S->bytes += S->ebytes;
        S->ebytes = 0;
        S->n_don = 0;  // what this work handed on is final too
    }
    wsync();
}

__device__ __forceinline__ void drop_pending(WaveState *S, int np, int ln) {
    for (int i = ln; i < np; i += W) S->task_acc[i] = 0;
    if (ln == 0) {
        S->ebytes = 0;
        S->abort = 0;
    }
    wsync();
}

// Depth-first walk of the trie for the directed edges [e0, e1). When the
// root has one child (a single depth-1 node, so each edge is one subtree),
// an edge whose sets outgrow the LDS buffers is handed alone to the HBM
// launch and the walk goes on with the next edge; otherwise the whole task
// is abandoned and re-run there.
template <bool GS, bool KEEP, bool PAIR>
__device__ __forceinline__ void run_task(const Ctx &C, long long e0, long long e1) {
    const KArgs &a = C.a;
    const GatPlanDev &P = C.P;
    WaveState *S = C.S;
    const GatNode &root = P.nodes[0];
    const bool edge_grain = !GS && root.child_count == 1;
    long long e = e0;
    while (e < e1) {
        // row of edge e: last v with off[v] <= e
        int lo = 0, hi = a.n;  // invariant off[lo] <= e < off[hi]
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (a.off[mid] <= e) lo = mid; else hi = mid;
        }
        const int v0 = uni(lo);
        const long long rb = a.off[v0], re = a.off[v0 + 1];
        const long long se = e1 < re ? e1 : re;
        if (C.ln == 0) {
            S->val[0] = v0;
            S->rb = rb;
            S->sub_edge = -1;
            S->base_depth = 2;
            S->base_lo = 0;
        }
        wsync();
        for (int k = 0; k < root.op_count; k++) exec_op_uniform<GS>(C, P.ops[root.op_begin + k], 0, v0, false);
        wsync();
        const int lo1 = (int)(e - rb), hi1 = (int)(se - rb);
        int d = 1;
        push_frame<GS>(C, 1, root.child_begin, lo1, hi1);
        while (d >= 1) {
            const int node = uni(S->f_node[d]);
            const GatNode &N = P.nodes[node];
            bool exhausted = false;
            // loops at depth >= 2 may be handed to a split launch
            const bool can_split = d >= 2;
            if (N.leaf) {
                leaf<GS, KEEP>(C, N, d, uni(S->f_cur[d]), uni(S->f_hi[d]), can_split, node);
                exhausted = true;
            } else if (PAIR && N.pair && d >= 2) {
                const int cur = uni(S->f_cur[d]), fh = uni(S->f_hi[d]);
                if (can_split && cur < fh && due_to_split<GS>(a, S, d, cur, fh, C.ln) && split_shallowest<GS>(C, d)) continue;
                pair_leaf<GS>(C, d, node, cur, fh, can_split);
                exhausted = true;
            } else {
                const int cur = uni(S->f_cur[d]), fh = uni(S->f_hi[d]);
                if (can_split && cur < fh && due_to_split<GS>(a, S, d, cur, fh, C.ln) && split_shallowest<GS>(C, d)) continue;
                if (cur < fh) {
                    const int c = uni(with_slot<GS>(C, N.loop_slot, [&](auto p) { return p[cur]; }));
                    if (C.ln == 0) S->f_cur[d] = cur + 1;
                    wsync();
                    if (N.excl && equals_any(S, N.excl, d, c)) continue;
                    if (edge_grain && d == 1) commit_pending(S, P.n_patterns, C.ln);  // previous edge done
                    if (!visit<GS>(C, N, d, c)) {  // a set outgrew its LDS buffer
                        if (!edge_grain) return;  // the whole task goes to the HBM launch
                        if (C.ln == 0) {
                            const unsigned long long idx = atomicAdd(a.ovf_n, 1ull);
                            const long long edge = rb + (uni(S->f_cur[1]) - 1);
                            if ((long long)idx < a.ovf_cap) a.ovf[idx] = edge; else atomicOr(a.err, 2u);
                        }
                        cancel_donations(a, S, C.ln);
                        drop_pending(S, P.n_patterns, C.ln);
                        d = 1;
                        continue;
                    }
                    if (N.child_count > 0) {
                        d++;
                        push_frame<GS>(C, d, N.child_begin, 0, INT_MAX);
                    }
                    continue;
                }
                exhausted = true;
            }
            if (exhausted) {
                if (N.next_sibling >= 0)
                    push_frame<GS>(C, d, N.next_sibling, d == 1 ? lo1 : 0, d == 1 ? hi1 : INT_MAX);
                else
                    d--;
            }
        }
        e = se;
    }
    if (edge_grain) commit_pending(S, P.n_patterns, C.ln);
}

// Split subtask *g (in subs[]): the sets of the root and of the nodes on its
// path are rebuilt (neither counted nor accounted again), then the walk
// covers candidates [lo, hi) of its node and their subtrees only. A set that
// outgrows its LDS buffer leaves S->abort set (the HBM launch re-runs it).
template <bool GS, bool KEEP, bool PAIR>
__device__ __forceinline__ void run_sub(const Ctx &C, const SplitTask *g) {
    const KArgs &a = C.a;
    const GatPlanDev &P = C.P;
    WaveState *S = C.S;
    const long long e = uni64(g->edge);
    const int sub_node = uni(g->node), D = uni(g->depth), sub_lo = uni(g->lo), sub_hi = uni(g->hi);
    int lo = 0, hi = a.n;  // off[lo] <= e < off[hi]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (a.off[mid] <= e) lo = mid; else hi = mid;
    }
    const int v0 = uni(lo);
    const long long rb = a.off[v0];
    const unsigned long long eb = S->ebytes;
    if (C.ln == 0) {
        S->val[0] = v0;
        S->rb = rb;
        S->sub_edge = e;
        S->base_depth = D;
        S->base_lo = max(sub_lo, 0);
    }
    for (int j = 2 + C.ln; j < D; j += W) S->path_pos[j] = g->pos[j];
    wsync();
    const GatNode &root = P.nodes[0];
    for (int k = 0; k < root.op_count; k++) exec_op_uniform<GS>(C, P.ops[root.op_begin + k], 0, v0, false);
    wsync();
    bool ok = true;
    for (int j = 1; j < D && ok; j++) {
        int nj = sub_node;  // the ancestor of the subtask's node at depth j
        for (int t = D; t > j; t--) nj = P.nodes[nj].parent;
        const GatNode &Nj = P.nodes[nj];
        const int pos = j == 1 ? (int)(e - rb) : uni(S->path_pos[j]);
        const int vj = uni(with_slot<GS>(C, Nj.loop_slot, [&](auto p) { return p[pos]; }));
        ok = visit<GS>(C, Nj, j, vj, true);
    }
    if (C.ln == 0) S->ebytes = eb;
    wsync();
    if (!ok) return;
    const bool can_split = !GS && a.sub_mode < kSplitLevels;
    const int sum_op = KEEP ? uni(g->pos[0]) - 1 : -1;
    if (KEEP && sum_op >= 0) {
        if (C.ln == 0) {
            S->f_node[D] = sub_node;
            S->f_cur[D] = sub_lo;
            S->f_hi[D] = sub_hi;
        }
        wsync();
    } else {
        push_frame<GS>(C, D, sub_node, sub_lo, sub_hi);
    }
    int d = D;
    while (d >= D) {
        const int node = uni(S->f_node[d]);
        const GatNode &N = P.nodes[node];
        bool exhausted = false;
        if (N.leaf) {
            leaf<GS, KEEP>(C, N, d, uni(S->f_cur[d]), uni(S->f_hi[d]), can_split, node, sum_op);
            exhausted = true;
        } else if (PAIR && N.pair) {
            const int cur = uni(S->f_cur[d]), fh = uni(S->f_hi[d]);
            if (can_split && cur < fh && due_to_split<GS>(a, S, d, cur, fh, C.ln) && split_shallowest<GS>(C, d)) continue;
            pair_leaf<GS>(C, d, node, cur, fh, can_split);
            exhausted = true;
        } else {
            const int cur = uni(S->f_cur[d]), fh = uni(S->f_hi[d]);
            if (can_split && cur < fh && due_to_split<GS>(a, S, d, cur, fh, C.ln) && split_shallowest<GS>(C, d)) continue;
            if (cur < fh) {
                const int c = uni(with_slot<GS>(C, N.loop_slot, [&](auto p) { return p[cur]; }));
                if (C.ln == 0) S->f_cur[d] = cur + 1;
                wsync();
                if (N.excl && equals_any(S, N.excl, d, c)) continue;
                if (!visit<GS>(C, N, d, c)) return;
                if (N.child_count > 0) {
                    d++;
                    push_frame<GS>(C, d, N.child_begin, 0, INT_MAX);
                }
                continue;
            }
            exhausted = true;
        }
        if (exhausted) {
            if (d > D && N.next_sibling >= 0)
                push_frame<GS>(C, d, N.next_sibling, 0, INT_MAX);
            else
                d--;
        }
    }
}

// The array-store kernels read their arguments from device memory (written
// by put_kargs before the count's launches): the walk hands a reference to them
// to out-of-line helpers, and a reference to a by-value kernel argument
// would make every lane copy the whole record to scratch first.
constexpr int kArgSlots = kSplitLevels + 3;  // the main launch, the LDS subtask levels, the HBM launch and its subtasks
struct KArgsSet {
    KArgs a[kArgSlots];
};
static_assert(sizeof(KArgsSet) <= 4000, "kernel arguments");
__global__ void put_kargs(KArgsSet set, KArgsSet *dst) {
    const int *src = reinterpret_cast<const int *>(&set);
    for (int i = threadIdx.x; i < (int)(sizeof(KArgsSet) / sizeof(int)); i += blockDim.x)
        reinterpret_cast<int *>(dst)[i] = src[i];
}

template <bool GS, bool KEEP, bool PAIR>
__device__ __forceinline__ void engine_main(const KArgs *__restrict__ ap, int wave_bytes, unsigned char *smem) {
    const KArgs &a = *ap;
    const int wid = threadIdx.x / W, ln = threadIdx.x % W;
    const int wpb = blockDim.x / W;
    WaveState *S = reinterpret_cast<WaveState *>(smem + (size_t)wid * wave_bytes);
    const GatPlanDev &P = *a.plan;
    int *store;
    if (GS)
        store = a.gstore + (long long)(blockIdx.x * wpb + wid) * P.n_store * (long long)a.cap;
    else
        store = reinterpret_cast<int *>(smem + (size_t)wid * wave_bytes + a.state_bytes);
    Ctx C{a, P, S, store, ln};
    const int np = P.n_patterns;
    const long long tl_t0 = wall_clock64();
    long long tl_items = 0;
    for (int i = ln; i < np; i += W) S->wave_acc[i] = 0;
    if (ln == 0) {
        S->bytes = 0;
        S->ebytes = 0;
    }
    wsync();
    int head = (int)((blockIdx.x * wpb + wid) % kHeads);
    const long long items = GS ? ((long long)*a.ovf_n < a.ovf_cap ? (long long)*a.ovf_n : a.ovf_cap)
                               : (a.e_hi - a.e_lo + a.chunk - 1) / a.chunk;
    for (;;) {
        long long e0;  // the task: directed edges [e0, e0 + chunk)
        const long long r = queue_next(a.queue, a.drained, GS ? kQueueOverflow : kQueueMain, items, &head, ln);
        if (r < 0) break;
        e0 = GS ? uni64(a.ovf[r]) : a.e_lo + r * a.chunk;
        tl_items++;
        for (int i = ln; i < np; i += W) S->task_acc[i] = 0;
        if (ln == 0) {
            S->abort = 0;
            S->n_don = 0;
            S->t0 = wall_clock64();
        }
        wsync();
        run_task<GS, KEEP, PAIR>(C, e0, e0 + a.chunk < a.e_hi ? e0 + a.chunk : a.e_hi);
        wsync();
        if (S->abort) {
            if (GS) {
                if (ln == 0) atomicOr(a.err, 1u);  // cannot happen: HBM buffers hold max degree
            } else {
                cancel_donations(a, S, ln);
                if (ln == 0) {
                    const unsigned long long idx = atomicAdd(a.ovf_n, 1ull);
                    if ((long long)idx < a.ovf_cap) a.ovf[idx] = e0; else atomicOr(a.err, 2u);
                }
            }
            if (ln == 0) S->ebytes = 0;  // the HBM launch does this task again
        } else {
            for (int i = ln; i < np; i += W) S->wave_acc[i] += S->task_acc[i];
            if (ln == 0) {
                S->bytes += S->ebytes;
                S->ebytes = 0;
            }
        }
        wsync();
    }
    for (int i = ln; i < np; i += W)
        if (S->wave_acc[i]) atomicAdd(&count_copy(a.counts)[i], S->wave_acc[i]);
    if (a.account && ln == 0 && S->bytes) atomicAdd(a.bytes, S->bytes);
    if (a.tl && ln == 0)
        tl_write(a.tl, a.tl_base + blockIdx.x * wpb + wid, GS ? kLevelsHbm : 0, blockIdx.x * wpb + wid, tl_t0,
                 wall_clock64(), 0, 0, tl_items, 0);
}

// Subtask launches: list sub_mode (1 .. kSplitLevels: LDS buffers; then the
// HBM list with HBM buffers). A subtask that outgrows LDS is copied to the
// HBM list for the last launch.
template <bool GS, bool KEEP, bool PAIR>
__device__ __forceinline__ void engine_sub(const KArgs *__restrict__ ap, int wave_bytes, unsigned char *smem) {
    const KArgs &a = *ap;
    const int wid = threadIdx.x / W, ln = threadIdx.x % W;
    const int wpb = blockDim.x / W;
    WaveState *S = reinterpret_cast<WaveState *>(smem + (size_t)wid * wave_bytes);
    const GatPlanDev &P = *a.plan;
    int *store;
    if (GS)
        store = a.gstore + (long long)(blockIdx.x * wpb + wid) * P.n_store * (long long)a.cap;
    else
        store = reinterpret_cast<int *>(smem + (size_t)wid * wave_bytes + a.state_bytes);
    Ctx C{a, P, S, store, ln};
    const int np = P.n_patterns;
    const long long tl_t0 = wall_clock64();
    long long tl_items = 0;
    for (int i = ln; i < np; i += W) S->wave_acc[i] = 0;
    if (ln == 0) {
        S->bytes = 0;
        S->ebytes = 0;
    }
    wsync();
    int head = (int)((blockIdx.x * wpb + wid) % kHeads);
    const unsigned long long made = *a.in_n;
    const long long items = (long long)made < a.in_cap ? (long long)made : a.in_cap;
    for (;;) {
        const long long r = queue_next(a.queue, a.drained, kQueueSub + a.sub_mode, items, &head, ln);
        if (r < 0) break;
        const SplitTask *g = a.subs + a.in_base + r;
        tl_items++;
        for (int i = ln; i < np; i += W) S->task_acc[i] = 0;
        if (ln == 0) {
            S->abort = 0;
            S->n_don = 0;
            S->t0 = wall_clock64();
        }
        wsync();
        if (uni(g->lo) < uni(g->hi)) run_sub<GS, KEEP, PAIR>(C, g);
        wsync();
        if (S->abort) {
            if (GS) {
                if (ln == 0) atomicOr(a.err, 1u);  // cannot happen: HBM buffers hold max degree
            } else {
                cancel_donations(a, S, ln);
                unsigned long long idx = 0;
                if (ln == 0) idx = atomicAdd(a.sovf_n, 1ull);
                idx = (unsigned long long)uni64((long long)__shfl(idx, 0));
                if ((long long)idx < a.sovf_cap) {
                    SplitTask *t = a.subs + a.sovf_base + idx;
                    for (int k = ln; k < (int)(sizeof(SplitTask) / sizeof(int)); k += W)
                        reinterpret_cast<int *>(t)[k] = reinterpret_cast<const int *>(g)[k];
                } else if (ln == 0) {
                    atomicOr(a.err, 2u);
                }
                if (ln == 0) atomicAdd(&a.ovf_n[2], 1ull);  // statistics
            }
            if (ln == 0) S->ebytes = 0;
        } else {
            for (int i = ln; i < np; i += W) S->wave_acc[i] += S->task_acc[i];
            if (ln == 0) {
                S->bytes += S->ebytes;
                S->ebytes = 0;
            }
        }
        wsync();
    }
    for (int i = ln; i < np; i += W)
        if (S->wave_acc[i]) atomicAdd(&count_copy(a.counts)[i], S->wave_acc[i]);
    if (a.account && ln == 0 && S->bytes) atomicAdd(a.bytes, S->bytes);
    if (a.tl && ln == 0)
        tl_write(a.tl, a.tl_base + blockIdx.x * wpb + wid, a.sub_mode + (GS ? 1 : 0), blockIdx.x * wpb + wid, tl_t0,
                 wall_clock64(), 0, 0, tl_items, 0);
}

// Kernels of plans that keep COUNT values in tables, and of those that do not
// (and of W_alg accounting, which charges every value): the code of the tables
// costs the others 8 % (C4 + P4 on a sparse random graph), and that of
// pair_leaf costs plans without pair nodes 15 % (house on Chung-Lu 65,536).
template <bool GS>
__global__ void __launch_bounds__(256, 4) engine_kernel(const KArgs *__restrict__ ap, int wave_bytes) {
    extern __shared__ __align__(16) unsigned char smem[];
    engine_main<GS, true, false>(ap, wave_bytes, smem);
}
template <bool GS>
__global__ void __launch_bounds__(256, 4) engine_sub_kernel(const KArgs *__restrict__ ap, int wave_bytes) {
    extern __shared__ __align__(16) unsigned char smem[];
    engine_sub<GS, true, false>(ap, wave_bytes, smem);
}
template <bool GS>
__global__ void __launch_bounds__(256, 4) engine_pair_kernel(const KArgs *__restrict__ ap, int wave_bytes) {
    extern __shared__ __align__(16) unsigned char smem[];
    engine_main<GS, true, true>(ap, wave_bytes, smem);
}
template <bool GS>
__global__ void __launch_bounds__(256, 4) engine_pair_sub_kernel(const KArgs *__restrict__ ap, int wave_bytes) {
    extern __shared__ __align__(16) unsigned char smem[];
    engine_sub<GS, true, true>(ap, wave_bytes, smem);
}
template <bool GS>
__global__ void __launch_bounds__(256) engine_plain_kernel(const KArgs *__restrict__ ap, int wave_bytes) {
    extern __shared__ __align__(16) unsigned char smem[];
    engine_main<GS, false, false>(ap, wave_bytes, smem);
}
template <bool GS>
__global__ void __launch_bounds__(256) engine_plain_sub_kernel(const KArgs *__restrict__ ap, int wave_bytes) {
    extern __shared__ __align__(16) unsigned char smem[];
    engine_sub<GS, false, false>(ap, wave_bytes, smem);
}

// ---------------------------------------------------------------------------
// Bitmap vertex store for clique plans (the reference declares
// VertexStoreType::Bitmap in include/configs/vertex_set_config.hpp:3-6 but
// never implements it). On the degree-oriented graph every k-clique is a
// chain v0 > v1 > ... with v_{i+1} in N+(v_i). Per vertex v0 with list
// L = N+(v0) (sorted, d entries) the oriented adjacency of the subgraph
// induced on L is built as bit rows over positions in L:
//   M_p = { q < p : L[q] in N+(L[p]) }.
// Every clique with top vertex v0 is then a clique of these rows:
//   #K3 += sum_p popc(M_p)
//   #K4 += sum_p sum_{q in M_p} popc(M_p & M_q)
//   #K5 += sum over q in M_p, r in M_p & M_q of popc(M_p & M_q & M_r)
//   #K6 one level deeper.
//
// Rows. One ballot of the wave gives 64 bits of a row: lane q tests whether
// L[q] lies in N+(L[p]) with one word of the core bitmap (dense rows of the
// first core_n vertices, see core_row), or by a search of the list when L[p]
// is not a core vertex. That is d^2/128 wave steps for a vertex, with no
// shared writes; the sweep of the lists N+(L[p]) it replaces took
// sum_p |N+(L[p])| / 64 steps with a hash probe and an LDS atomic each (on
// R-MAT s20: 2 to 13 times more steps for d >= 16).
//
// Tiers by d: the main launch gives a vertex with d <= CMAIN (64) one wave,
// whose rows are single 64-bit words; larger vertices are shared by the
// waves of a workgroup with rows in LDS (d <= 256, 512, 1024) or in HBM.
constexpr int CMAXD = 256;  // largest slot_capacity the clique store honours
constexpr int CMAIN = 64;   // main launch: d <= min(CMAIN, slot_capacity)
constexpr int CDEFER = 32;  // #K6: it hands on denser vertices with d > CDEFER
constexpr int CT0W = 8;     // workgroup tier 0: rows of 8 words, d <= 256
constexpr int CT1W = 16;    // workgroup tier 1: d <= 512
constexpr int CT2W = 32;    // workgroup tier 2: d <= 1024
constexpr int CTIERS = 4;   // tier 3: any d, rows in HBM
// Items of a tier's queue: clique_parts() per vertex, which share out its
// counting (each builds the rows). One part when the vertices fill the
// launch's workgroups four times over, else more, up to what the depth of the
// counting pays for: with whole vertices the last ones of R-MAT s20's tier 2
// (665 vertices, 256 workgroups) end unevenly, and a single vertex of 259
// neighbours took 3.7 ms for #K6 on one workgroup.
__host__ __device__ constexpr int clique_max_parts(int kmax) {
    return kmax >= 6 ? 16 : kmax == 5 ? 8 : kmax == 4 ? 4 : 1;
}
__device__ __forceinline__ int clique_parts(int kmax, unsigned long long vertices, int groups) {
    const unsigned long long want = 4ull * groups, mx = clique_max_parts(kmax);
    const unsigned long long p = vertices ? (want + vertices - 1) / vertices : 1;
    return (int)(p < mx ? p : mx);
}
// Waves per workgroup: enough to share one vertex's work, few enough that
// the workgroups of a CU (bounded by LDS, 11, 37 and 139 KB each, and by
// registers) overlap one's row build with another's counting.
constexpr int CNW0 = 4, CNW1 = 4, CNW2 = 8, CNW3 = 16;
// Waves per SIMD that the tiers' registers are held to. Tiers 0 and 1 spill for it
// (93 and 11 registers): without spills, with three and two waves, K4 + K5 on
// R-MAT s20 takes 14.3 ms instead of 12.1 (K4 on R-MAT s14 149 us instead of 167).
constexpr int clique_occupancy(int tier) { return tier == 0 ? 4 : tier == 1 ? 3 : 2; }
// Words per bit row of a list of d vertices: enough for d bits, rounded up
// to an odd number so that lanes reading the same word of different rows
// hit different LDS banks (an even stride folds them onto a few banks).
__host__ __device__ constexpr int row_words(int d) { return ((d + 31) >> 5) | 1; }
// LDS of a workgroup tier with rows of up to mw words: the rows of lcap = 32
// mw vertices, slack for the chunks of four words the matrix operands are
// read in, and the waves' column lists (the list L shares their space: it is
// not needed once the rows are built).
__host__ __device__ constexpr int tier_row_words(int mw) { return 32 * mw * row_words(32 * mw) + 8; }
constexpr size_t tier_lds(int mw, int nw) {
    return (size_t)4 * tier_row_words(mw) + (size_t)4 * (32 * mw > 128 * nw ? 32 * mw : 128 * nw);
}

// Core bitmap: for x < core_n, row x holds bit y set iff y in N+(x), y < x,
// in ceil(x / 32) words; the rows follow one another from x = 1 on.
__host__ __device__ __forceinline__ unsigned core_row(int x) {
    if (x < 1) return 0;
    const unsigned k = (unsigned)(x - 1) >> 5;
    return (k + 1) * ((unsigned)(x - 1) - 16 * k);
}

struct CArgs {
    const long long *off;
    const int *adj;
    const int *split;
    const unsigned *core;        // core bitmap
    int core_n;                  // its vertices: [0, core_n)
    int n;
    long long m;
    int root_lo, root_hi;        // top vertices of this count: [root_lo, root_hi)
    unsigned long long *counts;
    int pat_of_k[8];
    int kmax;
    unsigned long long *queue;   // [0] main vertex queue, [1 + t] workgroup tier t
    int *tier[CTIERS];           // vertices of the workgroup tiers
    long long tier_cap[CTIERS];
    // [t] vertices of tier t, [4] vertices with d > cap, [5] of those the
    // ones with d <= 512
    unsigned long long *ovf_n;
    unsigned long long *bytes;   // W_alg accumulator of this launch
    unsigned int *err;
    unsigned *grows;             // HBM tier: per-workgroup rows, hcap * row_words(hcap) words
    int *goff;                   // HBM tier: per-workgroup pair offsets, hcap + 1 entries
    int hcap;                    // HBM tier capacity (>= maximum out-degree)
    int lds_dmax;                // largest d of the LDS tiers
    int account;
    int cap;                     // slot_capacity as the clique store takes it
    int main_max;                // largest d of the main launch: min(CMAIN, cap)
    int chunk;                   // vertices per main-queue grab
    long long *tl;               // timeline records (GAT_FLAG_TIMELINE), or null
    int tl_base;                 // first record of this launch
};

// hit[u] |= y[u] in the n[u] entries from a.adj[base[u]] on: U searches of lists
// side by side, so that a round of them waits for one memory latency.
template <int U>
__device__ __forceinline__ void search_below(const CArgs &a, long long (&base)[U], int (&n)[U], const int (&y)[U],
                                             bool (&hit)[U]) {
    int longest = 0;
#pragma unroll
    for (int u = 0; u < U; u++) longest = max(longest, n[u]);
    // halve every list until one entry is left (the last entry <= y, if any)
    while (ballot(longest > 1)) {
        int v[U];
#pragma unroll
        for (int u = 0; u < U; u++) v[u] = n[u] > 1 ? a.adj[base[u] + (n[u] >> 1)] : INT_MAX;
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int half = n[u] >> 1;
            if (v[u] <= y[u]) base[u] += half;
            if (n[u] > 1) n[u] -= half;
        }
        longest -= longest >> 1;
    }
#pragma unroll
    for (int u = 0; u < U; u++) hit[u] |= n[u] > 0 && a.adj[base[u]] == y[u];
}

// Rows of the list L (d entries) for p = first, first + stride, ... (a
// workgroup's waves interleave their rows, so light and heavy rows mix), w
// words each, all of them written. Returns the bits set (the pairs of these
// rows). R rows and two ballots of each are taken at a time, so that 2 R reads
// are in flight (one row at a time: 2.0 instead of 1.8 ms for the rows of
// R-MAT s20's tier 0; 8 rows are no faster than 4).
template <bool ACC, class LP, class RP>
__device__ __forceinline__ unsigned long long vtx_rows(const CArgs &a, LP L, int d, RP rows, int w, int first,
                                                       int stride, int ln, unsigned long long &bytes) {
    constexpr int R = 4;
    unsigned long long pairs = 0;
    auto put = [&](int p, int b, unsigned long long m) {  // the 64 bits of ballot b of row p
        pairs += __popcll(m);
        const int k = 2 * b + ln;
        if (ln < 2 && k < w) rows[(long long)p * w + k] = ln ? (unsigned)(m >> 32) : (unsigned)m;
    };
    for (int p0 = first; p0 < d; p0 += R * stride) {
        const int last = min(R - 1, (d - 1 - p0) / stride);  // rows p0 + j stride, j = 0 .. last
        const int nb = (p0 + last * stride + W - 1) / W;      // ballots of the longest of them
        int x[R];
#pragma unroll
        for (int j = 0; j < R; j++) x[j] = uni(L[p0 + min(j, last) * stride]);
        if (ACC && ln == 0)
            for (int j = 0; j <= last; j++) {
                const int p = p0 + j * stride;
                bytes += 4ull * (a.split[x[j]] + p) + 16ull + 4ull * ((p >> 5) + 1);
            }
        if (x[R - 1] < a.core_n) {  // the largest of the x
            const unsigned *cr[R];
#pragma unroll
            for (int j = 0; j < R; j++) cr[j] = a.core + core_row(x[j]);
            for (int b = 0; b < nb; b += 2) {
                unsigned v[2][R];
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const int q = (b + u) * W + ln;
                    const int y = q < d ? L[q] : 0;
#pragma unroll
                    for (int j = 0; j < R; j++) {
                        v[u][j] = 0;
                        if (q < p0 + j * stride && j <= last) v[u][j] = cr[j][y >> 5] >> (y & 31);
                    }
                }
#pragma unroll
                for (int u = 0; u < 2; u++)
#pragma unroll
                    for (int j = 0; j < R; j++)
                        if (j <= last) put(p0 + j * stride, b + u, ballot(v[u][j] & 1u));
            }
        } else {
            long long xb[R];
            int xn[R];
#pragma unroll
            for (int j = 0; j < R; j++) {
                xb[j] = a.off[x[j]];
                xn[j] = a.split[x[j]];
            }
            for (int b = 0; b < nb; b++) {
                const int q = b * W + ln;
                int y[R], n[R];
                long long base[R];
                bool hit[R];
#pragma unroll
                for (int j = 0; j < R; j++) {
                    const bool in = j <= last && q < p0 + j * stride, core = x[j] < a.core_n;
                    y[j] = in ? L[q] : 0;
                    hit[j] = in && core && (a.core[core_row(x[j]) + (y[j] >> 5)] >> (y[j] & 31) & 1u);
                    base[j] = xb[j];
                    n[j] = in && !core ? xn[j] : 0;
                }
                search_below<R>(a, base, n, y, hit);
#pragma unroll
                for (int j = 0; j < R; j++)
                    if (j <= last) put(p0 + j * stride, b, ballot(hit[j]));
            }
        }
        const int done = x[R - 1] < a.core_n ? 2 * ((nb + 1) / 2 * 2) : 2 * nb;  // words written
        for (int j = 0; j <= last; j++)
            for (int k = done + ln; k < w; k += W) rows[(long long)(p0 + j * stride) * w + k] = 0u;
    }
    return pairs;
}

// ---- counting on the matrix cores ------------------------------------------
// The deepest two levels of a clique count are, for a set T of positions (the
// AND of 1, 2 or 3 rows for #K4, #K5, #K6: one "column"),
//   sum_{r in T} |T & M_r| = sum_r [r in T] |T & M_r|,   and one level up |T|.
// Both factors are products over positions of 0/1 vectors: for 16 columns and
// the 16 rows of a tile of consecutive positions r, the counts |T & M_r| are
// one 16x16x128 matrix instruction per 128 positions with operands M_r and T,
// and the bits [r in T] are one more with unit vectors e_r in the place of
// M_r. The operands are 4-bit floats (2.0, 1.0 or 0.5, their products always
// 1), made from a word of a row by shifts and masks: lane i + 16 g of an
// operand holds word g of the row's 128-bit chunk, so one LDS word is one
// lane's operand, and the order of the 32 positions within it is the same on
// both sides. The sums of a batch of columns are taken in FP32, below 2^24.
//
// A wave keeps RT row tiles (a group of 16 RT positions) in registers and
// streams its columns past them, 16 at a time from a list in LDS, whatever
// set they come from: the tiles are full even where the sets are small. Only
// columns with an element above the group's first position are listed. The
// pair walk this replaces spent about 100 lane-instructions per triple (find
// the next bit, read two words of its row, AND, popcount) with half of the
// lanes idle; here a column tile costs RT (chunks + 1) matrix instructions of
// 16 cycles and about half as many cycles of vector instructions. R-MAT s20,
// K4 + K5, tiers 0 to 2: 28.0 ms with the pair walk and swept rows, 10.6 ms
// with this (rows 2.6 ms of it); K6 on R-MAT s16: 840 ms against 5.4 ms. The
// tiles in registers are what counts, because every column tile is read and
// unpacked once per group: two row tiles instead of four cost 2 ms in tier 1
// and 0.25 ms in tier 2 (in spite of 12 waves per CU instead of 8); eight in
// tier 1, with two waves per SIMD instead of three, cost 1 ms.
typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
constexpr int kFp4 = 4;  // operand format of the instruction: 4-bit float
__device__ __forceinline__ v4i operand_rows(unsigned x) {  // bits 0..3 of each nibble as 2.0, 1.0, 0.5, 0.5
    return v4i{(int)((x << 2) & 0x44444444u), (int)(x & 0x22222222u), (int)((x >> 2) & 0x11111111u),
               (int)((x >> 3) & 0x11111111u)};
}
__device__ __forceinline__ v4i operand_cols(unsigned x) {  // ... as 0.5, 1.0, 2.0, 2.0
    return v4i{(int)(x & 0x11111111u), (int)(x & 0x22222222u), (int)(x & 0x44444444u), (int)((x >> 1) & 0x44444444u)};
}
// 4-bit operands take four registers; scale arguments 0 select the unscaled form.
__device__ __forceinline__ v4f mfma_bits(v4i rows, v4i cols, v4f c) {
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
        __builtin_shufflevector(rows, rows, 0, 1, 2, 3, -1, -1, -1, -1),
        __builtin_shufflevector(cols, cols, 0, 1, 2, 3, -1, -1, -1, -1), c, kFp4, kFp4, 0, 0, 0, 0);
}

constexpr int CCOLS = 64;  // columns a wave lists before it counts them

// Counts of the columns of the rows p = first, first + stride, ... < d by one
// wave: DEPTH 1: M_p; 2: M_p & M_q, q in M_p; 3: M_p & M_q & M_x, x in M_p &
// M_q. deep += sum |T & M_r| over r in T, mid += |T|; for DEPTH 3 cols +=
// number of columns. KC: chunks of 128 positions a row can have; buf: 2 CCOLS
// entries of this wave in LDS. Row 0 has no bits: entry 0 pads a tile.
template <int KC, int RT, int DEPTH, bool ACC>
__device__ __forceinline__ void count_columns(const unsigned *rows, int w, int d, unsigned *buf, int first, int stride,
                                              int ln, unsigned long long &deep, unsigned long long &mid,
                                              unsigned long long &cols, unsigned long long &bytes) {
    constexpr int GP = 16 * RT;  // positions of a row group
    const int i = ln & 15, g = ln >> 4;
    for (int r0 = 0; r0 < d; r0 += GP) {
        const int khi = (min(d, r0 + GP) - 1) >> 7;  // the chunk of the group; rows have bits up to there
        v4i A[RT][KC], E[RT];
#pragma unroll
        for (int t = 0; t < RT; t++) {
            const int r = r0 + 16 * t + i;
            const unsigned *rr = rows + __umul24(min(r, d - 1), w) + g;
#pragma unroll
            for (int k = 0; k < KC; k++) {
                if (k > khi) break;
                A[t][k] = operand_rows(4 * k + g < w ? rr[4 * k] : 0u);
            }
            E[t] = operand_rows(r < d && (r >> 5) == 4 * khi + g ? 1u << (r & 31) : 0u);
        }
        // the group's own words of a column: this lane's word of chunk khi
        const int own = 4 * khi + g;
        const unsigned own_mask = own >= r0 >> 5 && own <= (r0 + GP - 1) >> 5 && own < w ? ~0u : 0u;
        unsigned size = 0;
        float tri = 0.f;
        auto tile = [&](int at) {  // the 16 columns buf[at ..]
            const unsigned e = buf[at + i];
            const unsigned *r1 = rows + __umul24((int)(e & 1023u), w) + g;
            const unsigned *r2 = rows + __umul24((int)(e >> 10 & 1023u), w) + g;
            const unsigned *r3 = rows + __umul24((int)(e >> 20), w) + g;
            v4f D[RT] = {}, M[RT] = {};
#pragma unroll
            for (int k = 0; k < KC; k++) {
                if (k > khi) break;
                unsigned c = r1[4 * k];
                if (DEPTH >= 2) c &= r2[4 * k];
                if (DEPTH >= 3) c &= r3[4 * k];
                const v4i B = operand_cols(c);
#pragma unroll
                for (int t = 0; t < RT; t++) D[t] = mfma_bits(A[t][k], B, D[t]);
                if (k == khi) {
#pragma unroll
                    for (int t = 0; t < RT; t++) M[t] = mfma_bits(E[t], B, M[t]);
                    const unsigned n = __popc(c & own_mask);
                    size += n;
                    if (ACC) bytes += 8ull * n * (own + 1);
                }
            }
#pragma unroll
            for (int t = 0; t < RT; t++)
#pragma unroll
                for (int x = 0; x < 4; x++) tri += D[t][x] * M[t][x];
        };
        int n = 0;
        // the last CCOLS columns listed; their sums are below 2^24, so exact
        auto batch = [&]() {
            n -= CCOLS;
#pragma unroll 1
            for (int c = 0; c < CCOLS; c += 16) tile(n + c);
            deep += (unsigned)tri;
            tri = 0.f;
            wsync();
        };
        auto list = [&](unsigned long long m, int b, unsigned entry, int shift) {  // a column per bit of m
            if (m >> ln & 1ull) {
                buf[n + mbcnt(m)] = entry | (unsigned)(b * W + ln) << shift;
                if (ACC && r0 == 0) bytes += 8ull * (((b * W + ln) >> 5) + 1);
            }
            n += __popcll(m);
            wsync();
            if (n >= CCOLS) batch();
        };
        // bits of the 64-position block b at or above the group's first position
        auto above = [&](int b) { return b * W >= r0 ? ~0ull : ~0ull << (r0 & (W - 1)); };
        auto block = [&](unsigned word, int b) {  // block b of the words the lanes hold
            return ((unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)word, 2 * b + 1) << 32 |
                    (unsigned)__builtin_amdgcn_readlane((int)word, 2 * b)) & above(b);
        };
        if (DEPTH == 1) {
            for (int p = r0 + 1 + first; p < d; p += stride * W) {  // lanes list their rows
                const int q = p + ln * stride;
                const unsigned long long m = ballot(q < d);
                if (q < d) buf[n + mbcnt(m)] = (unsigned)q;
                n += __popcll(m);
                wsync();
                if (n >= CCOLS) batch();
            }
        } else {
            // rows p of this wave above the group, the next row's words read ahead
            int p = first;
            if (p <= r0) p += (r0 + stride - first) / stride * stride;
            unsigned next = p < d && ln < w ? rows[p * w + ln] : 0u;
            for (; p < d; p += stride) {
                const unsigned word = next;
                next = p + stride < d && ln < w ? rows[(p + stride) * w + ln] : 0u;
                for (int b = r0 / W; b * W < p; b++) {
                    unsigned long long m = block(word, b);
                    if (DEPTH == 2) {
                        if (m) list(m, b, (unsigned)p, 10);
                    } else {
                        for (; m; m &= m - 1) {
                            const int q = b * W + __ffsll((long long)m) - 1;
                            if (ACC && r0 == 0 && ln == 0) bytes += 8ull * ((q >> 5) + 1);
                            const unsigned both = word & (ln < w ? rows[q * w + ln] : 0u);
                            for (int c = r0 / W; c * W < q; c++) {
                                const unsigned long long mm = block(both, c);
                                if (r0 == 0 && ln == 0) cols += (unsigned long long)__popcll(mm);
                                if (mm) list(mm, c, (unsigned)p | (unsigned)q << 10, 20);
                            }
                        }
                    }
                }
            }
        }
        if (n) {
            if (ln < (-n & 15)) buf[n + ln] = 0u;
            wsync();
#pragma unroll 1
            for (int c = 0; c < n; c += 16) tile(c);
            deep += (unsigned)tri;
            wsync();
        }
        mid += size;
    }
}

// Position of the j-th set bit (0-based) of x, j < popc(x).
__device__ __forceinline__ int select_bit(unsigned x, int j) {
    int pos = 0, c;
    c = __popc(x & 0xffffu);
    if (j >= c) { j -= c; x >>= 16; pos += 16; }
    c = __popc(x & 0xffu);
    if (j >= c) { j -= c; x >>= 8; pos += 8; }
    c = __popc(x & 0xfu);
    if (j >= c) { j -= c; x >>= 4; pos += 4; }
    c = __popc(x & 0x3u);
    if (j >= c) { j -= c; x >>= 2; pos += 2; }
    if (j >= (int)(x & 1u)) pos += 1;
    return pos;
}

// HBM tier: counts at and below the pair level, one pair per lane. The pairs
// (p, q), q in M_p, are numbered through off[p] = sum of popc(M_p') over p' <
// p (off[d] = P); worker k takes pairs first, first + step, ... For a pair:
// t = M_p & M_q gives #K4 += popc(t); each r in t adds popc(t & M_r) to #K5;
// each s in t & M_r adds popc(t & M_r & M_s) to #K6.
template <bool ACC>
__device__ void vtx_pairs(const CArgs &a, const unsigned *rows, int d, int w, const int *off, int P, int first,
                          int step, unsigned long long *acc, unsigned long long &bytes) {
    for (int k = first; k < P; k += step) {
        int lo = 0, hi = d;  // off[lo] <= k < off[hi]
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (off[mid] <= k) lo = mid; else hi = mid;
        }
        const unsigned *rp = rows + (long long)lo * w;
        int j = k - off[lo];
        int q = 0;
        for (int u = 0; u <= (lo >> 5); u++) {
            const unsigned x = rp[u];
            const int c = __popc(x);
            if (j < c) {
                q = u * 32 + select_bit(x, j);
                break;
            }
            j -= c;
        }
        const int wq = (q >> 5) + 1;
        if (ACC) bytes += 8ull * wq;
        const unsigned *rq = rows + (long long)q * w;
        unsigned c4 = 0;
        for (int u = 0; u < wq; u++) c4 += __popc(rp[u] & rq[u]);
        acc[4] += c4;
        if (a.kmax < 5) continue;
        unsigned long long c5 = 0;
        for (int rw = 0; rw < wq; rw++) {
            unsigned br = rp[rw] & rq[rw];
            while (br) {
                const int r = rw * 32 + __ffs(br) - 1;
                br &= br - 1;
                const unsigned *rr = rows + (long long)r * w;
                if (ACC) bytes += 8ull * (rw + 1);
                for (int u = 0; u <= rw; u++) c5 += __popc(rp[u] & rq[u] & rr[u]);
                if (a.kmax < 6) continue;
                unsigned long long c6 = 0;
                for (int sw = 0; sw <= rw; sw++) {
                    unsigned bs = rp[sw] & rq[sw] & rr[sw];
                    while (bs) {
                        const int sx = sw * 32 + __ffs(bs) - 1;
                        bs &= bs - 1;
                        const unsigned *rs = rows + (long long)sx * w;
                        if (ACC) bytes += 8ull * ((sx >> 5) + 1);
                        for (int u = 0; u <= (sx >> 5); u++) c6 += __popc(rp[u] & rq[u] & rr[u] & rs[u]);
                    }
                }
                acc[6] += c6;
            }
        }
        acc[5] += c5;
    }
}

template <bool ACC>
__device__ __forceinline__ void clique_flush(const CArgs &a, unsigned long long *acc, unsigned long long bytes,
                                             int ln) {
    for (int k = 3; k <= 6; k++) acc[k] = wave_sum64(acc[k]);
    if (ACC) bytes = wave_sum64(bytes);
    if (ln == 0) {
        for (int k = 3; k <= 6; k++)
            if (a.pat_of_k[k] >= 0 && acc[k]) atomicAdd(&count_copy(a.counts)[a.pat_of_k[k]], acc[k]);
        if (ACC && bytes) atomicAdd(a.bytes, bytes);
    }
}

// Largest d whose pairs all fit one 64-bit word: d (d - 1) / 2 <= 64.
constexpr int CTINY = 11;
// LDS of one wave of the main launch: L, the rows (or the tiny vertices'
// words) and the pair list.
struct alignas(16) CWave {
    int L[CMAIN];
    int deferred[W];
    unsigned long long rows[CMAIN];
    unsigned short pairs[W * (CTINY * (CTINY - 1) / 2)];
};
static_assert(W * (CTINY * (CTINY - 1) / 2) >= CMAIN * (CMAIN - 1) / 2, "pairs of one vertex fit");
// p and q of the k-th pair (q < p) in the order of the triangle, k < 2^22.
__device__ __forceinline__ void tri_pair(int k, int *p, int *q) {
    int x = (int)((1.f + __builtin_amdgcn_sqrtf(1.f + 8.f * (float)k)) * 0.5f);
    if (x * (x - 1) / 2 > k) x--;
    if ((x + 1) * x / 2 <= k) x++;
    *p = x;
    *q = k - x * (x - 1) / 2;
}

// Pairs (p, q), q in M_p, of a main-launch vertex, one per lane: rows are
// single words, row(r) gives M_r.
template <bool ACC, class F>
__device__ __forceinline__ void word_pair(const CArgs &a, F row, unsigned long long mp, unsigned long long mq, int q,
                                          unsigned long long *acc, unsigned long long &bytes) {
    const unsigned long long t = mp & mq;
    if (ACC) bytes += 8ull * ((q >> 5) + 1);
    acc[4] += __popcll(t);
    if (a.kmax < 5) return;
    unsigned c5 = 0;
    unsigned long long c6 = 0;
    for (unsigned long long br = t; br; br &= br - 1) {
        const int r = __ffsll((long long)br) - 1;
        const unsigned long long mr = t & row(r);
        if (ACC) bytes += 8ull * ((r >> 5) + 1);
        c5 += __popcll(mr);
        if (a.kmax < 6) continue;
        for (unsigned long long bs = mr; bs; bs &= bs - 1) {
            const int x = __ffsll((long long)bs) - 1;
            if (ACC) bytes += 8ull * ((x >> 5) + 1);
            c6 += __popcll(mr & row(x));
        }
    }
    acc[5] += c5;
    acc[6] += c6;
}

// The workgroup tiers' lists: every vertex of the count with d > main_max. A
// workgroup counts its slab's vertices per tier, reserves their places with
// one atomic per tier and writes them in a second pass (the main launch's
// waves did this themselves, at several atomics per chunk on one cache line:
// 1.2 of the 1.5 ms of R-MAT s20's main launch). Few, large workgroups for the
// same reason.
constexpr int kClassifyThreads = 1024;
__global__ void __launch_bounds__(kClassifyThreads) clique_classify(CArgs a) {
    __shared__ unsigned long long cnt[CTIERS + 2];
    const int per = (int)(((long long)(a.root_hi - a.root_lo) + gridDim.x - 1) / gridDim.x);
    const long long lo = a.root_lo + (long long)blockIdx.x * per;
    const long long hi = lo + per < a.root_hi ? lo + per : a.root_hi;
    auto tier_of = [&](int d) {
        return d <= a.main_max ? -1 : d <= 32 * CT0W ? 0 : d <= 32 * CT1W ? 1 : d <= a.lds_dmax ? 2 : 3;
    };
    if (threadIdx.x < CTIERS + 2) cnt[threadIdx.x] = 0;
    __syncthreads();
    for (long long v = lo + threadIdx.x; v < hi; v += kClassifyThreads) {
        const int d = a.split[v], t = tier_of(d);
        if (t >= 0) atomicAdd(&cnt[t], 1ull);
        if (d > a.cap) atomicAdd(&cnt[CTIERS], 1ull);
        if (d > a.cap && d <= 512) atomicAdd(&cnt[CTIERS + 1], 1ull);
    }
    __syncthreads();
    if (threadIdx.x < CTIERS + 2) {
        const unsigned long long c = cnt[threadIdx.x];
        if (c) cnt[threadIdx.x] = atomicAdd(&a.ovf_n[threadIdx.x], c);
        if (threadIdx.x == 3 && c && !a.grows) atomicOr(a.err, 16u);  // no HBM tier in this count
    }
    __syncthreads();
    for (long long v = lo + threadIdx.x; v < hi; v += kClassifyThreads) {
        const int t = tier_of(a.split[v]);
        if (t < 0) continue;
        const long long idx = (long long)atomicAdd(&cnt[t], 1ull);
        if (idx < a.tier_cap[t]) a.tier[t][idx] = (int)v;
        else if (a.tier_cap[t] > 0) atomicOr(a.err, 4u);
    }
}
static_assert(CTIERS == 4, "ovf_n[4] and [5] count vertices with d > cap");

// Main launch: vertices with d <= main_max; the tiers take the larger ones. The
// vertices are dealt out in chunks; chunk c of the N chunks holds the vertices
// root_lo + c + i N, so that the heavy vertices, which are neighbours in the
// degree order, spread over the chunks. A wave starts with the chunk of its
// own number and takes further ones from the queue: a grab is an atomic on
// one address, 17 ns each however many waves there are (chunks of 4 vertices
// from a counter alone held R-MAT s20's launch at 4.6 ms).
// #K6: the walk of one wave grows with the cube of d where the rows are dense
// (R-MAT s14: 1.75 ms with vertices up to 64 here, 0.60 up to 32), so a vertex
// with d > CDEFER and a quarter of the pairs adjacent goes to tier 0, its rows
// built in vain. By size alone sparse ones went too (a random graph of 200,000
// vertices and degree 60: 2.26 ms, now 1.46).
// Of a block of up to 64 vertices of a chunk, the tiny ones (d <= CTINY) are
// taken together, one position pair per lane, and keep all their rows in one
// word (row p at bit p (p - 1) / 2); the others follow one by one, with the
// next one's list read ahead.
// MODE bit 0: accumulate W_alg; bit 1: timeline records (separate
// instantiations, so that a timed count carries none of their work or
// registers).
// 128 registers (16 waves per CU where the config asks for as many; with 134, K4 on
// a random graph of 50,000 vertices and degree 40 took 262 us instead of 178).
template <int MODE>
__global__ void __launch_bounds__(256, 4) clique_kernel(CArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int wid = threadIdx.x / W, ln = threadIdx.x % W;
    CWave &C = reinterpret_cast<CWave *>(smem)[wid];
    unsigned long long acc[7] = {0, 0, 0, 0, 0, 0, 0}, bytes = 0;  // per lane
    constexpr bool ACC = MODE & 1, tl = (MODE & 2) != 0;
    const long long tl_t0 = tl ? wall_clock64() : 0;
    long long tl_build = 0, tl_count = 0, tl_items = 0, tl_pairs = 0;
    const int lim = a.main_max;
    const long long chunks = ((long long)(a.root_hi - a.root_lo) + a.chunk - 1) / a.chunk;
    const int wpb = blockDim.x / W;
    const long long waves = (long long)gridDim.x * wpb;
    long long chunk = uni64((long long)blockIdx.x * wpb + wid);
    while (chunk < chunks) {
        for (int cb = 0; cb < a.chunk; cb += W) {
            const long long v = a.root_lo + chunk + (cb + ln) * chunks;
            const bool mine = cb + ln < a.chunk && v < a.root_hi;
            const int d_l = mine ? a.split[v] : 0;
            const long long b_l = mine ? a.off[v] : 0;
            const unsigned long long tiny = ballot(d_l >= 2 && d_l <= min(lim, CTINY));
            if (tiny) {
                const long long c0 = tl ? clock64() : 0;
                const bool is = tiny >> ln & 1ull;
                C.rows[ln] = 0;
                if (ACC && is) {
                    bytes += 4ull * d_l + 16ull;
                    for (int p = 0; p < d_l; p++) bytes += 4ull * (a.split[a.adj[b_l + p]] + p) + 16ull + 4ull;
                }
                int T = 0, run = 0;
                const int myoff = excl_scan(is ? d_l * (d_l - 1) / 2 : 0, &T);
                wsync();
                constexpr int U = 4;  // steps in flight
                for (int k0 = 0; k0 < T; k0 += U * W) {
                    int x[U], y[U], s[U], pos[U];
                    unsigned word[U];
                    bool in[U];
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        const int k = k0 + u * W + ln;
                        s[u] = 0;
#pragma unroll
                        for (int step = 32; step >= 1; step >>= 1)
                            if (bperm(myoff, s[u] + step) <= k && s[u] + step < W) s[u] += step;
                        in[u] = k < T;
                        pos[u] = k - bperm(myoff, s[u]);
                        const long long rb = bperm64(b_l, s[u]);
                        x[u] = y[u] = 0;
                        if (in[u]) {
                            int p, q;
                            tri_pair(pos[u], &p, &q);
                            x[u] = a.adj[rb + p];
                            y[u] = a.adj[rb + q];
                        }
                    }
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        word[u] = 0;
                        if (in[u] && x[u] < a.core_n) word[u] = a.core[core_row(x[u]) + (y[u] >> 5)] >> (y[u] & 31);
                    }
                    bool hit[U];
                    long long base[U];
                    int n[U];
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        hit[u] = word[u] & 1u;
                        base[u] = 0;
                        n[u] = 0;
                        if (in[u] && x[u] >= a.core_n) {
                            base[u] = a.off[x[u]];
                            n[u] = a.split[x[u]];
                        }
                    }
                    search_below<U>(a, base, n, y, hit);
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        const unsigned long long m = ballot(hit[u]);
                        if (hit[u] && a.kmax >= 4) {
                            atomicOr(reinterpret_cast<unsigned *>(&C.rows[s[u]]) + (pos[u] >> 5), 1u << (pos[u] & 31));
                            C.pairs[run + mbcnt(m)] = (unsigned short)(s[u] << 6 | pos[u]);
                        }
                        run += __popcll(m);
                    }
                }
                if (ln == 0) acc[3] += (unsigned long long)run;
                wsync();
                const long long c1 = tl ? clock64() : 0;
                if (a.kmax >= 4) {
                    for (int k = ln; k < run; k += W) {
                        const int e = C.pairs[k];
                        const unsigned long long m = C.rows[e >> 6];
                        int p, q;
                        tri_pair(e & 63, &p, &q);
                        auto row = [&](int r) { return (m >> (r * (r - 1) / 2)) & ((1ull << r) - 1); };
                        word_pair<ACC>(a, row, row(p), row(q), q, acc, bytes);
                    }
                    wsync();
                }
                if (tl) {
                    tl_build += c1 - c0;
                    tl_count += clock64() - c1;
                    tl_items += __popcll(tiny);
                    tl_pairs += run;
                }
            }
            unsigned long long todo = ballot(d_l > CTINY && d_l <= lim);
            int d = 0, y = 0, vertex = 0, n_deferred = 0;
            if (todo) {
                const int l = __ffsll((long long)todo) - 1;
                d = LanePull{l}(d_l);
                vertex = LanePull{l}((int)v);
                const long long rb = LanePull{l}(b_l);
                if (ln < d) y = a.adj[rb + ln];
            }
            while (todo) {
                const long long c0 = tl ? clock64() : 0;
                todo &= todo - 1;
                int dn = 0, yn = 0, vn = 0;  // the next vertex's list
                if (todo) {
                    const int l = __ffsll((long long)todo) - 1;
                    dn = LanePull{l}(d_l);
                    vn = LanePull{l}((int)v);
                    const long long rb = LanePull{l}(b_l);
                    if (ln < dn) yn = a.adj[rb + ln];
                }
                int run = 0;
                C.L[ln] = y;
                // core vertices come first in the sorted list
                const int pc = __popcll(ballot(ln < d && y < a.core_n));
                // the others' lists, for the searches below
                const bool far = pc < d && ln < d && y >= a.core_n;
                const long long far_base = far ? a.off[y] : 0;
                const int far_n = far ? a.split[y] : 0;
                unsigned long long row_l = 0;  // row ln
                constexpr int U = 8;           // row reads in flight
                for (int p = 1; p < pc; p += U) {
                    unsigned v[U];
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        v[u] = 0;
                        const int x = LanePull{min(p + u, W - 1)}(y);
                        if (ln < p + u && p + u < pc) v[u] = a.core[core_row(x) + (y >> 5)] >> (y & 31);
                    }
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        const unsigned long long m = ballot(v[u] & 1u);
                        if (ln == p + u) row_l = m;
                        if (v[u] & 1u) C.pairs[run + mbcnt(m)] = (unsigned short)((p + u) << 8 | ln);
                        run += __popcll(m);
                    }
                }
                C.rows[ln] = row_l;
                wsync();
                // the other vertices' rows: one pair (p, q) per lane, eight searches of
                // a lane in flight where that many are left (of four at a time, K3 on a
                // random graph of 200,000 vertices and degree 60 took 1.54 ms, now 1.43)
                const int p0 = max(pc, 1), k0 = p0 * (p0 - 1) / 2, k1 = d * (d - 1) / 2;
                auto search = [&](auto flight, int kb) {  // so many searches side by side
                    constexpr int F = decltype(flight)::value;
                    int p[F], q[F], n[F], z[F];
                    long long base[F];
                    bool hit[F];
#pragma unroll
                    for (int u = 0; u < F; u++) {
                        const int k = kb + u * W + ln;
                        hit[u] = false;
                        p[u] = q[u] = 0;
                        if (k < k1) tri_pair(k, &p[u], &q[u]);
                        base[u] = bperm64(far_base, p[u]);
                        const int len = bperm(far_n, p[u]);  // by every lane
                        n[u] = k < k1 ? len : 0;
                        z[u] = C.L[q[u]];
                    }
                    search_below<F>(a, base, n, z, hit);
#pragma unroll
                    for (int u = 0; u < F; u++) {
                        const unsigned long long m = ballot(hit[u]);
                        if (hit[u]) {
                            atomicOr(reinterpret_cast<unsigned *>(&C.rows[p[u]]) + (q[u] >> 5), 1u << (q[u] & 31));
                            C.pairs[run + mbcnt(m)] = (unsigned short)(p[u] << 8 | q[u]);
                        }
                        run += __popcll(m);
                    }
                };
                int kb = k0;
                for (; kb + 4 * W < k1; kb += 8 * W) search(std::integral_constant<int, 8>{}, kb);
                if (kb < k1) search(std::integral_constant<int, 4>{}, kb);
                wsync();
                const long long c1 = tl ? clock64() : 0;
                const bool defer = a.kmax >= 6 && d > CDEFER && 8 * run > d * (d - 1);
                if (defer) {
                    if (ln == 0) C.deferred[n_deferred] = vertex;
                    n_deferred++;
                } else {
                    if (ln == 0) acc[3] += (unsigned long long)run;
                    if (ACC) {
                        if (ln == 0) bytes += 4ull * d + 16ull;
                        if (ln < d) bytes += 4ull * (a.split[y] + ln) + 16ull + 4ull * ((ln >> 5) + 1);
                    }
                }
                if (a.kmax >= 4 && !defer) {
                    auto row = [&](int p) { return C.rows[p]; };
                    for (int k = ln; k < run; k += W) {
                        const int pq = C.pairs[k];
                        word_pair<ACC>(a, row, C.rows[pq >> 8], C.rows[pq & 255], pq & 255, acc, bytes);
                    }
                }
                wsync();
                if (tl) {
                    tl_build += c1 - c0;
                    tl_count += clock64() - c1;
                    tl_items++;
                    tl_pairs += run;
                }
                d = dn;
                y = yn;
                vertex = vn;
            }
            if (n_deferred) {
                wsync();
                unsigned long long r = 0;
                if (ln == 0) r = atomicAdd(&a.ovf_n[0], (unsigned long long)n_deferred);
                const long long at = uni64((long long)__shfl(r, 0)) + ln;
                if (ln < n_deferred) {
                    if (at < a.tier_cap[0]) a.tier[0][at] = C.deferred[ln];
                    else atomicOr(a.err, 4u);
                }
                wsync();
            }
        }
        // the queue counts the chunks after the waves' own; it is read before
        // it is grabbed, so that a drained queue costs no atomic
        if (waves >= chunks) break;
        unsigned long long r = 0;
        if (ln == 0) {
            r = __atomic_load_n(&a.queue[0], __ATOMIC_RELAXED);
            if ((long long)r + waves < chunks) r = atomicAdd(&a.queue[0], 1ull);
        }
        chunk = waves + uni64((long long)__shfl(r, 0));
    }
    clique_flush<ACC>(a, acc, bytes, ln);
    if (tl && ln == 0) {
        const int unit = blockIdx.x * (blockDim.x / W) + wid;
        tl_write(a.tl, a.tl_base + unit, 0, unit, tl_t0, wall_clock64(), tl_build, tl_count, tl_items, tl_pairs);
    }
}

// Next item of a tier's queue: the vertex, or -1 when the queue is drained. A
// workgroup takes several at a time where there are many (an atomic on one
// address takes 17 ns, 1.7 ms for 100,000 vertices). next, last: its items.
__device__ __forceinline__ int tier_item(const CArgs &a, int tier, unsigned long long *next, unsigned long long *last,
                                         int *part, int *parts) {
    const unsigned long long made = a.ovf_n[tier], cap = (unsigned long long)a.tier_cap[tier];
    const unsigned long long vertices = made < cap ? made : cap;
    const int np = clique_parts(a.kmax, vertices, (int)gridDim.x);
    if (*next == *last) {
        const unsigned long long share = vertices * np / (16ull * gridDim.x), grab = share < 1 ? 1 : share < 16 ? share : 16;
        *next = atomicAdd(&a.queue[1 + tier], grab);
        *last = *next + grab;
    }
    const unsigned long long r = (*next)++;
    *part = (int)(r % np);
    *parts = np;
    return r / np < vertices ? a.tier[tier][r / np] : -1;
}

// Workgroup tiers with rows in LDS: the NW waves of a workgroup share one
// vertex of tier list TIER, d <= 32 MW. They split the rows for the build, and
// the columns of the count by their first row.
template <int MW, int TIER, int NW, int MODE>
__global__ void __launch_bounds__(64 * NW, clique_occupancy(TIER)) clique_block_kernel(CArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int wid = threadIdx.x / W, ln = threadIdx.x % W;
    constexpr int lcap = 32 * MW;
    constexpr int KC = MW / 4;            // chunks of 128 positions
    constexpr int RT = 4;  // row tiles held at once
    unsigned *rows = reinterpret_cast<unsigned *>(smem);
    int *L = reinterpret_cast<int *>(rows + tier_row_words(MW));
    unsigned *buf = reinterpret_cast<unsigned *>(L) + wid * 2 * CCOLS;
    __shared__ int vsh, psh, nsh;
    unsigned long long next = 0, last = 0;  // thread 0: items taken from the queue
    unsigned long long acc[7] = {0, 0, 0, 0, 0, 0, 0}, bytes = 0;
    constexpr bool ACC = MODE & 1, tl = (MODE & 2) != 0;
    const long long tl_t0 = tl ? wall_clock64() : 0;
    long long tl_build = 0, tl_count = 0, tl_items = 0, tl_pairs = 0, c0 = 0, c1 = 0;
    for (;;) {
        if (tl) c0 = clock64();
        if (threadIdx.x == 0) {
            int part, parts;
            vsh = tier_item(a, TIER, &next, &last, &part, &parts);
            psh = part;
            nsh = parts;
        }
        __syncthreads();
        const int v0 = vsh, part = psh, parts = nsh;
        if (v0 < 0) break;
        const int d = a.split[v0];
        const long long rb = a.off[v0];
        const int w = row_words(d);
        const bool fits = d <= lcap;  // always: lists are split by d
        if (!fits && threadIdx.x == 0) atomicOr(a.err, 8u);
        if (fits)
            for (int k = threadIdx.x; k < d; k += 64 * NW) L[k] = a.adj[rb + k];
        __syncthreads();
        bool any = false;
        if (fits) {
            unsigned long long bb = 0;  // every part builds the rows; W_alg and #K3 charge one build
            const unsigned long long pr = vtx_rows<ACC>(a, (const int *)L, d, rows, w, wid, NW, ln, bb);
            if (part == 0) {
                if (ln == 0) acc[3] += pr;
                if (ACC) bytes += bb + (threadIdx.x == 0 ? 4ull * d + 16ull : 0ull);
                tl_pairs += (long long)pr;
            }
            any = pr != 0;
        }
        any = __syncthreads_or(any);  // the rows are complete, and L is free for the column lists
        if (tl) c1 = clock64();
        if (any && a.kmax >= 4) {
            const int first = part * NW + wid, stride = NW * parts;
            unsigned long long none = 0;
            if (a.kmax == 4)
                count_columns<KC, RT, 1, ACC>(rows, w, d, buf, first, stride, ln, acc[4], none, none, bytes);
            else if (a.kmax == 5)
                count_columns<KC, RT, 2, ACC>(rows, w, d, buf, first, stride, ln, acc[5], acc[4], none, bytes);
            else
                count_columns<KC, RT, 3, ACC>(rows, w, d, buf, first, stride, ln, acc[6], acc[5], acc[4], bytes);
        }
        __syncthreads();
        if (tl) {
            tl_build += c1 - c0;
            tl_count += clock64() - c1;
            tl_items++;
        }
    }
    clique_flush<ACC>(a, acc, bytes, ln);
    if (tl && threadIdx.x == 0)
        tl_write(a.tl, a.tl_base + blockIdx.x, 1 + TIER, blockIdx.x, tl_t0, wall_clock64(), tl_build, tl_count,
                 tl_items, tl_pairs);
}

// Workgroup tier 3: vertices whose rows do not fit LDS. Rows and pair
// offsets sit in the workgroup's HBM scratch; the waves split the rows for
// the build and take pairs round-robin for the count.
template <int MODE>
__global__ void __launch_bounds__(64 * CNW3) clique_hbm_kernel(CArgs a) {
    constexpr int TIER = 3, NW = CNW3;
    const int wid = threadIdx.x / W, ln = threadIdx.x % W;
    __shared__ int vsh, psh, nsh;
    unsigned long long next = 0, last = 0;  // thread 0: items taken from the queue
    __shared__ int wtot[NW];
    unsigned *rows = a.grows + (long long)blockIdx.x * a.hcap * row_words(a.hcap);
    int *off = a.goff + (long long)blockIdx.x * (a.hcap + 1);
    unsigned long long acc[7] = {0, 0, 0, 0, 0, 0, 0}, bytes = 0;
    constexpr bool ACC = MODE & 1, tl = (MODE & 2) != 0;
    const long long tl_t0 = tl ? wall_clock64() : 0;
    long long tl_build = 0, tl_count = 0, tl_items = 0, tl_pairs = 0, c0 = 0, c1 = 0;
    for (;;) {
        if (tl) c0 = clock64();
        if (threadIdx.x == 0) {
            int part, parts;
            vsh = tier_item(a, TIER, &next, &last, &part, &parts);
            psh = part;
            nsh = parts;
        }
        __syncthreads();
        const int v0 = vsh, part = psh, parts = nsh;
        if (v0 < 0) break;
        const int d = a.split[v0];
        const int w = row_words(d);
        const bool fits = d <= a.hcap;  // always: hcap is the maximum out-degree
        if (!fits && threadIdx.x == 0) atomicOr(a.err, 8u);
        unsigned long long bb = 0;
        if (fits) (void)vtx_rows<ACC>(a, a.adj + a.off[v0], d, rows, w, wid, NW, ln, bb);
        if (ACC && fits && part == 0) bytes += bb + (threadIdx.x == 0 ? 4ull * d + 16ull : 0ull);
        __threadfence();
        __syncthreads();
        // pair offsets: block-wide exclusive prefix of popc(M_p)
        int run = 0;
        for (int pb = 0; fits && pb < d; pb += 64 * NW) {
            const int p = pb + (int)threadIdx.x;
            int c = 0;
            if (p < d)
                for (int u = 0; u <= (p >> 5); u++) c += __popc(rows[(long long)p * w + u]);
            int tot = 0;
            const int x = excl_scan(c, &tot);
            if (ln == 0) wtot[wid] = tot;
            __syncthreads();
            int pre = 0, all = 0;
            for (int k = 0; k < NW; k++) {
                const int t = wtot[k];
                if (k < wid) pre += t;
                all += t;
            }
            if (p < d) off[p] = run + pre + x;
            run += all;
            __syncthreads();
        }
        if (fits && threadIdx.x == 0) {
            off[d] = run;
            if (part == 0) acc[3] += (unsigned long long)run;
        }
        __threadfence();
        __syncthreads();
        if (tl) c1 = clock64();
        if (fits && a.kmax >= 4)
            vtx_pairs<ACC>(a, rows, d, w, off, run, part * 64 * NW + (int)threadIdx.x, 64 * NW * parts, acc, bytes);
        __syncthreads();
        if (tl) {
            tl_build += c1 - c0;
            tl_count += clock64() - c1;
            tl_items++;
            tl_pairs += run;
        }
    }
    clique_flush<ACC>(a, acc, bytes, ln);
    if (tl && threadIdx.x == 0)
        tl_write(a.tl, a.tl_base + blockIdx.x, 1 + TIER, blockIdx.x, tl_t0, wall_clock64(), tl_build, tl_count,
                 tl_items, tl_pairs);
}

// Core bitmap rows of the vertices [0, core_n): a wave builds a row in its
// LDS slice (core_n <= CCORE bits) and writes it out whole.
constexpr int CCORE = 1 << 16;
__global__ void __launch_bounds__(256) core_rows_kernel(const long long *off, const int *adj, const int *split,
                                                        int core_n, unsigned *core) {
    __shared__ unsigned buf[4][CCORE / 32];
    const int wid = threadIdx.x / W, ln = threadIdx.x % W;
    unsigned *b = buf[wid];
    for (int x = blockIdx.x * 4 + wid; x < core_n; x += gridDim.x * 4) {
        const int words = (x + 31) >> 5, len = split[x];
        const long long xb = off[x];
        for (int k = ln; k < words; k += W) b[k] = 0u;
        wsync();
        for (int k = ln; k < len; k += W) {
            const int y = adj[xb + k];
            atomicOr(&b[y >> 5], 1u << (y & 31));
        }
        wsync();
        unsigned *row = core + core_row(x);
        for (int k = ln; k < words; k += W) row[k] = b[k];
        wsync();
    }
}

__global__ void fill_u64(unsigned long long *p, long long n, unsigned long long v) {
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        p[i] = v;
}

__global__ void split_kernel(const long long *off, const int *adj, int n, int *split) {
    for (long long v = blockIdx.x * (long long)blockDim.x + threadIdx.x; v < n; v += (long long)gridDim.x * blockDim.x)
        split[v] = lbound(adj + off[v], (int)(off[v + 1] - off[v]), (int)v);
}

// Bitmap row h of hub vertex hub_vertex[h] (or h when hub_vertex is null);
// rows start zeroed.
__global__ void hub_rows_kernel(const long long *off, const int *adj, const int *hub_vertex, int n_hubs,
                                unsigned *bits, long long words) {
    for (int h = blockIdx.x; h < n_hubs; h += gridDim.x) {
        const int v = hub_vertex ? hub_vertex[h] : h;
        unsigned *row = bits + (long long)h * words;
        for (long long k = off[v] + threadIdx.x; k < off[v + 1]; k += blockDim.x) {
            const int x = adj[k];
            atomicOr(&row[x >> 5], 1u << (x & 31));
        }
    }
}

__global__ void copy_kernel(const int4 *__restrict__ src, int4 *__restrict__ dst, long long n) {
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

}  // namespace gatk

// ===========================================================================
// Host side
// ===========================================================================
namespace gat {

// (The runtime keeps an error until it is asked for: read here, it does not
// turn up in the next count's check of its launches.)
#define HIPCHECK(x)                                                                                  \
    do {                                                                                             \
        hipError_t e_ = (x);                                                                         \
        if (e_ != hipSuccess) {                                                                      \
            (void)hipGetLastError();                                                                 \
            GAT_FAIL(GAT_ENODEV, "%s failed: %s", #x, hipGetErrorString(e_));                        \
        }                                                                                            \
    } while (0)

struct DeviceInfo {
    bool ok = false;
    int cus = 0;
    size_t lds_per_block = 0;
    size_t lds_per_cu = 0;
    long long wall_khz = 0;  // wall_clock64() ticks per millisecond
    char arch[64] = {};
};

static int device_info(DeviceInfo *out) {
    static DeviceInfo info;
    static std::once_flag once;
    static int rc = GAT_OK;
    std::call_once(once, [] {
        int n = 0;
        if (hipGetDeviceCount(&n) != hipSuccess || n == 0) {
            set_error("no HIP device visible");
            rc = GAT_ENODEV;
            return;
        }
        hipDeviceProp_t p;
        if (hipGetDeviceProperties(&p, 0) != hipSuccess) {
            set_error("hipGetDeviceProperties failed");
            rc = GAT_ENODEV;
            return;
        }
        info.cus = p.multiProcessorCount;
        info.lds_per_block = p.sharedMemPerBlock;
        info.lds_per_cu = p.maxSharedMemoryPerMultiProcessor ? p.maxSharedMemoryPerMultiProcessor : p.sharedMemPerBlock;
        int khz = 0;
        if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, 0) != hipSuccess || khz <= 0) khz = 100000;
        info.wall_khz = khz;
        std::snprintf(info.arch, sizeof(info.arch), "%s", p.gcnArchName);
        if (std::strncmp(p.gcnArchName, "gfx950", 6) != 0) {
            set_error("libgat is built for gfx950; device is %s", p.gcnArchName);
            rc = GAT_ENODEV;
            return;
        }
        info.ok = true;
    });
    if (rc) {
        set_error("no usable gfx950 device");
        return rc;
    }
    *out = info;
    return GAT_OK;
}

// Bitmap rows of the n most connected vertices of a graph, in the order of
// degree (descending, then id). A count that needs fewer uses the first of
// them, so plans of different thresholds share one set. It is shared: whoever
// replaces it leaves it to the counts that were prepared with it.
struct HubRows {
    size_t n = 0;
    unsigned *bits = nullptr;
    int *map = nullptr;  // null when the graph is degree-ordered
    int *vertex = nullptr;
    ~HubRows() {
        for (void *p : {(void *)bits, (void *)map, (void *)vertex})
            if (p) (void)hipFree(p);
    }
};

// Core bitmap of the clique store: the rows of the vertices [0, n), shared like
// the hub rows.
struct CoreRows {
    int n = 0;
    unsigned *bits = nullptr;
    ~CoreRows() {
        if (bits) (void)hipFree(bits);
    }
};

// Memory that makes counts faster and that they can do without (bitmaps of a
// graph, tables of kept counts of a plan) stays with the graph or plan. What
// holds some of it is listed here: an allocation that a count cannot do without
// and that finds no memory takes it from those that no count is using (need_malloc).
struct PlanDevice;
struct DeviceGraph;
struct Holders {
    std::mutex mu;
    std::set<PlanDevice *> plans;
    std::set<DeviceGraph *> graphs;
};
static Holders &holders() {
    static Holders *h = new Holders;  // plans may be freed after this file's statics
    return *h;
}
// After an optional allocation found no memory, the next kRetry counts do not
// ask for it again.
constexpr int kRetry = 64;

struct DeviceGraph {
    long long *off = nullptr;
    int *adj = nullptr;
    int *split = nullptr;
    std::mutex mu;  // guards what follows; held while the bitmaps are built
    std::shared_ptr<CoreRows> core;
    std::shared_ptr<HubRows> hubs;
    std::vector<int> at_least;  // degree_stats: at_least[d]: vertices of degree >= d, d <= max_deg + 1
    bool ordered = false;       // ids by descending degree
    double neighbour_degree = 0;  // mean degree of a neighbour: sum of d^2 over sum of d
    int hubs_wait = 0;          // counts until the optional rows are asked for again
    DeviceGraph() {
        std::lock_guard<std::mutex> lk(holders().mu);
        holders().graphs.insert(this);
    }
    ~DeviceGraph() {
        {
            std::lock_guard<std::mutex> lk(holders().mu);
            holders().graphs.erase(this);
        }
        if (off) (void)hipFree(off);
        if (adj) (void)hipFree(adj);
        if (split) (void)hipFree(split);
    }
};

struct PlanDevice {
    std::mutex busy;  // held by a count from its preparation to its end
    hipStream_t stream = nullptr;
    GatPlanDev pd;                          // the plan as it runs on its graph (choose_kept)
    GatPlanDev *plan = nullptr;             // a copy on the device
    unsigned long long *ctl = nullptr;      // control words (kCtl*)
    unsigned long long *result = nullptr;   // the first kCtlResult of them in pinned host memory
    long long *ovf = nullptr;
    gatk::SplitTask *subs = nullptr;  // split subtasks (array store)
    gatk::KArgsSet *dargs = nullptr;  // arguments of the array-store launches of a count
    long long *tl = nullptr;          // timeline records of the last GAT_FLAG_TIMELINE count
    int tl_n = 0;                     // records that count reserved (0: none)
    int *tier[gatk::CTIERS] = {};  // clique vertices of the workgroup tiers
    long long ovf_cap = 0;
    int *gstore = nullptr;
    size_t gstore_bytes = 0;
    // kept COUNT values (array store)
    gatk::KeptEdge *edge_tab[4] = {};
    gatk::KeptEntry *pool = nullptr;
    long long pool_entries = 0;
    unsigned pool_tables = 0, epoch = 0;
    int tab_size = 0;
    bool keep = false;
    int tables_wait = 0;  // counts until tables are asked for again
    int ovf_grid = 0;
    hipEvent_t ev[5] = {};  // start, after the main launch, end, after the second launches, start of the main launch
    bool cleared = false;   // the last count cleared tables between its start and its main launch
    // clique HBM-tier rows and pair offsets
    unsigned *grows = nullptr;
    int *goff = nullptr;
    int big_groups = 0, big_cap = 0;
    std::shared_ptr<DeviceGraph> dg;
    // captured graph
    hipGraphExec_t gexec = nullptr;
    hipGraph_t graph = nullptr;
    PlanDevice() {
        std::lock_guard<std::mutex> lk(holders().mu);
        holders().plans.insert(this);
    }
    // Frees the tables of kept counts; true if there were any.
    bool drop_tables() {
        bool any = false;
        for (auto &t : edge_tab)
            if (t) {
                (void)hipFree(t);
                t = nullptr;
                any = true;
            }
        if (pool) {
            (void)hipFree(pool);
            pool = nullptr;
            any = true;
        }
        keep = false;
        return any;
    }
};

void destroy_plan_device(PlanDevice *d) {
    if (!d) return;
    {
        std::lock_guard<std::mutex> lk(holders().mu);
        holders().plans.erase(d);
    }
    d->drop_tables();
    if (d->gexec) (void)hipGraphExecDestroy(d->gexec);
    if (d->graph) (void)hipGraphDestroy(d->graph);
    for (auto &e : d->ev)
        if (e) (void)hipEventDestroy(e);
    for (void *p : {(void *)d->plan, (void *)d->dargs, (void *)d->tl, (void *)d->ctl, (void *)d->ovf, (void *)d->subs,
                    (void *)d->tier[0], (void *)d->tier[1], (void *)d->tier[2], (void *)d->tier[3],
                    (void *)d->gstore, (void *)d->grows, (void *)d->goff})
        if (p) (void)hipFree(p);
    if (d->result) (void)hipHostFree(d->result);
    if (d->stream) (void)hipStreamDestroy(d->stream);
    delete d;
}

// Memory that a count can do without: false, and *p null, if there is none left.
template <class T>
static bool try_malloc(T **p, size_t bytes, int *rc) {
    *p = nullptr;
    const hipError_t e = hipMalloc((void **)p, bytes);
    if (e == hipSuccess) return true;
    *p = nullptr;
    (void)hipGetLastError();
    if (e != hipErrorOutOfMemory) {
        gat::set_error("hipMalloc failed: %s", hipGetErrorString(e));
        *rc = GAT_ENODEV;
    }
    return false;
}

// Frees what idle plans and graphs can do without; true if that was anything.
// mine, if given, is a plan whose lock the caller holds (prepared: its tables
// are in the arguments of a count already), and locked a graph whose lock it holds.
static bool give_back(PlanDevice *mine, bool prepared, const DeviceGraph *locked) {
    Holders &h = holders();
    std::lock_guard<std::mutex> lk(h.mu);
    bool any = mine && !prepared && mine->drop_tables();
    for (PlanDevice *d : h.plans) {
        if (d == mine || !d->busy.try_lock()) continue;
        any |= d->drop_tables();
        d->busy.unlock();
    }
    for (DeviceGraph *g : h.graphs) {
        if (g == locked || !g->mu.try_lock()) continue;
        // a count holds its graph's bitmaps and takes them under the graph's lock
        if (g->hubs && g->hubs.use_count() == 1) {
            g->hubs.reset();
            any = true;
        }
        if (g->core && g->core.use_count() == 1) {
            g->core.reset();
            any = true;
        }
        g->mu.unlock();
    }
    return any;
}

bool give_back_memory() { return give_back(nullptr, false, nullptr); }

// Memory that a count cannot do without (mine, prepared, locked: see give_back).
template <class T>
static int need_malloc(T **p, size_t bytes, PlanDevice *mine, const DeviceGraph *locked = nullptr, bool prepared = false) {
    int rc = GAT_OK;
    if (try_malloc(p, bytes, &rc)) return GAT_OK;
    if (rc) return rc;
    if (give_back(mine, prepared, locked) && try_malloc(p, bytes, &rc)) return GAT_OK;
    if (!rc) GAT_FAIL(GAT_ENODEV, "hipMalloc of %zu bytes failed: %s", bytes, hipGetErrorString(hipErrorOutOfMemory));
    return rc;
}

static int ensure_device_graph(Graph &g, std::shared_ptr<DeviceGraph> *out) {
    std::lock_guard<std::mutex> lk(*g.dev_mu);
    if (g.dev) {
        *out = std::static_pointer_cast<DeviceGraph>(g.dev);
        return GAT_OK;
    }
    auto dg = std::make_shared<DeviceGraph>();
    int rc = need_malloc(&dg->off, sizeof(long long) * (size_t(g.n) + 1), nullptr);
    if (!rc) rc = need_malloc(&dg->adj, sizeof(int) * std::max<size_t>(1, size_t(g.m)), nullptr);
    if (!rc) rc = need_malloc(&dg->split, sizeof(int) * std::max<size_t>(1, size_t(g.n)), nullptr);
    if (rc) return rc;
    HIPCHECK(hipMemcpy(dg->off, g.off.data(), sizeof(long long) * (size_t(g.n) + 1), hipMemcpyHostToDevice));
    if (g.m) HIPCHECK(hipMemcpy(dg->adj, g.adj.data(), sizeof(int) * size_t(g.m), hipMemcpyHostToDevice));
    if (g.n) {
        hipLaunchKernelGGL(gatk::split_kernel, dim3(1024), dim3(256), 0, nullptr, dg->off, dg->adj, g.n, dg->split);
        HIPCHECK(hipGetLastError());
    }
    HIPCHECK(hipDeviceSynchronize());
    g.dev = dg;
    *out = dg;
    return GAT_OK;
}

// The largest number of neighbours below a vertex.
static int32_t max_out_degree(Graph &g) {
    std::lock_guard<std::mutex> lk(*g.dev_mu);
    if (g.max_out < 0) {
        int32_t mo = 0;
        for (int32_t v = 0; v < g.n; v++) {
            const int32_t *b = g.adj.data() + g.off[v], *en = g.adj.data() + g.off[v + 1];
            mo = std::max(mo, int32_t(std::lower_bound(b, en, v) - b));
        }
        g.max_out = mo;
    }
    return g.max_out;
}

// Neighbourhood bitmaps, most connected vertices first, within kHubBytes: of
// every vertex of degree >= the configured threshold, or by default of those of
// degree >= kHubDegree and, within kHubMoreBytes, of further ones down to
// hub_default(n). One word of a bitmap replaces a search of about log2(degree)
// dependent reads, but in many sparse rows every word is a cache line of its
// own. ms with a threshold of 256 / 64 / 16: house on Chung-Lu 65,536 18.6 /
// 16.7 / 16.8, C5 on R-MAT s13 18.1 / 15.2 / 15.0, 21 patterns on R-MAT s10
// 10.3 / 8.3 / 6.9, C4 + P4 on a random graph of 100,000 vertices and mean
// degree 16 3.9 / 3.9 / 5.7. Built outside the timed count, like the graph
// upload itself, when a graph's first count needs them or a later one needs more.
constexpr double kHubBytes = 8.0 * (1ull << 30), kHubMoreBytes = 1.0 * (1ull << 30);
constexpr int kHubDegree = 256;
static int hub_default(int64_t n) { return n <= 16384 ? 16 : 64; }

// Counts of the array store need the graph's degrees; dg->mu is held.
static void degree_stats(const Graph &g, DeviceGraph *dg) {
    if (!dg->at_least.empty()) return;
    std::vector<int> c((size_t)g.max_deg + 2, 0);
    bool ordered = true;
    for (int32_t v = 0; v < g.n; v++) {
        c[g.deg(v)]++;
        ordered = ordered && (v == 0 || g.deg(v) <= g.deg(v - 1));
    }
    double squares = 0;
    for (size_t d = 0; d < c.size(); d++) squares += (double)c[d] * d * d;
    for (size_t d = c.size() - 1; d-- > 0;) c[d] += c[d + 1];
    dg->ordered = ordered;
    dg->neighbour_degree = g.m ? squares / (double)g.m : 0;
    dg->at_least = std::move(c);
}

// What a count uses of them: the first n rows. full: every vertex from this
// degree on has one.
struct HubUse {
    std::shared_ptr<HubRows> rows;
    int n = 0, full = INT_MAX;
};

// optional: *out stays empty where there is no memory for the rows.
static int build_hubs(const Graph &g, DeviceGraph *dg, size_t n, int least, bool optional, PlanDevice *mine,
                      std::shared_ptr<HubRows> *out) {
    const long long words = ((long long)g.n + 31) / 32, n_u64 = ((long long)n * words + 1) / 2;
    auto h = std::make_shared<HubRows>();
    h->n = n;
    int rc = GAT_OK;
    if (optional) try_malloc(&h->bits, 8 * (size_t)n_u64, &rc);
    else rc = need_malloc(&h->bits, 8 * (size_t)n_u64, mine, dg);
    if (rc || !h->bits) return rc;
    hipLaunchKernelGGL(gatk::fill_u64, dim3(2048), dim3(256), 0, nullptr, (unsigned long long *)h->bits, n_u64, 0ull);
    if (!dg->ordered) {
        std::vector<int32_t> hubs, map(size_t(g.n), -1);
        for (int32_t v = 0; v < g.n; v++)
            if (g.deg(v) >= least) hubs.push_back(v);
        std::stable_sort(hubs.begin(), hubs.end(), [&](int32_t x, int32_t y) { return g.deg(x) > g.deg(y); });
        hubs.resize(n);
        for (size_t k = 0; k < n; k++) map[hubs[k]] = int32_t(k);
        rc = need_malloc(&h->map, sizeof(int) * size_t(g.n), mine, dg);
        if (!rc) rc = need_malloc(&h->vertex, sizeof(int) * n, mine, dg);
        if (rc) return rc;
        HIPCHECK(hipMemcpy(h->map, map.data(), sizeof(int) * size_t(g.n), hipMemcpyHostToDevice));
        HIPCHECK(hipMemcpy(h->vertex, hubs.data(), sizeof(int) * n, hipMemcpyHostToDevice));
    }
    hipLaunchKernelGGL(gatk::hub_rows_kernel, dim3((unsigned)std::min<size_t>(n, 65535)), dim3(256), 0, nullptr, dg->off,
                       dg->adj, h->vertex, (int)n, h->bits, words);
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipDeviceSynchronize());
    *out = h;
    return GAT_OK;
}

// thr: the configured threshold, 0 for the default. The graph's rows serve if
// there are enough of them; else they are built anew, and on a failure the
// graph is left without any, for the next count to build.
static int ensure_hubs(const Graph &g, DeviceGraph *dg, int thr, PlanDevice *mine, HubUse *out) {
    std::lock_guard<std::mutex> lk(dg->mu);
    degree_stats(g, dg);
    const std::vector<int> &at_least = dg->at_least;
    auto vertices = [&](int degree) -> size_t { return degree < (int)at_least.size() ? at_least[degree] : 0; };
    const int least = thr ? thr : hub_default(g.n);
    const double row_bytes = 4.0 * (double)std::max(1ll, ((long long)g.n + 31) / 32);
    const size_t found = vertices(least), most = (size_t)(kHubBytes / row_bytes);
    // rows that only kHubBytes limits
    const size_t always = std::min(thr ? found : vertices(std::max(least, kHubDegree)), most);
    size_t n = std::min({found, std::max(always, (size_t)(kHubMoreBytes / row_bytes)), most});
    auto missing = [&] { return n > (dg->hubs ? dg->hubs->n : 0); };
    if (missing() && n > always) {  // the rows beyond kHubDegree only where there is room
        if (dg->hubs_wait > 0) {
            dg->hubs_wait--;
        } else {
            std::shared_ptr<HubRows> rows;
            const int rc = build_hubs(g, dg, n, least, true, mine, &rows);
            if (rc) return rc;
            if (rows) dg->hubs = rows; else dg->hubs_wait = kRetry;
        }
        if (missing()) n = always;
    }
    if (missing()) {
        dg->hubs.reset();
        const int rc = build_hubs(g, dg, n, least, false, mine, &dg->hubs);
        if (rc) return rc;
    }
    out->rows = dg->hubs;
    out->n = (int)n;
    // one more than the degree of the last row's vertex, if some are left without
    out->full = n == found ? least
                : n == 0   ? INT_MAX
                           : (int)(std::partition_point(at_least.begin(), at_least.end(),
                                                        [&](int c) { return (size_t)c >= n; }) -
                                   at_least.begin());
    return GAT_OK;
}

// Core bitmap of the clique store: the rows of the first core vertices, at
// most gatk::CCORE of them and within `words` words (about four times the
// CSR: on R-MAT s20 the 65,536 core vertices hold 86-100 % of the positions,
// 268 MB against 126 MB of lists).
static int core_vertices(int64_t n, long long words) {
    int lo = 0, hi = (int)std::min<int64_t>(n, gatk::CCORE);  // the largest x with core_row(x) <= words
    while (lo < hi) {
        const int mid = lo + (hi - lo + 1) / 2;
        if ((long long)gatk::core_row(mid) <= words) lo = mid; else hi = mid - 1;
    }
    return lo;
}

static int ensure_core(const Graph &g, DeviceGraph *dg, std::shared_ptr<CoreRows> *out) {
    std::lock_guard<std::mutex> lk(dg->mu);
    if (dg->core) {
        *out = dg->core;
        return GAT_OK;
    }
    auto c = std::make_shared<CoreRows>();
    int rc = GAT_OK;
    // fewer core vertices where memory is short, down to none
    for (long long budget = std::max<long long>(1 << 21, 4ll * g.m);; budget = std::max<long long>(1 << 21, budget / 4)) {
        c->n = core_vertices(g.n, budget);
        if (try_malloc(&c->bits, sizeof(unsigned) * std::max<size_t>(gatk::core_row(c->n), 16), &rc)) break;
        if (rc) return rc;
        if (budget <= 1 << 21) {
            c->n = 0;
            break;
        }
    }
    if (c->n > 0) {
        hipLaunchKernelGGL(gatk::core_rows_kernel, dim3(std::min((c->n + 3) / 4, 4096)), dim3(256), 0, nullptr, dg->off,
                           dg->adj, dg->split, c->n, c->bits);
        HIPCHECK(hipGetLastError());
        HIPCHECK(hipDeviceSynchronize());
    }
    dg->core = c;
    *out = c;
    return GAT_OK;
}

// Split subtasks: capacity of each level's list, and the default time a
// task runs in the tail of a launch before it hands on its unfinished loops.
// Subtask counters live at ovf_n[8 + k] (k = 1 .. levels: LDS levels, then
// the HBM list).
constexpr long long kSubCap = 1ll << 20;
constexpr int kLevels = gatk::kSplitLevels;
constexpr int kSplitUs = 2000;
// Control words of a count, one allocation: first what the host reads back (the
// copies of the counts, 16 list sizes, 4 W_alg sums, the error flags), then the
// clique store's queues, and for the array store the queue heads and drained
// flags. One launch clears them and one copy into pinned memory reads them: five
// fills and four copies were 50 us of a small count.
constexpr int kCtlOvf = GATP_MAX_TERMS * gatk::kCountCopies, kCtlBytes = kCtlOvf + 16, kCtlErr = kCtlBytes + 4;
constexpr int kCtlResult = kCtlErr + 1, kCtlQueue = (kCtlResult + 15) / 16 * 16, kCtlHeads = kCtlQueue + 16;
constexpr int kCtlDrained = kCtlHeads + gatk::kQueueWords, kCtlWords = kCtlDrained + gatk::kQueues;
static_assert(kCtlQueue % 16 == 0 && kCtlHeads % 16 == 0, "queue heads on cache lines of their own");
// timeline capacity (records of gatk::kTlFields int64 each)
constexpr int kTlCap = 1 << 15;

constexpr int64_t kTasksPerWave = 8;

struct Launch {
    gatk::KArgs a;
    dim3 grid, block;
    size_t lds = 0;
    int wave_bytes = 0;
    dim3 ovf_grid;
    size_t ovf_lds = 0;
    int ovf_wave_bytes = 0;
    gatk::KArgs ao;
    bool clique = false;  // bitmap clique path
    gatk::CArgs ca;
    size_t clique_lds = 0;
    dim3 tier_grid[gatk::CTIERS];  // workgroup tiers; x = 0: no vertex can reach the tier
    size_t tier_lds[gatk::CTIERS] = {};
    long long tasks = 0;  // root edges of the count
    int chunk = 1;        // queue_chunk
    int64_t waves = 1;    // waves of the main launch
    bool edge_grain = false;  // the HBM launch takes single edges
    bool may_overflow = true; // some intersection may outgrow its LDS buffer
    bool pair = false;        // the plan has nodes swept with their leaf (GatNode::pair)
    std::unique_lock<std::mutex> busy;  // of the plan
    HubUse hubs;                        // kept, like the core rows, for as long as the count may read them
    std::shared_ptr<CoreRows> core;
    bool heavy = false;   // clique: some vertex may have more than main_max neighbours below it
};

// Vertices per chunk of the clique main launch: a wave's whole share, or half to
// a quarter of it, and no fewer than configured, where shares are long for the
// number of waves. Chunks mix heavy and light vertices, so that whole shares
// balance well; every further chunk is a grab, an atomic on one address (17 ns
// each, one after another), and should cost a few per cent of the vertices it
// hands out. us with chunks of a quarter share / of this rule: K3 on Chung-Lu
// 130,000 of degree 12 364 / 102, K4 on random graphs of degree 40 (50,000
// vertices) 357 / 271, 24 (200,000) 649 / 437 and 8 (1 M) 460 / 207, K3-K5 on
// Chung-Lu 262,144 of degree 24 845 / 772.
static int clique_chunk(int configured, long long vertices, long long waves) {
    const long long share = std::max(1ll, (vertices + waves - 1) / waves);
    const long long chunks = std::max(1ll, std::min({4ll, share / std::max(1, configured), 1 + 6 * share / waves}));
    return (int)((share + chunks - 1) / chunks);
}

// Restrict a prepared count to the root vertices [lo, hi): the array store
// takes the directed edges of those vertices, the bitmap store those top
// vertices.
static void set_edges(Launch *L, int64_t lo, int64_t hi) {
    L->a.e_lo = L->ao.e_lo = lo;
    L->a.e_hi = L->ao.e_hi = hi;
    L->tasks = hi - lo;
    // edges per task: as configured, but at least kTasksPerWave tasks per wave
    // (few edges: R-MAT s10 with 16 edges per task left two thirds of the waves
    // without one)
    L->a.chunk = (int)std::max<int64_t>(1, std::min<int64_t>(L->chunk, (hi - lo) / (kTasksPerWave * L->waves)));
    L->ao.chunk = L->edge_grain ? 1 : L->a.chunk;
}
static void set_roots(Launch *L, const Graph &g, int32_t lo, int32_t hi) {
    set_edges(L, g.off[lo], g.off[hi]);
    L->ca.root_lo = lo;
    L->ca.root_hi = hi;
    if (!L->clique) return;
    L->ca.chunk = clique_chunk(L->chunk, hi - lo, (long long)L->grid.x * (L->block.x / 64));
}

static void fill_defaults(gat_kernel_config *c) {
    if (c->block_waves <= 0) c->block_waves = 1;
    if (c->waves_per_cu <= 0) c->waves_per_cu = 8;
    if (c->queue_chunk <= 0) c->queue_chunk = 16;
    if (c->slot_capacity <= 0) c->slot_capacity = 1024;
    if (c->intersect_strategy < 0 || c->intersect_strategy > 4) c->intersect_strategy = 0;
    if (c->gallop_ratio <= 0) c->gallop_ratio = 32;
    if (c->search_linear_threshold < 0) c->search_linear_threshold = 0;
    if (c->split_us == 0) c->split_us = kSplitUs;
}

// Knobs and launch shapes of the clique store: the main launch (one wave
// per vertex) and the workgroup tiers with rows in LDS. max_out: an upper
// bound of the out-degrees; tiers beyond it are not launched.
static int clique_shape(const DeviceInfo &di, const gat_kernel_config &cfg, int max_out, Launch *L) {
    gatk::CArgs &c = L->ca;
    c.cap = std::max(32, std::min(gatk::CMAXD, cfg.slot_capacity / 32 * 32));
    L->chunk = cfg.queue_chunk;
    L->block = dim3(64 * cfg.block_waves);
    L->grid = dim3(std::max(1, std::max(1, cfg.waves_per_cu * di.cus) / cfg.block_waves));
    L->clique_lds = sizeof(gatk::CWave) * cfg.block_waves;
    const size_t lds[3] = {gatk::tier_lds(gatk::CT0W, gatk::CNW0), gatk::tier_lds(gatk::CT1W, gatk::CNW1),
                           gatk::tier_lds(gatk::CT2W, gatk::CNW2)};
    if (lds[1] + 64 > di.lds_per_block) GAT_FAIL(GAT_EINFEASIBLE, "device LDS too small for the clique block tiers");
    // 64 B: the kernels' own static LDS
    c.lds_dmax = lds[2] + 64 <= di.lds_per_block ? 32 * gatk::CT2W : 32 * gatk::CT1W;
    const int waves[3] = {gatk::CNW0, gatk::CNW1, gatk::CNW2};
    // (#K3 to #K5 lose up to 10 % below 64)
    c.main_max = std::min(gatk::CMAIN, c.cap);
    const int above[4] = {c.kmax >= 6 ? std::min(gatk::CDEFER, c.main_max) : c.main_max, 32 * gatk::CT0W, 32 * gatk::CT1W,
                          c.lds_dmax};
    for (int t = 0; t < 3; t++) {
        L->tier_lds[t] = lds[t];
        const int per_cu = std::max(1, std::min((int)(di.lds_per_cu / (lds[t] + 64)), 4 * gatk::clique_occupancy(t) / waves[t]));
        L->tier_grid[t] = dim3(max_out > above[t] && above[t] < c.lds_dmax ? per_cu * di.cus : 0);
    }
    L->tier_grid[3] = dim3(max_out > above[3] ? 2 * di.cus : 0);
    L->heavy = max_out > c.main_max;
    return GAT_OK;
}

// Tables of kept COUNT values (GATP_KEEP_*): an int per directed edge and
// truncation, cleared by every count, and the pools. A pool's table covers the
// first kTabVertices vertices (of a degree-ordered graph the most visited
// ones); there are as many tables as kPoolBytes for all pools holds, or where
// memory is short a quarter, a sixteenth or a 64th of that. Values have 24 bits
// and keys 32: larger graphs go without.
constexpr long long kPoolBytes = 1ll << 29, kPoolLeast = 1ll << 23;
constexpr int kTabVertices = 1 << 14;
static int ensure_tables(gat_plan *p) {
    PlanDevice *d = p->dev;
    const GatPlanDev &pd = d->pd;
    const Graph &g = *p->graph;
    if (d->keep || !(pd.edge_tables || pd.n_tables)) return GAT_OK;
    if (g.m == 0 || g.max_deg >= 1 << 24 || g.m >= (1ll << 32) - 1) return GAT_OK;
    if (d->tables_wait > 0) {
        d->tables_wait--;
        return GAT_OK;
    }
    int rc = GAT_OK;
    bool all = true;
    for (int k = 0; k < 4 && all; k++)
        if (pd.edge_tables >> k & 1)
            all = try_malloc(&d->edge_tab[k], sizeof(gatk::KeptEdge) * (((size_t)g.m + 1) / 2 * 2), &rc);
    d->tab_size = std::min(g.n, kTabVertices);
    for (long long bytes = kPoolBytes; all && pd.n_tables && !d->pool; bytes /= 4) {
        const long long most = bytes / (8ll * pd.n_tables * d->tab_size);
        d->pool_tables = (unsigned)std::max(1ll, std::min<long long>(most, pd.key_edges ? g.m : g.n));
        d->pool_entries = (long long)pd.n_tables * d->pool_tables * d->tab_size;
        d->epoch = 255;  // cleared by the first count
        if (!try_malloc(&d->pool, sizeof(gatk::KeptEntry) * d->pool_entries, &rc)) all = !rc && bytes > kPoolLeast;
    }
    if (all) {
        d->keep = true;
    } else {
        d->drop_tables();
        d->tables_wait = kRetry;
    }
    return rc;
}

static int prepare(gat_plan *p, const gat_kernel_config *cfg_in, Launch *L) {
    DeviceInfo di;
    int rc = device_info(&di);
    if (rc) return rc;
    gat_kernel_config cfg{};
    if (cfg_in) cfg = *cfg_in;
    // the array store's waves wait on dependent list reads: its default grid
    // keeps twice the clique store's waves per CU (16 against 8)
    if (cfg.waves_per_cu <= 0 && (p->cp.clique_ks == 0 || cfg.vertex_store == 1)) cfg.waves_per_cu = 16;
    fill_defaults(&cfg);
    if (cfg.block_waves > 4) GAT_FAIL(GAT_EINFEASIBLE, "block_waves %d > 4", cfg.block_waves);
    Graph &g = *p->graph;
    const GatPlanDev &pd = p->cp.dev;
    if (!p->dev) {  // complete or not at all: after a failure the next count starts over
        std::unique_ptr<PlanDevice, void (*)(PlanDevice *)> d(new PlanDevice(), destroy_plan_device);
        rc = ensure_device_graph(g, &d->dg);
        if (rc) return rc;
        HIPCHECK(hipStreamCreateWithFlags(&d->stream, hipStreamNonBlocking));
        rc = need_malloc(&d->plan, sizeof(GatPlanDev), nullptr);
        if (!rc) rc = need_malloc(&d->ctl, sizeof(unsigned long long) * kCtlWords, nullptr);
        if (!rc) rc = need_malloc(&d->dargs, sizeof(gatk::KArgsSet), nullptr);
        if (rc) return rc;
        if (pd.edge_tables || pd.n_tables) {
            std::lock_guard<std::mutex> lk(d->dg->mu);
            degree_stats(g, d->dg.get());
        }
        choose_kept(pd, d->dg->neighbour_degree, (double)g.m, &d->pd);
        HIPCHECK(hipMemcpy(d->plan, &d->pd, sizeof(GatPlanDev), hipMemcpyHostToDevice));
        HIPCHECK(hipHostMalloc((void **)&d->result, sizeof(unsigned long long) * kCtlResult, hipHostMallocDefault));
        for (auto &e : d->ev) HIPCHECK(hipEventCreate(&e));
        p->dev = d.release();
    }
    PlanDevice *d = p->dev;
    L->busy = std::unique_lock<std::mutex>(d->busy);
    const long long chunk = cfg.queue_chunk;
    const bool clique = p->cp.clique_ks != 0 && cfg.vertex_store != 1;
    if (!clique && !d->gstore) {
        // HBM set buffers of the overflow launch, where every set fits in the
        // maximum degree: 16 waves per CU hide the latency of HBM-resident
        // sets, within 4 GiB of buffers.
        const size_t per_wave = (size_t)std::max(1, pd.n_store) * (size_t)std::max(1, g.max_deg) * 4;
        int waves = std::max(64, 16 * di.cus);
        while (waves > 64 && (double)waves * per_wave > 4.0 * (1 << 30)) waves /= 2;
        d->ovf_grid = waves;
        d->gstore_bytes = (size_t)waves * per_wave;
        rc = need_malloc(&d->gstore, std::max<size_t>(d->gstore_bytes, 64), d);
        if (rc) return rc;
    }
    if (cfg.vertex_store == 2 && !clique)
        GAT_FAIL(GAT_EINFEASIBLE, "bitmap vertex store needs a plan of cliques K3..K6 in unique or labeled mode");
    // single-child roots hand over single edges (run_task), others whole tasks
    const bool edge_grain = pd.nodes[0].child_count == 1;
    // overflow entries: edges or tasks, and split subtasks
    const long long waves = (long long)std::max(1, cfg.waves_per_cu * di.cus);
    const long long ovf_cap =
        clique ? 1 : (edge_grain ? g.m + 1 : std::max((g.m + chunk - 1) / chunk, 2 * kTasksPerWave * waves) + 1);
    const bool split = !clique && cfg.split_us > 0;
    // subtask lists: the LDS levels (kSubCap each), then the HBM list (LDS
    // overflow of the levels plus the HBM launch's splits, 3 kSubCap)
    if (split && !d->subs) {
        rc = need_malloc(&d->subs, sizeof(gatk::SplitTask) * (kLevels + 3) * kSubCap, d);
        if (rc) return rc;
    }
    if (ovf_cap > d->ovf_cap) {
        if (d->ovf) HIPCHECK(hipFree(d->ovf));
        d->ovf = nullptr;
        d->ovf_cap = 0;
        rc = need_malloc(&d->ovf, sizeof(long long) * ovf_cap, d);
        if (rc) return rc;
        d->ovf_cap = ovf_cap;
    }
    // A wave's LDS: its state (with the leaf counters the plan needs) and its
    // set buffers. A neighbour list is staged for binary searches; where
    // every vertex of its length has a bitmap, that serves, so the buffer ends
    // there (house: 17.9 KB per wave with full buffers, 8 waves per CU; 9 KB and
    // 16 with these). Configs are judged by the full size, whatever a plan needs of it.
    const size_t full = (sizeof(gatk::WaveState) + size_t(pd.n_store) * cfg.slot_capacity * 4 + 15) / 16 * 16;
    if (full * cfg.block_waves > di.lds_per_block)
        GAT_FAIL(GAT_EINFEASIBLE, "config needs %zu B of LDS per workgroup (device allows %zu)",
                 full * cfg.block_waves, di.lds_per_block);
    const int state_bytes = int((sizeof(gatk::WaveState) -
                                 size_t(GATP_MAX_LEAF_OPS - pd.max_leaf_ops) * sizeof(int) * 64 + 15) / 16 * 16);
    if (!clique && cfg.hub_degree >= 0) {
        rc = ensure_hubs(g, d->dg.get(), cfg.hub_degree, d, &L->hubs);
        if (rc) return rc;
    }
    const int staged = !clique && cfg.hub_degree >= 0 ? std::min(cfg.slot_capacity, L->hubs.full) : cfg.slot_capacity;
    const int stage_cap = std::min(cfg.slot_capacity, (staged + 3) / 4 * 4);
    long long store_off[GATP_MAX_STORE] = {}, entries = 0;
    for (int r = 0; r < pd.n_store; r++) {
        bool list = false;  // does some slot keep an intersection here?
        for (int i = 0; i < pd.n_slots; i++) list |= pd.slots[i].store == r && pd.slots[i].kind == GATP_LIST;
        store_off[r] = entries;
        entries += list ? cfg.slot_capacity : stage_cap;
    }
    const int wave_bytes = int((size_t(state_bytes) + size_t(entries) * 4 + 15) / 16 * 16);
    const size_t lds = size_t(wave_bytes) * cfg.block_waves;
    gatk::KArgs a{};
    a.off = d->dg->off;
    a.adj = d->dg->adj;
    a.split = d->dg->split;
    a.n = g.n;
    a.m = g.m;
    a.e_lo = 0;
    a.e_hi = g.m;
    a.plan = d->plan;
    a.counts = d->ctl;
    a.queue = d->ctl + kCtlHeads;
    a.drained = reinterpret_cast<unsigned *>(d->ctl + kCtlDrained);
    a.ovf = d->ovf;
    a.ovf_n = d->ctl + kCtlOvf;
    a.ovf_cap = d->ovf_cap;
    a.gstore = d->gstore;
    a.bytes = d->ctl + kCtlBytes;
    a.err = reinterpret_cast<unsigned *>(d->ctl + kCtlErr);
    a.cap = cfg.slot_capacity;
    a.stage_cap = stage_cap;
    a.state_bytes = state_bytes;
    for (int r = 0; r < GATP_MAX_STORE; r++) a.store_off[r] = store_off[r];
    a.chunk = cfg.queue_chunk;
    L->chunk = cfg.queue_chunk;
    a.lin_thr = cfg.search_linear_threshold;
    a.gallop_ratio = cfg.gallop_ratio;
    a.strategy = cfg.intersect_strategy;
    a.account = 0;
    a.sub_mode = 0;
    a.subs = d->subs;
    a.in_n = nullptr;
    a.out_n = a.ovf_n + 8 + 1;  // the main launch splits into level 1
    a.in_base = a.out_base = 0;
    a.in_cap = a.out_cap = kSubCap;
    a.sovf_n = a.ovf_n + 8 + kLevels + 1;
    a.sovf_base = kLevels * kSubCap;
    a.sovf_cap = 3 * kSubCap;
    if (!clique) {
        rc = ensure_tables(p);
        if (rc) return rc;
        for (int k = 0; k < 4; k++) a.edge_tab[k] = d->edge_tab[k];
        a.pool = d->pool;
        a.pool_tables = d->pool_tables;
        a.tab_size = d->tab_size;
        a.keep = d->keep;
    }
    a.split_ticks = split ? (long long)cfg.split_us * di.wall_khz / 1000 : 0;
    if (L->hubs.n) {
        a.hub_bits = L->hubs.rows->bits;
        a.hub_map = L->hubs.rows->map;
        a.hub_words = ((long long)g.n + 31) / 32;
        a.n_hubs = L->hubs.n;
    }
    L->a = a;
    L->block = dim3(64 * cfg.block_waves);
    const int total_waves = std::max(1, cfg.waves_per_cu * di.cus);
    L->grid = dim3(std::max(1, total_waves / cfg.block_waves));
    L->lds = lds;
    L->wave_bytes = wave_bytes;
    L->ao = a;
    L->waves = waves;
    L->edge_grain = edge_grain;
    bool lists = false;
    for (int i = 0; i < pd.n_ops; i++) lists |= pd.ops[i].kind == GATP_LIST;
    L->may_overflow = lists && g.max_deg > cfg.slot_capacity;
    for (int i = 0; i < pd.n_nodes; i++) L->pair |= pd.nodes[i].pair != 0;
    L->ao.cap = std::max(1, g.max_deg);
    for (int r = 0; r < GATP_MAX_STORE; r++) L->ao.store_off[r] = (long long)r * L->ao.cap;
    L->ovf_grid = dim3(d->ovf_grid);
    L->ovf_wave_bytes = state_bytes;
    L->ovf_lds = L->ovf_wave_bytes;
    L->clique = clique;
    if (clique) {
        const int max_out = max_out_degree(g);
        rc = ensure_core(g, d->dg.get(), &L->core);
        if (rc) return rc;
        gatk::CArgs c{};
        c.off = a.off;
        c.adj = a.adj;
        c.split = a.split;
        c.core = L->core->bits;
        c.core_n = L->core->n;
        c.n = a.n;
        c.m = a.m;
        c.root_lo = 0;
        c.root_hi = a.n;
        c.counts = a.counts;
        for (int k = 0; k < 8; k++) c.pat_of_k[k] = p->cp.clique_pattern[k];
        c.kmax = 31 - __builtin_clz(p->cp.clique_ks);
        c.queue = d->ctl + kCtlQueue;
        c.ovf_n = a.ovf_n;
        c.bytes = a.bytes;
        c.err = a.err;
        L->ca = c;
        rc = clique_shape(di, cfg, max_out, L);
        if (rc) return rc;
        for (int t = 0; t < gatk::CTIERS; t++) {
            if (L->tier_grid[t].x && !d->tier[t]) {
                rc = need_malloc(&d->tier[t], sizeof(int) * ((size_t)g.n + 1), d);
                if (rc) return rc;
            }
            L->ca.tier[t] = d->tier[t];
            L->ca.tier_cap[t] = d->tier[t] ? g.n + 1ll : 0;
        }
        if (L->tier_grid[3].x) {
            // HBM tier: one scratch area per workgroup, sized by the maximum out-degree
            const int hcap = std::max(32, max_out), ws = gatk::row_words(hcap);
            int groups = (int)L->tier_grid[3].x;
            while (groups > 64 && (double)groups * hcap * ws * 4 > 16e9) groups /= 2;
            if (d->big_cap < hcap || d->big_groups < groups) {
                if (d->grows) HIPCHECK(hipFree(d->grows));
                if (d->goff) HIPCHECK(hipFree(d->goff));
                d->grows = nullptr;
                d->goff = nullptr;
                d->big_cap = d->big_groups = 0;
                rc = need_malloc(&d->grows, (size_t)groups * hcap * ws * 4, d);
                if (!rc) rc = need_malloc(&d->goff, (size_t)groups * (hcap + 1) * 4, d);
                if (rc) return rc;
                d->big_cap = hcap;
                d->big_groups = groups;
            }
            L->tier_grid[3] = dim3(std::min(groups, d->big_groups));
            L->ca.grows = d->grows;
            L->ca.goff = d->goff;
            L->ca.hcap = d->big_cap;
        }
    }
    set_roots(L, g, 0, g.n);
    return GAT_OK;
}

static unsigned classify_grid(const gatk::CArgs &c) {
    const long long n = (long long)c.root_hi - c.root_lo;
    return (unsigned)std::max(1ll, std::min(64ll, n / (4 * gatk::kClassifyThreads)));
}

// Launch of a workgroup tier with rows in LDS.
template <int MODE, int MW, int TIER, int NW, class F>
static void launch_tier(const Launch &L, gatk::CArgs &c, hipStream_t s, F &&tl_take) {
    if (!L.tier_grid[TIER].x) return;
    c.tl_base = tl_take((int)L.tier_grid[TIER].x);
    hipLaunchKernelGGL((gatk::clique_block_kernel<MW, TIER, NW, MODE>), L.tier_grid[TIER], dim3(64 * NW),
                       L.tier_lds[TIER], s, c);
}

// Enqueue the whole count on the plan's stream (capturable: no memsets).
static int enqueue(PlanDevice *d, const Launch &L, bool account, bool events, bool timeline = false) {
    hipStream_t s = d->stream;
    // timeline: one record per wave (array store, clique main launch) or per
    // workgroup (clique tiers), launch after launch
    long long *tl = nullptr;
    int tl_next = 0;
    auto tl_take = [&](int units) {  // first record of the next launch
        const int b = tl_next;
        tl_next += units;
        return b;
    };
    if (timeline) {
        const int waves = (int)(L.grid.x * (L.block.x / 64));
        const long long need = L.clique ? (long long)waves + L.tier_grid[0].x + L.tier_grid[1].x + L.tier_grid[2].x +
                                              L.tier_grid[3].x
                                        : (long long)waves * (1 + (L.a.split_ticks > 0 ? kLevels : 0)) +
                                              (long long)L.ovf_grid.x * (L.a.split_ticks > 0 ? 2 : 1);
        if (need > kTlCap) GAT_FAIL(GAT_ELIMIT, "timeline needs %lld records (> %d)", need, kTlCap);
        if (!d->tl) {
            const int rc = need_malloc(&d->tl, sizeof(long long) * gatk::kTlFields * kTlCap, d, nullptr, true);
            if (rc) return rc;
        }
        hipLaunchKernelGGL(gatk::fill_u64, dim3(64), dim3(256), 0, s, (unsigned long long *)d->tl,
                           (long long)gatk::kTlFields * kTlCap, ~0ull);
        tl = d->tl;
    }
    hipLaunchKernelGGL(gatk::fill_u64, dim3(8), dim3(256), 0, s, d->ctl, (long long)(L.clique ? kCtlHeads : kCtlWords),
                       0ull);
    gatk::KArgs a = L.a, ao = L.ao;
    a.account = ao.account = account ? 1 : 0;
    if (account) {  // W_alg is accumulated where the values are computed
        a.keep = ao.keep = 0;
    }
    if (events) HIPCHECK(hipEventRecord(d->ev[0], s));
    d->cleared = false;
    if (!L.clique && a.keep && a.pool) {
        // epochs 1 .. 254 for counts in turn, with the pool cleared before the
        // first; the replays of a captured count share one, so each clears it
        const bool clear = !events || d->epoch >= 254;
        if (events) d->epoch = clear ? 1 : d->epoch + 1;
        a.epoch = ao.epoch = events ? d->epoch : 255;
        d->cleared = clear;
        if (clear)
            hipLaunchKernelGGL(gatk::fill_u64, dim3(2048), dim3(256), 0, s, (unsigned long long *)d->pool,
                               d->pool_entries, 0ull);
    }
    for (int k = 0; k < 4 && !L.clique && a.keep; k++)
        if (a.edge_tab[k]) {
            d->cleared = true;
            hipLaunchKernelGGL(gatk::fill_u64, dim3(2048), dim3(256), 0, s, (unsigned long long *)a.edge_tab[k],
                               (a.m + 1) / 2, ~0ull);
        }
    if (events && d->cleared) HIPCHECK(hipEventRecord(d->ev[4], s));
    a.tl = ao.tl = tl;
    ao.bytes = a.bytes + 1;  // second launch: its own W_alg counter
    const int waves = (int)(L.grid.x * (L.block.x / 64));
    gatk::CArgs c = L.ca;
    c.account = account ? 1 : 0;
    c.tl = tl;
    if (L.clique) {
        // W_alg accounting and timeline records come from separate kernel
        // instantiations (MODE bits 0 and 1)
        auto run = [&](auto mode_tag) -> int {
            constexpr int T = decltype(mode_tag)::value;
            if (L.heavy)
                hipLaunchKernelGGL(gatk::clique_classify, dim3(classify_grid(c)), dim3(gatk::kClassifyThreads), 0, s, c);
            c.tl_base = tl_take(waves);
            hipLaunchKernelGGL(gatk::clique_kernel<T>, L.grid, L.block, L.clique_lds, s, c);
            if (events) HIPCHECK(hipEventRecord(d->ev[1], s));
            c.bytes = a.bytes + 1;  // tiers 0 and 1: their own W_alg counter
            launch_tier<T, gatk::CT0W, 0, gatk::CNW0>(L, c, s, tl_take);
            launch_tier<T, gatk::CT1W, 1, gatk::CNW1>(L, c, s, tl_take);
            if (events) HIPCHECK(hipEventRecord(d->ev[3], s));
            c.bytes = a.bytes + 2;  // tiers 2 and 3
            launch_tier<T, gatk::CT2W, 2, gatk::CNW2>(L, c, s, tl_take);
            if (L.tier_grid[3].x) {
                c.tl_base = tl_take((int)L.tier_grid[3].x);
                hipLaunchKernelGGL(gatk::clique_hbm_kernel<T>, L.tier_grid[3], dim3(64 * gatk::CNW3), 0, s, c);
            }
            return GAT_OK;
        };
        const int mode = (account ? 1 : 0) | (timeline ? 2 : 0);
        const int rc = mode == 0   ? run(std::integral_constant<int, 0>{})
                       : mode == 1 ? run(std::integral_constant<int, 1>{})
                       : mode == 2 ? run(std::integral_constant<int, 2>{})
                                   : run(std::integral_constant<int, 3>{});
        if (rc) return rc;
    } else {
        const bool pair = a.keep && L.pair;
        auto pick = [&](auto plain, auto kept, auto paired) { return pair ? paired : a.keep ? kept : plain; };
        const auto main_k = pick(gatk::engine_plain_kernel<false>, gatk::engine_kernel<false>, gatk::engine_pair_kernel<false>);
        const auto sub_k = pick(gatk::engine_plain_sub_kernel<false>, gatk::engine_sub_kernel<false>,
                                gatk::engine_pair_sub_kernel<false>);
        const auto main_hbm_k = pick(gatk::engine_plain_kernel<true>, gatk::engine_kernel<true>, gatk::engine_pair_kernel<true>);
        const auto sub_hbm_k = pick(gatk::engine_plain_sub_kernel<true>, gatk::engine_sub_kernel<true>,
                                    gatk::engine_pair_sub_kernel<true>);
        const bool split = a.split_ticks > 0;
        gatk::KArgsSet set;
        a.tl_base = tl_take(waves);
        set.a[0] = a;
        for (int k = 1; k <= kLevels; k++) {
            gatk::KArgs &sk = set.a[k] = a;
            sk.sub_mode = k;
            sk.in_n = a.ovf_n + 8 + k;
            sk.in_base = (k - 1) * kSubCap;
            sk.out_n = k < kLevels ? a.ovf_n + 8 + k + 1 : nullptr;  // the last level does not split
            sk.out_base = k * kSubCap;
            sk.bytes = a.bytes + 1;
            sk.tl_base = split ? tl_take(waves) : 0;
        }
        ao.out_n = a.ovf_n + 8 + kLevels + 1;  // the HBM launch splits into the HBM list
        ao.out_base = kLevels * kSubCap;
        ao.out_cap = 3 * kSubCap;
        ao.tl_base = tl_take((int)L.ovf_grid.x);
        set.a[kLevels + 1] = ao;
        gatk::KArgs &sh = set.a[kLevels + 2] = ao;
        sh.sub_mode = kLevels + 1;  // HBM buffers, no further splitting
        sh.in_n = a.ovf_n + 8 + kLevels + 1;
        sh.in_base = kLevels * kSubCap;
        sh.in_cap = 3 * kSubCap;
        sh.out_n = nullptr;
        sh.tl_base = split ? tl_take((int)L.ovf_grid.x) : 0;
        hipLaunchKernelGGL(gatk::put_kargs, dim3(1), dim3(256), 0, s, set, d->dargs);
        const gatk::KArgs *args = d->dargs->a;
        hipLaunchKernelGGL(main_k, L.grid, L.block, L.lds, s, args, L.wave_bytes);
        if (events) HIPCHECK(hipEventRecord(d->ev[1], s));
        for (int k = 1; k <= kLevels && split; k++)  // split subtasks, level by level, in LDS like the main launch
            hipLaunchKernelGGL(sub_k, L.grid, L.block, L.lds, s, args + k, L.wave_bytes);
        if (L.may_overflow) {
            hipLaunchKernelGGL(main_hbm_k, L.ovf_grid, dim3(64), L.ovf_lds, s, args + kLevels + 1, L.ovf_wave_bytes);
            if (split)
                hipLaunchKernelGGL(sub_hbm_k, L.ovf_grid, dim3(64), L.ovf_lds, s, args + kLevels + 2,
                                   L.ovf_wave_bytes);
        }
        if (events) HIPCHECK(hipEventRecord(d->ev[3], s));
    }
    if (events) HIPCHECK(hipEventRecord(d->ev[2], s));
    HIPCHECK(hipGetLastError());
    d->tl_n = timeline ? tl_next : 0;
    return GAT_OK;
}

// counts_out: the requested counts, or with raw set the engine's raw sums
// (a shard's share of divisor * count, before the divisor and multiplier).
static int finish(gat_plan *p, const Launch &L, uint64_t *counts_out, gat_count_stats *st, bool timed,
                  bool raw_sums = false) {
    PlanDevice *d = p->dev;
    const int np = p->cp.dev.n_patterns;
    unsigned long long raw[GATP_MAX_TERMS] = {};
    HIPCHECK(hipMemcpyAsync(d->result, d->ctl, sizeof(unsigned long long) * kCtlResult, hipMemcpyDeviceToHost,
                            d->stream));
    HIPCHECK(hipStreamSynchronize(d->stream));
    const unsigned long long *copies = d->result, *ovf = copies + kCtlOvf, *bytes = copies + kCtlBytes;
    const unsigned int err = (unsigned)copies[kCtlErr];
    for (int c = 0; c < gatk::kCountCopies; c++)
        for (int i = 0; i < np; i++) raw[i] += copies[c * GATP_MAX_TERMS + i];
    // flags 2 and 4: a device work list (overflow tasks, subtasks, clique
    // tiers) filled up; 1 and 8: states the host's sizing rules out
    if (err & 6u) GAT_FAIL(GAT_ELIMIT, "a device work list overflowed (engine flags 0x%x)", err);
    if (err) GAT_FAIL(GAT_EINTERNAL, "engine reported an internal inconsistency (flags 0x%x)", err);
    for (int i = 0; i < np && raw_sums; i++)
        if (counts_out) counts_out[i] = raw[i];
    for (int i = 0; i < np && !raw_sums; i++) {
        const PatternInfo &pi = p->cp.patterns[i];
        if (raw[i] % pi.divisor)
            GAT_FAIL(GAT_EINVAL, "internal: raw count %llu of pattern %d not divisible by %llu", raw[i], i,
                     (unsigned long long)pi.divisor);
        if (counts_out) counts_out[i] = raw[i] / pi.divisor * pi.multiplier;
    }
    if (st) {
        std::memset(st, 0, sizeof(*st));
        if (timed) {
            float ms = 0, ms_main = 0, ms_second = 0;
            HIPCHECK(hipEventElapsedTime(&ms, d->ev[0], d->ev[2]));
            HIPCHECK(hipEventElapsedTime(&ms_main, d->ev[d->cleared ? 4 : 0], d->ev[1]));
            HIPCHECK(hipEventElapsedTime(&ms_second, d->ev[1], d->ev[3]));
            st->seconds = ms / 1000.0;
            st->main_kernel_ms = ms_main;
            st->second_kernel_ms = ms_second;
        }
        st->overflow_tasks = L.clique ? ovf[4] : ovf[0];
        unsigned long long made = 0;
        for (int k = 1; k <= kLevels; k++) made += std::min<unsigned long long>(ovf[8 + k], (unsigned long long)kSubCap);
        made += std::min<unsigned long long>(ovf[8 + kLevels + 1], (unsigned long long)(3 * kSubCap));
        st->split_tasks = L.clique ? 0 : (int32_t)(made - ovf[2]);
        st->split_overflow = L.clique ? 0 : (int32_t)ovf[2];
        for (int k = 0; k < 4; k++)
            st->split_level[k] = L.clique ? 0
                                          : (int64_t)std::min<unsigned long long>(
                                                ovf[8 + 1 + k], (unsigned long long)(k < kLevels ? kSubCap : 3 * kSubCap));
        st->alg_bytes = bytes[0] + bytes[1] + bytes[2];
        st->alg_bytes_main = bytes[0];
        st->alg_bytes_second = bytes[1];
        st->tasks = (uint64_t)L.tasks;
        st->grid_blocks = (int)L.grid.x;
        st->block_threads = (int)L.block.x;
        st->lds_bytes = (int)L.lds;
    }
    return GAT_OK;
}

}  // namespace gat

using namespace gat;

extern "C" int gat_device_count(int32_t *out) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) n = 0;
    if (out) *out = n;
    return GAT_OK;
}

extern "C" int gat_count(gat_plan *p, const gat_kernel_config *cfg, uint32_t flags, uint64_t *counts_out,
                         gat_count_stats *stats) {
    if (!p) GAT_FAIL(GAT_EINVAL, "null plan");
    Launch L;
    int rc = prepare(p, cfg, &L);
    if (rc) return rc;
    rc = enqueue(p->dev, L, (flags & GAT_FLAG_ACCOUNT) != 0, true, (flags & GAT_FLAG_TIMELINE) != 0);
    if (rc) return rc;
    return finish(p, L, counts_out, stats, true);
}

extern "C" int gat_plan_timeline(const gat_plan *p, int64_t *out, int64_t cap, int64_t *n_out,
                                 double *ticks_per_ms) {
    if (!p || !n_out) GAT_FAIL(GAT_EINVAL, "null plan or n_out");
    DeviceInfo di;
    int rc = device_info(&di);
    if (rc) return rc;
    PlanDevice *d = p->dev;
    *n_out = 0;
    if (ticks_per_ms) *ticks_per_ms = (double)di.wall_khz;
    if (!d || !d->tl || d->tl_n == 0) return GAT_OK;
    std::vector<long long> rec((size_t)d->tl_n * gatk::kTlFields);
    HIPCHECK(hipStreamSynchronize(d->stream));
    HIPCHECK(hipMemcpy(rec.data(), d->tl, rec.size() * sizeof(long long), hipMemcpyDeviceToHost));
    long long t_min = LLONG_MAX;
    for (int i = 0; i < d->tl_n; i++)
        if (rec[(size_t)i * gatk::kTlFields] >= 0) t_min = std::min(t_min, rec[(size_t)i * gatk::kTlFields + 2]);
    int64_t n = 0;
    for (int i = 0; i < d->tl_n; i++) {
        const long long *r = &rec[(size_t)i * gatk::kTlFields];
        if (r[0] < 0) continue;  // a unit that wrote no record
        if (out && n < cap)
            for (int f = 0; f < gatk::kTlFields; f++) out[n * gatk::kTlFields + f] = (f == 2 || f == 3) ? r[f] - t_min : r[f];
        n++;
    }
    *n_out = n;
    return GAT_OK;
}

extern "C" int gat_count_shard(gat_plan *p, const gat_kernel_config *cfg, uint32_t flags, int32_t root_begin,
                               int32_t root_end, uint64_t *raw_out, gat_count_stats *stats) {
    if (!p) GAT_FAIL(GAT_EINVAL, "null plan");
    const int32_t n = p->graph->n;
    if (root_begin < 0 || root_end < root_begin || root_end > n)
        GAT_FAIL(GAT_EINVAL, "root range [%d, %d) is not within [0, %d)", root_begin, root_end, n);
    Launch L;
    int rc = prepare(p, cfg, &L);
    if (rc) return rc;
    set_roots(&L, *p->graph, root_begin, root_end);
    rc = enqueue(p->dev, L, (flags & GAT_FLAG_ACCOUNT) != 0, true, (flags & GAT_FLAG_TIMELINE) != 0);
    if (rc) return rc;
    return finish(p, L, raw_out, stats, true, true);
}

extern "C" int gat_count_shard_edges(gat_plan *p, const gat_kernel_config *cfg, uint32_t flags, int64_t edge_begin,
                                     int64_t edge_end, uint64_t *raw_out, gat_count_stats *stats) {
    if (!p) GAT_FAIL(GAT_EINVAL, "null plan");
    const long long m = p->graph->m;
    if (edge_begin < 0 || edge_end < edge_begin || edge_end > m)
        GAT_FAIL(GAT_EINVAL, "edge range [%lld, %lld) is not within [0, %lld)", (long long)edge_begin,
                 (long long)edge_end, m);
    Launch L;
    int rc = prepare(p, cfg, &L);
    if (rc) return rc;
    if (L.clique)
        GAT_FAIL(GAT_EUNSUPPORTED, "edge shards need the array store (vertex_store = 1): the bitmap clique store "
                                   "shards by top vertex (gat_count_shard)");
    // the array store's queue runs over root edges; every task finds its
    // root by binary search, so any edge range is a shard
    set_edges(&L, edge_begin, edge_end);
    rc = enqueue(p->dev, L, (flags & GAT_FLAG_ACCOUNT) != 0, true, (flags & GAT_FLAG_TIMELINE) != 0);
    if (rc) return rc;
    return finish(p, L, raw_out, stats, true, true);
}

// ---- allocation-free clique count ---------------------------------------
// Scratch of gat_count_cliques_noalloc, one copy per device for the life of
// the process: kNaHead words of counters (queues [8,24), work-list sizes
// [24,40), W_alg [40,44), error flags at word 44, the copies of the counts
// from word 64 on), then
// kNaBody int32 entries laid out for the graph's size: the split[] array (n),
// the lists of workgroup tiers 0 (n), 1 (kNaTierCap) and 2 (kNaTierCap / 2),
// and the core bitmap within the rest (28 to 58 MiB, so up to 31,000 core
// vertices). 64 MiB and 17 KiB in all.
constexpr int kNaMaxV = 1 << 22;
constexpr long long kNaTierCap = 1 << 20;
constexpr long long kNaHead = 64 + GATP_MAX_TERMS * gatk::kCountCopies;
constexpr long long kNaBody = 1 << 24;
constexpr long long kNaWords = kNaHead + kNaBody / 2;
static __device__ __align__(256) unsigned long long scratch[kNaWords];

// Device address of this device's scratch, looked up once per device (the
// host-side name `scratch` is only a handle for the runtime, never an address).
static int noalloc_scratch(unsigned long long **out) {
    static std::mutex mu;
    static unsigned long long *addr[64] = {};
    int dev = 0;
    HIPCHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) GAT_FAIL(GAT_ENODEV, "device index %d out of range", dev);
    std::lock_guard<std::mutex> lk(mu);
    if (!addr[dev]) {
        void *ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr)
            GAT_FAIL(GAT_ENODEV, "hipGetSymbolAddress(scratch) failed on device %d: %s", dev, hipGetErrorString(e));
        addr[dev] = static_cast<unsigned long long *>(ptr);
    }
    *out = addr[dev];
    return GAT_OK;
}

extern "C" int gat_count_cliques_noalloc(const int64_t *d_offsets, const int32_t *d_adj, int32_t v_cnt, int32_t kmax,
                                         const gat_kernel_config *cfg_in, void *stream, uint64_t *counts_out) {
    if (!d_offsets || !d_adj || !counts_out) GAT_FAIL(GAT_EINVAL, "null graph or counts pointer");
    if (kmax < 3 || kmax > 6) GAT_FAIL(GAT_EINVAL, "kmax %d is not within [3, 6]", kmax);
    if (v_cnt < 0) GAT_FAIL(GAT_EINVAL, "negative v_cnt");
    if (v_cnt > kNaMaxV)
        GAT_FAIL(GAT_ELIMIT, "v_cnt %d exceeds the allocation-free count's limit of %d vertices", v_cnt, kNaMaxV);
    DeviceInfo di;
    int rc = device_info(&di);
    if (rc) return rc;
    gat_kernel_config cfg{};
    if (cfg_in) cfg = *cfg_in;
    fill_defaults(&cfg);
    if (cfg.block_waves > 4) GAT_FAIL(GAT_EINFEASIBLE, "block_waves %d > 4", cfg.block_waves);
    Launch L;
    L.ca = {};
    L.ca.kmax = kmax;
    rc = clique_shape(di, cfg, 32 * gatk::CT2W, &L);  // the out-degrees are not known here: every LDS tier runs
    if (rc) return rc;
    if (L.ca.lds_dmax < 32 * gatk::CT2W)
        GAT_FAIL(GAT_EINFEASIBLE, "the allocation-free count needs %d KiB of LDS per workgroup",
                 (int)((gatk::tier_lds(gatk::CT2W, gatk::CNW2) + 1023) / 1024));
    unsigned long long *h = nullptr;
    rc = noalloc_scratch(&h);
    if (rc) return rc;
    gatk::CArgs &c = L.ca;
    c.off = reinterpret_cast<const long long *>(d_offsets);
    c.adj = d_adj;
    int *split = reinterpret_cast<int *>(h + kNaHead);
    c.split = split;
    c.tier[0] = split + v_cnt;
    c.tier[1] = c.tier[0] + v_cnt;
    c.tier[2] = c.tier[1] + kNaTierCap;
    c.tier[3] = nullptr;
    c.tier_cap[0] = v_cnt;
    c.tier_cap[1] = kNaTierCap;
    c.tier_cap[2] = kNaTierCap / 2;
    c.tier_cap[3] = 0;
    unsigned *core = reinterpret_cast<unsigned *>(c.tier[2] + c.tier_cap[2]);
    const long long used = reinterpret_cast<int *>(core) - split;
    c.core = core;
    // built in every call: as large as for a graph of degree 32 (58 MB of rows
    // for 50,000 vertices of degree 40 took 80 of 430 us)
    c.core_n = core_vertices(v_cnt, std::min(kNaBody - used, std::max<long long>(1 << 21, 128ll * v_cnt)));
    c.n = v_cnt;
    c.m = 0;
    c.root_lo = 0;
    c.root_hi = v_cnt;
    c.chunk = clique_chunk(L.chunk, v_cnt, (long long)L.grid.x * (L.block.x / 64));
    c.counts = h + 64;
    for (int k = 0; k < 8; k++) c.pat_of_k[k] = (k >= 3 && k <= kmax) ? k - 3 : -1;
    c.queue = h + 8;
    c.ovf_n = h + 24;
    c.bytes = h + 40;
    c.err = reinterpret_cast<unsigned *>(h + 44);
    c.grows = nullptr;  // no HBM tier: vertices with more than lds_dmax neighbours below them are refused
    c.goff = nullptr;
    c.hcap = c.lds_dmax;
    c.account = 0;
    c.tl = nullptr;
    c.tl_base = 0;
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(gatk::fill_u64, dim3(4), dim3(256), 0, s, h, kNaHead, 0ull);
    if (v_cnt > 0) {
        hipLaunchKernelGGL(gatk::split_kernel, dim3(1024), dim3(256), 0, s, reinterpret_cast<const long long *>(d_offsets),
                           d_adj, v_cnt, split);
        if (c.core_n > 0)
            hipLaunchKernelGGL(gatk::core_rows_kernel, dim3(std::min((c.core_n + 3) / 4, 4096)), dim3(256), 0, s,
                               reinterpret_cast<const long long *>(d_offsets), d_adj, split, c.core_n, core);
        hipLaunchKernelGGL(gatk::clique_classify, dim3(classify_grid(c)), dim3(gatk::kClassifyThreads), 0, s, c);
        hipLaunchKernelGGL(gatk::clique_kernel<0>, L.grid, L.block, L.clique_lds, s, c);
        auto no_tl = [](int) { return 0; };
        launch_tier<0, gatk::CT0W, 0, gatk::CNW0>(L, c, s, no_tl);
        launch_tier<0, gatk::CT1W, 1, gatk::CNW1>(L, c, s, no_tl);
        launch_tier<0, gatk::CT2W, 2, gatk::CNW2>(L, c, s, no_tl);
    }
    HIPCHECK(hipGetLastError());
    unsigned long long head[kNaHead], raw[8] = {};
    HIPCHECK(hipMemcpyAsync(head, h, sizeof(head), hipMemcpyDeviceToHost, s));
    HIPCHECK(hipStreamSynchronize(s));
    const unsigned long long *copies = head + 64, heavy = head[24 + 5];
    const unsigned int err = (unsigned)head[44];
    if (err & 16u)
        GAT_FAIL(GAT_ELIMIT, "a vertex has more than %d neighbours below it; the allocation-free count has no HBM tier",
                 c.lds_dmax);
    if ((err & 4u) || heavy > (unsigned long long)kNaTierCap)
        GAT_FAIL(GAT_ELIMIT, "more than %lld heavy vertices for one workgroup tier", kNaTierCap);
    if (err) GAT_FAIL(GAT_EINTERNAL, "engine reported an internal inconsistency (flags 0x%x)", err);
    for (int i = 0; i < gatk::kCountCopies; i++)
        for (int k = 0; k < 8; k++) raw[k] += copies[i * GATP_MAX_TERMS + k];
    for (int k = 3; k <= kmax; k++) counts_out[k - 3] = raw[k - 3];
    return GAT_OK;
}

extern "C" int gat_count_graph(gat_plan *p, const gat_kernel_config *cfg, int32_t replays, uint64_t *counts_out,
                               gat_count_stats *stats) {
    if (!p || replays < 1) GAT_FAIL(GAT_EINVAL, "null plan or replays < 1");
    Launch L;
    int rc = prepare(p, cfg, &L);
    if (rc) return rc;
    PlanDevice *d = p->dev;
    if (d->gexec) {
        (void)hipGraphExecDestroy(d->gexec);
        d->gexec = nullptr;
    }
    if (d->graph) {
        (void)hipGraphDestroy(d->graph);
        d->graph = nullptr;
    }
    HIPCHECK(hipStreamBeginCapture(d->stream, hipStreamCaptureModeThreadLocal));
    rc = enqueue(d, L, false, false);
    hipGraph_t graph = nullptr;
    const hipError_t ec = hipStreamEndCapture(d->stream, &graph);
    if (rc) return rc;
    if (ec != hipSuccess) GAT_FAIL(GAT_ENODEV, "hipStreamEndCapture failed: %s", hipGetErrorString(ec));
    d->graph = graph;
    HIPCHECK(hipGraphInstantiate(&d->gexec, graph, nullptr, nullptr, 0));
    for (int r = 0; r < replays; r++) {
        HIPCHECK(hipEventRecord(d->ev[0], d->stream));
        HIPCHECK(hipGraphLaunch(d->gexec, d->stream));
        HIPCHECK(hipEventRecord(d->ev[2], d->stream));
        if (r + 1 < replays) HIPCHECK(hipStreamSynchronize(d->stream));
    }
    rc = finish(p, L, counts_out, stats, false);
    if (rc) return rc;
    if (stats) {
        float ms = 0;
        HIPCHECK(hipEventElapsedTime(&ms, d->ev[0], d->ev[2]));
        stats->seconds = ms / 1000.0;
    }
    return GAT_OK;
}

extern "C" int gat_copy_probe(uint64_t bytes, int32_t reps, double *gbps_out) {
    DeviceInfo di;
    int rc = device_info(&di);
    if (rc) return rc;
    if (bytes < 16 || reps < 1) GAT_FAIL(GAT_EINVAL, "copy probe needs bytes >= 16 and reps >= 1");
    const long long n = (long long)(bytes / 16);
    int4 *src = nullptr, *dst = nullptr;
    rc = need_malloc(&src, n * 16, nullptr);
    if (!rc) rc = need_malloc(&dst, n * 16, nullptr);
    if (rc) {
        if (src) (void)hipFree(src);
        return rc;
    }
    hipEvent_t e0, e1;
    HIPCHECK(hipEventCreate(&e0));
    HIPCHECK(hipEventCreate(&e1));
    const int grid = di.cus * 8;
    hipLaunchKernelGGL(gatk::copy_kernel, dim3(grid), dim3(256), 0, nullptr, src, dst, n);
    HIPCHECK(hipEventRecord(e0, nullptr));
    for (int r = 0; r < reps; r++) hipLaunchKernelGGL(gatk::copy_kernel, dim3(grid), dim3(256), 0, nullptr, src, dst, n);
    HIPCHECK(hipEventRecord(e1, nullptr));
    HIPCHECK(hipEventSynchronize(e1));
    float ms = 0;
    HIPCHECK(hipEventElapsedTime(&ms, e0, e1));
    if (gbps_out) *gbps_out = 2.0 * n * 16 * reps / (ms * 1e-3) / 1e9;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipFree(src);
    (void)hipFree(dst);
    return GAT_OK;
}
