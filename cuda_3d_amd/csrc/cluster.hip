// cluster.hip -- Euclidean clustering and residual-based segmentation as connected components
// of the radius graph.
//
// Reference: cuda_euclidean_clustering (src/geometry/cuda_clustering.cu:31-110) and
// cuda_residual_based_segmentation (:251-341) download the radius-neighbour lists and run a
// breadth-first search on the host, seeding from the lowest unvisited index.  The residual form
// follows an edge only when the two points' absolute ICP residuals differ by less than 0.003
// (:291-293).  A search stops expanding once its queue holds max_cluster_size points (:75-96,
// :308-328), leaving the rest of that component to later seeds; a queue is kept as a cluster when
// it has at least min_cluster_size points, and clusters are numbered in seed order.
//
// Here the components come from a lock-free union-find on the device:
//   1. chain    size[i] = 0; parent[i] = the first point of i's run of consecutive indices whose
//               neighbours are linked (raster and lattice order put most neighbours side by side),
//               within the workgroup; a run's first point takes the point before it if linked: no
//               atomics, no search
//   2. pairs    (clouds large and dense enough for it, hook_direct) every point and the few before it in
//               cell order, if linked, are joined; snapshot: each point's root, in cell order, and the most
//               frequent root of a sample (`big`), if it is that of half the sample
//   3. hook     with a big component: the points outside it link their root with that of every linked
//               neighbour of another snapshot component.  An edge inside a component is already
//               there, and one into the big component is seen from its other end, so the bulk of
//               a scene takes no part.  Else every point does so with the neighbours before it in cell
//               order.  Linked: the radius search's own predicate, squared FP64 distance < r^2, and for the
//               residual form the residual gate
//   4. compress parent[i] = root (a read-only walk, then a store to the point's own entry),
//               size[root] += 1 and, after links by rank, low[root] = min(i) (one atomic per wave and root
//               run); lowest: the component's lowest index, the reference's seed, becomes its root
//   5. cut      only for components above max_cluster_size (listed by k_cc_lowest): the
//               reference's truncated searches, replayed exactly on the device (k_cc_truncate),
//               re-root the component's points on the seeds of the pieces it is cut into
//   6. rank     kept roots (size >= min) are numbered by an exclusive scan in index order
//   7. label    label[i] = number of its root's cluster, or -1
// A root is only ever linked, by compare-and-swap, under a point of lower rank (cc_rank; without pairs of
// lower index, so that the root is the lowest point) that was a root, so links form no cycle; parent pointers always name an ancestor, so the path-halving stores
// in find() may race with the compare-and-swaps without losing a link.
//
// Neighbour lists are visited in the radius search's canonical order, (squared distance,
// index), where the reference visits them in its grid-cell order; only the pieces of a cut
// component depend on that order.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <vector>

#include "gca_device.hpp"
#include "gca_internal.hpp"
#include "neighbours.hpp"

namespace gca {

namespace {

constexpr int kCcBlock = 256;

// Workgroup scope lets the load hit L1.  A stale parent is still an ancestor and every step goes
// towards the root, so walks on stale values end, and every link is validated by an agent-scope
// compare-and-swap; each failed one strictly lowers the rank of the higher of the two roots.
__device__ __forceinline__ int32_t cc_load(int32_t *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Root of x with path halving.
__device__ __forceinline__ int32_t cc_find(int32_t *parent, int32_t x)
{
    int32_t y = cc_load(parent + x);
    while (y != x) {
        const int32_t z = cc_load(parent + y);
        if (z == y) return y;
        __hip_atomic_store(parent + x, z, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        x = z;
        y = cc_load(parent + x);
    }
    return x;
}

// Root of x without writes: the compress pass stores each point's root into its own entry
// only, so a halving store from another thread can never replace a root with an ancestor.
__device__ __forceinline__ int32_t cc_root(int32_t *parent, int32_t x)
{
    int32_t y = cc_load(parent + x);
    while (y != x) {
        x = y;
        y = cc_load(parent + x);
    }
    return x;
}

// Which of two roots stays one: a mix of the index's bits (a bijection, so never a tie).  By index
// alone the rows of an image hang under one another one by one, and the walks grow with the image
// (289k points at 1 cm: pairs and hook 88 + 76 us by index, 38 + 49 by rank).
__device__ __forceinline__ uint32_t cc_rank(int32_t x)
{
    const uint32_t m = (uint32_t)x * 2654435769u;
    return m ^ m >> 15;
}

// Links the trees of u and v (any nodes of them; the point's own root is passed in).  LOWEST: by index, so
// that a tree's root is its lowest point.
template <bool LOWEST>
__device__ __forceinline__ void cc_union(int32_t *parent, int32_t u, int32_t v)
{
    while (u != v) {
        if (LOWEST ? u > v : cc_rank(u) > cc_rank(v)) {
            const int32_t t = u;
            u = v;
            v = t;
        }
        int32_t expect = v;  // link the root of higher rank under the other one
        if (__hip_atomic_compare_exchange_strong(parent + v, &expect, u, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT))
            return;
        u = cc_find(parent, u);
        v = cc_find(parent, expect);
    }
}

// Edge gate of the residual-based segmentation (cuda_clustering.cu:291-293): |r_a - r_b| in FP32,
// compared with the double 0.003.
__device__ __forceinline__ bool residual_close(float a, float b) { return (double)fabsf(a - b) < 0.003; }

// res == nullptr: plain Euclidean clustering.
__device__ __forceinline__ bool residual_gate(const float *__restrict__ res, int32_t a, int32_t b)
{
    return res == nullptr || residual_close(res[a], res[b]);
}

constexpr int kCcWide = 1024;

__global__ __launch_bounds__(kCcWide) void k_cc_chain(const CloudHdr *__restrict__ h, const float4 *__restrict__ xyzi,
                                                     const float *__restrict__ res, double r2,
                                                     int32_t *__restrict__ parent, uint32_t *__restrict__ size,
                                                     int32_t *__restrict__ low, int32_t *__restrict__ big,
                                                     uint32_t *__restrict__ oversized)
{
    __shared__ int32_t last[kCcWide / kWave];  // per wavefront: its last run's first point, -1 if it has none
    const int n = h->n;
    const int lane = lane_id(), w = threadIdx.x / kWave;
    const int i = blockIdx.x * kCcWide + threadIdx.x;
    if (i == 0) {
        *oversized = 0;
        *big = -1;
    }
    bool linked = false;
    if (i > 0 && i < n) {
        const float4 p = xyzi[i], q = xyzi[i - 1];
        linked = dist2(p.x, p.y, p.z, q.x, q.y, q.z) < r2 && residual_gate(res, i, i - 1);
    }
    const bool start = !linked || threadIdx.x == 0;
    const uint64_t starts = __ballot(start);
    if (lane == 0) last[w] = starts ? i + 63 - __builtin_clzll(starts) : -1;
    __syncthreads();
    if (i >= n) return;
    const uint64_t upto = starts & ((2ull << lane) - 1ull);
    int32_t head = upto ? i - lane + 63 - __builtin_clzll(upto) : -1;
    for (int v = w; head < 0;) head = last[--v];  // the workgroup's first point starts a run
    parent[i] = threadIdx.x == 0 && linked ? i - 1 : head;
    size[i] = 0;
    if (low) low[i] = INT_MAX;
}

template <bool LOWEST>
__device__ __forceinline__ void cc_link(int32_t *parent, int32_t &ri, int32_t j)
{
    const int32_t rj = cc_find(parent, j);
    if (rj != ri) {
        ri = cc_find(parent, ri);  // short walk: ri was a root not long ago
        if (rj != ri) {
            cc_union<LOWEST>(parent, ri, rj);  // a compare-and-swap only for distinct roots
            ri = cc_find(parent, ri);
        }
    }
}

// Pair t joins sorted point s = t * step / back and the one t % back + 1 before it.
__global__ __launch_bounds__(kCcBlock) void k_cc_pairs(const CloudHdr *__restrict__ h, const float4 *__restrict__ sxyzi,
                                                      const int32_t *__restrict__ order, const float *__restrict__ res,
                                                      double r2, int step, int back, int32_t *parent)
{
    const int n = h->n;
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t s = k / back * step, t = s - 1 - k % back;
    if (s >= n || t < 0) return;
    const float4 p = sxyzi[s], q = sxyzi[t];
    const int32_t i = order[s], j = order[t];
    if (!(dist2(p.x, p.y, p.z, q.x, q.y, q.z) < r2) || !residual_gate(res, i, j)) return;
    if (cc_load(parent + i) == cc_load(parent + j)) return;  // most pairs: joined already
    int32_t ri = cc_find(parent, i);
    cc_link<false>(parent, ri, j);
}

// Each point's root, in cell order, and its residual likewise (what the hook reads per candidate).
__global__ __launch_bounds__(kCcBlock) void k_cc_snapshot(const CloudHdr *__restrict__ h, const int32_t *__restrict__ order,
                                                         const float *__restrict__ res, int32_t *parent,
                                                         int32_t *__restrict__ snap, float *__restrict__ sres)
{
    const int n = h->n;
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const int32_t i = order[s];
    const int32_t r = cc_root(parent, i);
    __hip_atomic_store(parent + i, r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    snap[s] = r;
    if (res) sres[s] = res[i];
}

// The most frequent root among kCcSample points spread over the cloud (a tie: the lowest), or -1 if it is
// not half of them: the hook then takes each edge from one end, where leaving out a big component's points
// makes it look at the others' edges from both.  Any answer is right; a good one lets the hook leave out
// most points.
constexpr int kCcSample = 1024;

__global__ __launch_bounds__(kCcSample) void k_cc_big(const CloudHdr *__restrict__ h, const int32_t *__restrict__ snap,
                                                     int32_t *__restrict__ big)
{
    __shared__ int32_t key[2 * kCcSample];
    __shared__ uint32_t cnt[2 * kCcSample];
    __shared__ unsigned long long best;
    const int t = threadIdx.x, n = h->n;
    for (int e = t; e < 2 * kCcSample; e += kCcSample) {
        key[e] = -1;
        cnt[e] = 0u;
    }
    if (t == 0) best = 0ull;
    __syncthreads();
    if (n > 0) {
        const int32_t r = snap[(int64_t)t * n / kCcSample];
        // (not the multiplier of cc_rank: roots are of low rank, and would all fall into few entries)
        uint32_t e = ((uint32_t)r * 0x85ebca6bu) >> 21;
        for (;;) {  // the table is never full
            const int32_t old = atomicCAS(&key[e], -1, r);
            if (old == -1 || old == r) break;
            e = (e + 1) & (2 * kCcSample - 1);
        }
        atomicAdd(&cnt[e], 1u);
    }
    __syncthreads();
    unsigned long long mine = 0ull;
    for (int e = t; e < 2 * kCcSample; e += kCcSample)
        if (cnt[e]) mine = max(mine, ((unsigned long long)cnt[e] << 32) | (uint32_t)(INT_MAX - key[e]));
    for (int m = 1; m < kWave; m <<= 1) mine = max(mine, (unsigned long long)__shfl_xor(mine, m, kWave));
    if (lane_id() == 0) atomicMax(&best, mine);  // (one a wavefront: a thousand of them queue for 40 us)
    __syncthreads();
    if (t == 0) *big = 2 * (uint32_t)(best >> 32) >= kCcSample ? INT_MAX - (int32_t)(uint32_t)best : -1;
}

// Hook: kCcLanes lanes per point outside the big component (points in cell order), each lane a share of the point's
// candidates from the 27 cells around it.  Between two points outside the big component the later
// one in cell order takes the edge, and without one the walk ends at the point's own slot (and loads the
// neighbours' roots with them: 300k points in clusters of 150, 285 -> 240 us); the components do not depend
// on which end links an edge.  DIRECT: no pairs and no snapshot came before, each
// point stands for itself (snap is the cell order, sres the residuals by index).  The whole
// labelling is bound by the union-find's dependent loads and contended compare-and-swaps: 92k points of
// a 424x240 frame at 2 cm 97 us plain and 128 us gated, where hooking every edge of every point took
// 270 us for either; 289k points of a 640x480 frame at 1 cm 125 us (568 every edge).
constexpr int kCcLanes = 8;
constexpr int kCcUnroll = 4;

template <bool DIRECT>
__global__ __launch_bounds__(kCcBlock) void k_cc_hook(const CloudHdr *__restrict__ h, GridDesc g,
                                                     const uint32_t *__restrict__ start,
                                                     const float4 *__restrict__ sxyzi,
                                                     const int32_t *__restrict__ order,
                                                     const int32_t *__restrict__ snap,
                                                     const float *__restrict__ sres, const int32_t *__restrict__ big_p,
                                                     int32_t *parent)
{
    const int n = h->n;
    const int gl = (int)threadIdx.x & (kCcLanes - 1);
    const int s = (int)((blockIdx.x * blockDim.x + threadIdx.x) / kCcLanes);  // the group's point
    if (s >= n) return;  // the whole group
    const int32_t big = DIRECT ? -1 : *big_p, mine = snap[s];
    if (mine == big) return;
    const GridView v = make_view(g, start, order, sxyzi);
    const double r2 = (double)g.radius * (double)g.radius;
    const float4 p = sxyzi[s];
    const float res = sres ? sres[DIRECT ? mine : s] : 0.f;
    Box b;
    if (!grid_range(g, p.x, p.y, p.z, b.lo, b.hi)) return;
    int32_t ri = cc_find(parent, mine);
    if (big < 0) {
        group_walk_box<kCcUnroll, 3, true>(v, b, gl, kCcLanes, -1, -1, [&](uint32_t t, float4 q, bool valid, int32_t other) {
            if (!valid || other == mine || !(dist2(q.x, q.y, q.z, p.x, p.y, p.z) < r2)) return;
            if (sres && !residual_close(res, sres[DIRECT ? other : (int32_t)t])) return;
            cc_link<DIRECT>(parent, ri, other);
        }, [] { return true; }, (uint32_t)s, snap);
        return;
    }
    // once this component is part of the big one (by this point's doing or another's), its other
    // edges into the big one are done with; likewise a second edge into the component just joined
    bool joined = ri == cc_find(parent, big);
    int32_t done = mine;
    group_walk_box<kCcUnroll>(v, b, gl, kCcLanes, -1, -1, [&](uint32_t t, float4 q, bool valid) {
        if (!valid || !(dist2(q.x, q.y, q.z, p.x, p.y, p.z) < r2)) return;
        const int32_t other = snap[t];
        if (other == mine || other == done || (other == big ? joined : t > (uint32_t)s)) return;
        if (sres && !residual_close(res, sres[t])) return;
        cc_link<false>(parent, ri, other);
        done = other;
        joined |= other == big;
    }, [&] {
        joined = (__ballot(joined) >> (lane_id() & ~(kCcLanes - 1)) & ((1u << kCcLanes) - 1u)) != 0;
        return true;
    });
}

// The big component's points are counted per workgroup (its count takes one atomic a workgroup
// instead of one a wavefront: same-address atomics queue), the others' per wavefront and root.
__global__ __launch_bounds__(kCcWide) void k_cc_compress(const CloudHdr *__restrict__ h, int32_t *parent,
                                                        uint32_t *__restrict__ size, int32_t *__restrict__ low,
                                                        const int32_t *__restrict__ big_p)
{
    __shared__ uint32_t s_count;
    __shared__ int32_t s_big, s_low;
    const int n = h->n;
    const int i = blockIdx.x * kCcWide + threadIdx.x;
    const bool on = i < n;
    if (threadIdx.x == 0) {
        s_count = 0u;
        s_low = INT_MAX;
        s_big = *big_p < 0 ? -1 : cc_root(parent, *big_p);
    }
    const int32_t r = on ? cc_root(parent, i) : -1;
    __syncthreads();
    const int32_t big = s_big;
    if (on) __hip_atomic_store(parent + i, r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint64_t in_big = __ballot(on && r == big);
    if (lane_id() == 0 && in_big) {
        atomicAdd(&s_count, (uint32_t)__popcll(in_big));
        atomicMin(&s_low, i + __ffsll((long long)in_big) - 1);
    }
    // lanes sharing a root add once: the lowest such lane, whose index is their lowest
    uint64_t pending = __ballot(on && r != big);
    while (pending) {
        const int leader = __ffsll((long long)pending) - 1;
        const int32_t lr = __shfl(r, leader);
        const uint64_t same = __ballot(on && r == lr);
        if (lane_id() == leader) {
            atomicAdd(size + lr, (uint32_t)__popcll(same));
            if (low) atomicMin(low + lr, i);
        }
        pending &= ~same;
    }
    __syncthreads();
    if (threadIdx.x == 0 && s_count) {
        atomicAdd(size + big, s_count);
        atomicMin(low + big, s_low);  // (with a big component there is low)
    }
}

struct CutJob {
    int32_t root, size, base;  // base: the job's region of the queue buffer (set on the host)
    int32_t pad;
};

// Each component takes its lowest index as its root: every point's entry (read and written by its
// own thread only) and the size, which moves from the union-find's root.  Components above max_size:
// one job each (root, size) for the truncated searches; *n_jobs counts them (the jobs' order does not
// matter: each cut is independent of the others).
__global__ __launch_bounds__(kCcBlock) void k_cc_lowest(const CloudHdr *__restrict__ h, int32_t *__restrict__ parent,
                                                       uint32_t *__restrict__ size, const int32_t *__restrict__ low,
                                                       uint32_t max_size, CutJob *__restrict__ jobs,
                                                       uint32_t *__restrict__ n_jobs)
{
    const int n = h->n;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int32_t r = parent[i], m = low ? low[r] : r;
    parent[i] = m;
    if (r != i) return;
    const uint32_t sz = size[i];
    if (m != i) {
        size[m] = sz;
        size[i] = 0;
    }
    if (sz <= max_size) return;
    const uint32_t k = atomicAdd(n_jobs, 1u);
    jobs[k] = CutJob{m, (int32_t)sz, 0, 0};
}

// Claim words of the truncated searches: kUnvisited, kVisited, or the key (queue position + 1,
// list position) of the lowest proposal in the current round.
constexpr unsigned long long kUnvisited = ~0ull;
constexpr unsigned long long kVisited = 0ull;

__global__ __launch_bounds__(kCcBlock) void k_cc_claims_clear(const CloudHdr *__restrict__ h,
                                                             unsigned long long *__restrict__ claim)
{
    const int n = h->n;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) claim[i] = kUnvisited;
}

__device__ __forceinline__ unsigned long long claim_load(const unsigned long long *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void claim_store(unsigned long long *p, unsigned long long v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The reference's searches over one component above max_size (one workgroup per component):
// seeds in ascending index among the component's unvisited points; from each, a breadth-first
// queue that stops expanding once it holds max_size points.  The queue is grown a frontier chunk
// of up to kCutBlock elements at a time, reproducing the sequential order exactly:
//   1. each element proposes (its queue position, list position) for every unvisited, gated
//      neighbour with an atomic minimum on the neighbour's claim word;
//   2. an element's new points are the neighbours whose claim it holds, in list order (a point
//      goes to the first element, in queue order, that lists it, as in the sequential search);
//   3. element t is expanded only if the queue held fewer than max_size points before it (an
//      exclusive scan of the counts), so the chunk's expanded elements are a prefix;
//   4. claims of elements cut off (and every other non-winning proposal) are reset.
// A piece's points are then re-rooted on its seed, and size[seed] is the piece's size.  Claims
// never leave the component (its points' neighbours are its points), so workgroups are
// independent.
constexpr int kCutBlock = 1024;

__global__ __launch_bounds__(kCutBlock) void k_cc_truncate(const CloudHdr *__restrict__ h, const CutJob *__restrict__ jobs,
                                                          int32_t *__restrict__ parent, uint32_t *__restrict__ size,
                                                          const int32_t *__restrict__ off,
                                                          const int32_t *__restrict__ nbr,
                                                          const float *__restrict__ res,
                                                          unsigned long long *__restrict__ claim,
                                                          int32_t *__restrict__ queue, uint32_t max_size)
{
    __shared__ uint32_t lds[kCutBlock / kWave + 1];
    __shared__ int32_t s_seed;
    __shared__ uint32_t s_add, s_proc;
    const int n = h->n;
    const CutJob J = jobs[blockIdx.x];
    int32_t *q = queue + J.base;
    const int32_t root = J.root;
    const int t = threadIdx.x;
    int32_t cursor = root;
    for (;;) {
        // next seed: the lowest unvisited point of the component at or after the cursor
        if (t == 0) s_seed = INT_MAX;
        __syncthreads();
        for (; cursor < n; cursor += kCutBlock) {
            const int32_t i = cursor + t;
            if (i < n && parent[i] == root && claim_load(claim + i) != kVisited) atomicMin(&s_seed, i);
            __syncthreads();
            if (s_seed != INT_MAX) break;
        }
        const int32_t seed = s_seed;
        __syncthreads();
        if (seed == INT_MAX) break;
        cursor = seed + 1;
        if (t == 0) {
            q[0] = seed;
            claim_store(claim + seed, kVisited);
        }
        uint32_t qlen = 1, head = 0;
        __syncthreads();
        while (head < qlen && qlen < max_size) {
            const uint32_t level_end = qlen;
            while (head < level_end && qlen < max_size) {
                const uint32_t cnt = min((uint32_t)kCutBlock, level_end - head);
                const bool on = (uint32_t)t < cnt;
                const int32_t e = on ? q[head + t] : -1;
                const int32_t l0 = on ? off[e] : 0, l1 = on ? off[e + 1] : 0;
                const unsigned long long key_hi = (unsigned long long)(head + t + 1) << 32;
                for (int32_t l = l0; l < l1; ++l) {  // 1. proposals
                    const int32_t v = nbr[l];
                    if (residual_gate(res, e, v) && claim_load(claim + v) != kVisited)
                        atomicMin(claim + v, key_hi | (unsigned long long)(l - l0));
                }
                __syncthreads();
                uint32_t won = 0;  // 2. points this element takes
                for (int32_t l = l0; l < l1; ++l) {
                    const int32_t v = nbr[l];
                    won += residual_gate(res, e, v) && claim_load(claim + v) == (key_hi | (unsigned long long)(l - l0));
                }
                uint32_t total;
                const uint32_t before = block_excl_scan<kCutBlock>(won, lds, &total);
                (void)total;
                const bool expand = on && qlen + before < max_size;  // 3. a prefix of the chunk
                if (expand) {
                    uint32_t pos = qlen + before;
                    for (int32_t l = l0; l < l1; ++l) {
                        const int32_t v = nbr[l];
                        if (residual_gate(res, e, v) && claim_load(claim + v) == (key_hi | (unsigned long long)(l - l0))) {
                            q[pos++] = v;
                            claim_store(claim + v, kVisited);
                        }
                    }
                }
                // the last expanded element (the chunk's last, or the last before the queue is
                // full) publishes how many were expanded and how many points they added
                if (expand && (t + 1 == (int)cnt || qlen + before + won >= max_size)) {
                    s_proc = (uint32_t)t + 1;
                    s_add = before + won;
                }
                __syncthreads();
                for (int32_t l = l0; l < l1; ++l) {  // 4. reset proposals that did not win
                    const int32_t v = nbr[l];
                    if (residual_gate(res, e, v)) {
                        const unsigned long long c = claim_load(claim + v);
                        if (c != kVisited && c != kUnvisited) claim_store(claim + v, kUnvisited);
                    }
                }
                head += s_proc;
                qlen += s_add;
                __syncthreads();
            }
        }
        // the piece: every queued point (expanded or not) is re-rooted on the seed
        for (uint32_t k = t; k < qlen; k += kCutBlock) parent[q[k]] = seed;
        if (t == 0) size[seed] = qlen;
        __syncthreads();
    }
}

// kept roots: flag + per-block count for the scan
__global__ __launch_bounds__(kCcBlock) void k_cc_flag(const CloudHdr *__restrict__ h,
                                                     const int32_t *__restrict__ parent,
                                                     const uint32_t *__restrict__ size, uint32_t min_size,
                                                     uint8_t *__restrict__ kept, uint32_t *__restrict__ bcnt)
{
    __shared__ uint32_t wc[kCcBlock / kWave];
    const int n = h->n;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    bool k = false;
    if (i < n) {
        const uint32_t sz = parent[i] == i ? size[i] : 0u;
        k = sz > 0 && sz >= min_size;
        kept[i] = k ? 1 : 0;
    }
    const uint64_t m = __ballot(k);
    if (lane_id() == 0) wc[threadIdx.x / kWave] = (uint32_t)__popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (int w = 0; w < kCcBlock / kWave; ++w) t += wc[w];
        bcnt[blockIdx.x] = t;
    }
}

// cluster number of each kept root, written over its size entry
__global__ __launch_bounds__(kCcBlock) void k_cc_rank(const CloudHdr *__restrict__ h,
                                                     const uint8_t *__restrict__ kept,
                                                     const uint32_t *__restrict__ boff, uint32_t *__restrict__ size)
{
    __shared__ uint32_t wo[kCcBlock / kWave];
    const int n = h->n;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool k = i < n && kept[i];
    const uint64_t m = __ballot(k);
    const int w = threadIdx.x / kWave;
    if (lane_id() == 0) wo[w] = (uint32_t)__popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (int v = 0; v < kCcBlock / kWave; ++v) {
            const uint32_t c = wo[v];
            wo[v] = t;
            t += c;
        }
    }
    __syncthreads();
    if (k) size[i] = boff[blockIdx.x] + wo[w] + (uint32_t)__popcll(m & ((1ull << lane_id()) - 1ull));
}

__global__ __launch_bounds__(kCcBlock) void k_cc_label(const CloudHdr *__restrict__ h, const uint8_t *__restrict__ kept,
                                                      const uint32_t *__restrict__ rank, int32_t *__restrict__ label)
{
    const int n = h->n;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int32_t r = label[i];
    label[i] = kept[r] ? (int32_t)rank[r] : -1;
}

// Whether the hook takes every edge at once.  Pairs, snapshot and the search for a big component cost three
// launches, 20 to 30 us, and pay where a component of most points spares the hook its bulk: in larger clouds
// whose points lie close (their number per column of cells along the grid's shortest side tells, for the
// surfaces that a camera sees).  us a labelling, every edge at once / pairs first, plain then gated; rendered
// frames: 80x60 at 2 cm 73 / 100, 73 / 97; 160x120 at 1, 2 and 4 cm (0.3, 1.1 and 4 points a column) 80 / 106,
// 92 / 106, 190 / 98, gated 78 / 101, 92 / 105, 130 / 107; 240x180 at 1 and 2 cm (0.6 and 2.4) 92 / 113, 229 / 115,
// gated 91 / 113, 126 / 109; 320x240 at 1 cm (1.1) 172 / 122, gated 108 / 114; 640x480 at 5 mm (1.1) 415 / 277,
// gated 298 / 216.  16k points scattered on a surface at 2 cm (3 a column): 237 / 130, gated 89 / 106.
bool hook_direct(const GridDesc &g, int64_t n, bool gated)
{
    int64_t d[3] = {g.dims[0], g.dims[1], g.dims[2]};
    std::sort(d, d + 3);
    return n < (gated ? 20000 : 12000) || 4 * n < 3 * d[1] * d[2];
}

}  // namespace

int32_t launch_euclidean_clustering(gca_ctx ctx, gca_cloud c, float tolerance, uint32_t min_size,
                                    uint32_t max_size, int32_t *label, uint32_t *counts_dev, const float *res)
{
    Grid G = c->grid;  // the grid may be one built for a nearby radius: search at the tolerance
    G.desc.radius = tolerance;
    const int64_t nb = std::max<int64_t>(1, (c->cap + kCcBlock - 1) / kCcBlock);
    uint32_t *size = (uint32_t *)ctx_scratch(ctx, 25, sizeof(uint32_t) * (size_t)c->cap, false);
    uint8_t *kept = (uint8_t *)ctx_scratch(ctx, 2, (size_t)c->cap, false);
    uint32_t *bcnt = (uint32_t *)ctx_scratch(ctx, 3, sizeof(uint32_t) * (nb + 1), false);
    uint32_t *boff = (uint32_t *)ctx_scratch(ctx, 4, sizeof(uint32_t) * (nb + 1), false);
    CutJob *jobs = (CutJob *)ctx_scratch(ctx, 28, sizeof(CutJob) * (size_t)std::max<int64_t>(c->cap, 1), false);
    if (!size || !kept || !bcnt || !boff || !jobs) return GCA_ERR_OUT_OF_MEMORY;
    const dim3 grid((unsigned)nb), block(kCcBlock);
    int32_t *big = (int32_t *)ctx_scratch(ctx, 46, 256, false);
    const bool direct = hook_direct(G.desc, c->host_hdr.n, res != nullptr);
    int32_t *low = direct ? nullptr : (int32_t *)ctx_scratch(ctx, 9, sizeof(int32_t) * (size_t)c->cap, false);
    if (!big || (!direct && !low)) return GCA_ERR_OUT_OF_MEMORY;
    const double r2 = (double)tolerance * (double)tolerance;
    const dim3 wide((unsigned)std::max<int64_t>(1, (c->cap + kCcWide - 1) / kCcWide));
    hipLaunchKernelGGL(k_cc_chain, wide, dim3(kCcWide), 0, ctx->stream, c->hdr, c->xyzi, res, r2, label, size, low, big,
                       counts_dev + 1);
    const dim3 grid_hook((unsigned)std::max<int64_t>(1, (c->cap * kCcLanes + kCcBlock - 1) / kCcBlock));
    if (direct) {
        hipLaunchKernelGGL(k_cc_hook<true>, grid_hook, block, 0, ctx->stream, c->hdr, G.desc, G.start, G.sxyzi, G.order,
                           (const int32_t *)G.order, res, (const int32_t *)big, label);
    } else {
        int32_t *snap = (int32_t *)ctx_scratch(ctx, 11, sizeof(int32_t) * (size_t)c->cap, false);
        float *sres = res ? (float *)ctx_scratch(ctx, 12, sizeof(float) * (size_t)c->cap, false) : nullptr;
        if (!snap || (res && !sres)) return GCA_ERR_OUT_OF_MEMORY;
        // Every second point and its predecessor connect the rows that a cell holds; the residual gate
        // lets about a third of the neighbours through, so it takes more pairs before a scene's bulk
        // holds together.  Pairs / hook of a 424x240 frame at 2 cm: 19 / 36 us plain (every fourth: 16 /
        // 53), gated 51 / 79 us with three predecessors of every point (two 38 / 118, four 70 / 67); at
        // 640x480 gated 93 / 276 (two 73 / 387, four 120 / 236).  (Linked by index; by rank, as now, 22 / 35
        // and 37 / 58.)
        const int step = res ? 1 : 2, back = res ? 3 : 1;
        const dim3 grid_pairs((unsigned)std::max<int64_t>(1, (c->cap / step * back + back + kCcBlock - 1) / kCcBlock));
        hipLaunchKernelGGL(k_cc_pairs, grid_pairs, block, 0, ctx->stream, c->hdr, G.sxyzi, G.order, res, r2, step, back, label);
        hipLaunchKernelGGL(k_cc_snapshot, grid, block, 0, ctx->stream, c->hdr, G.order, res, label, snap, sres);
        hipLaunchKernelGGL(k_cc_big, dim3(1), dim3(kCcSample), 0, ctx->stream, c->hdr, (const int32_t *)snap, big);
        hipLaunchKernelGGL(k_cc_hook<false>, grid_hook, block, 0, ctx->stream, c->hdr, G.desc, G.start, G.sxyzi, G.order,
                           (const int32_t *)snap, (const float *)sres, (const int32_t *)big, label);
    }
    hipLaunchKernelGGL(k_cc_compress, wide, dim3(kCcWide), 0, ctx->stream, c->hdr, label, size, low,
                       (const int32_t *)big);
    hipLaunchKernelGGL(k_cc_lowest, grid, block, 0, ctx->stream, c->hdr, label, size, (const int32_t *)low, max_size, jobs,
                       counts_dev + 1);
    GCA_HIP(hipGetLastError());
    GCA_HIP(hipMemcpyAsync(ctx->pinned, counts_dev + 1, sizeof(uint32_t), hipMemcpyDeviceToHost, ctx->stream));
    GCA_HIP(hipStreamSynchronize(ctx->stream));
    const uint32_t n_jobs = *(const uint32_t *)ctx->pinned;
    if (n_jobs > 0) {
        // Components above max_size are cut as the reference's searches cut them.  Their
        // neighbour lists (radius search of the cloud against itself, canonical order) and a
        // queue region per component, laid out on the host.
        std::vector<CutJob> hj(n_jobs);
        GCA_HIP(hipMemcpyAsync(hj.data(), jobs, sizeof(CutJob) * n_jobs, hipMemcpyDeviceToHost, ctx->stream));
        GCA_HIP(hipStreamSynchronize(ctx->stream));
        int64_t base = 0;
        for (auto &j : hj) {
            j.base = (int32_t)base;
            base += j.size;
        }
        GCA_HIP(hipMemcpyAsync(jobs, hj.data(), sizeof(CutJob) * n_jobs, hipMemcpyHostToDevice, ctx->stream));
        const int64_t n = c->host_hdr.n;
        int32_t *off = (int32_t *)ctx_scratch(ctx, 29, sizeof(int32_t) * (size_t)(n + 1), false);
        int32_t *queue = (int32_t *)ctx_scratch(ctx, 30, sizeof(int32_t) * (size_t)std::max<int64_t>(base, 1), false);
        unsigned long long *claim =
            (unsigned long long *)ctx_scratch(ctx, 31, sizeof(unsigned long long) * (size_t)std::max<int64_t>(n, 1), false);
        if (!off || !queue || !claim) return GCA_ERR_OUT_OF_MEMORY;
        int64_t total = 0;
        GCA_TRY(launch_radius(ctx, c, c, tolerance, 0, off, nullptr, 0, &total));
        int32_t *nbr = (int32_t *)ctx_scratch(ctx, 32, sizeof(int32_t) * (size_t)std::max<int64_t>(total, 1), false);
        if (!nbr) return GCA_ERR_OUT_OF_MEMORY;
        GCA_TRY(launch_radius(ctx, c, c, tolerance, 0, off, nbr, total, &total));
        hipLaunchKernelGGL(k_cc_claims_clear, grid, block, 0, ctx->stream, c->hdr, claim);
        hipLaunchKernelGGL(k_cc_truncate, dim3(n_jobs), dim3(kCutBlock), 0, ctx->stream, c->hdr, jobs, label, size, off, nbr,
                           res, claim, queue, max_size);
        GCA_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(k_cc_flag, grid, block, 0, ctx->stream, c->hdr, label, size, min_size, kept, bcnt);
    GCA_HIP(hipGetLastError());
    GCA_TRY(exclusive_scan_u32(ctx, bcnt, boff, nb, counts_dev));
    hipLaunchKernelGGL(k_cc_rank, grid, block, 0, ctx->stream, c->hdr, kept, boff, size);
    hipLaunchKernelGGL(k_cc_label, grid, block, 0, ctx->stream, c->hdr, kept, size, label);
    GCA_HIP(hipGetLastError());
    return GCA_OK;
}

}  // namespace gca
