// neighbours.hpp -- device building blocks of the neighbour queries (grid.hip, normals.hip, icp.hip): the
// walk of a query's grid cells by a group of lanes, and the selection of the smallest
// (distance, index) keys without sorting them all.
#pragma once

#include <cfloat>
#include <climits>

#include "gca_device.hpp"
#include "gca_internal.hpp"

namespace gca {

struct GridView {
    GridDesc g;
    const uint32_t *start;
    const int32_t *order;
    const float4 *sxyzi;
};

__device__ __forceinline__ GridView make_view(const GridDesc &g, const uint32_t *start, const int32_t *order,
                                              const float4 *sxyzi)
{
    GridView v;
    v.g = g;
    v.start = start;
    v.order = order;
    v.sxyzi = sxyzi;
    return v;
}

// Orders a wavefront's LDS writes before its later reads.
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---- sums over a group of G <= 16 aligned lanes ------------------------------------------------
// Butterflies by data-parallel moves inside a row of 16 lanes (no LDS round trip, unlike shuffles).
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_move(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xf, 0xf, true);
}

template <int CTRL>
__device__ __forceinline__ double dpp_move(double v)
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const uint32_t lo = dpp_move<CTRL>((uint32_t)u), hi = dpp_move<CTRL>((uint32_t)(u >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

template <int CTRL>
__device__ __forceinline__ long long dpp_move(long long v)
{
    return __double_as_longlong(dpp_move<CTRL>(__longlong_as_double(v)));
}

template <int G, class T>
__device__ __forceinline__ T group_min(T v)
{
    static_assert(G == 4 || G == 8 || G == 16, "a group lies within a row");
    v = min(v, dpp_move<0xB1>(v));
    v = min(v, dpp_move<0x4E>(v));
    if constexpr (G >= 8) v = min(v, dpp_move<0x141>(v));
    if constexpr (G >= 16) v = min(v, dpp_move<0x140>(v));
    return v;
}

template <int G, class T>
__device__ __forceinline__ T group_sum(T v)
{
    static_assert(G == 1 || G == 2 || G == 4 || G == 8 || G == 16, "a group lies within a row");
    if constexpr (G >= 2) v += dpp_move<0xB1>(v);    // quad_perm 1,0,3,2
    if constexpr (G >= 4) v += dpp_move<0x4E>(v);    // quad_perm 2,3,0,1
    if constexpr (G >= 8) v += dpp_move<0x141>(v);   // row_half_mirror
    if constexpr (G >= 16) v += dpp_move<0x140>(v);  // row_mirror
    return v;
}

// ---- candidate walk of a lane group --------------------------------------------------------
// A query's candidates are the z-runs of its box's columns of cells, 3 x 3 columns when the cell is
// at least the radius (more only where rounding widens the box by a cell: the walk then goes on in
// further blocks of 3 x 3).
struct Box {
    int32_t lo[3], hi[3];
};

// Holds a loaded value here: without it the compiler moves the load to its use, under the use's
// condition, and waits for each load by itself.
template <class T>
__device__ __forceinline__ void keep_loaded(T &v)
{
    asm volatile("" : "+v"(v));
}

// Run r of the A x A columns from (x0, y0) on: candidates cum[r] .. cum[r + 1], at slot off[r] + f;
// columns outside the box, and column (sx, sy), are empty, and so is what lies at slots from `limit` on.
// Cell numbers fit 32 bits (at most
// 2^25 cells), and the columns lie a fixed stride apart, so a bound is one 32-bit offset: numbering
// the columns by division cost more than the walk's distances.
template <int A>
__device__ __forceinline__ void block_runs(const uint32_t *__restrict__ start, const GridDesc &g, const Box &b, int x0, int y0,
                                           int sx, int sy, uint32_t limit, uint32_t off[A * A], uint32_t cum[A * A + 1])
{
    const uint32_t dy = (uint32_t)g.dims[2], dx = (uint32_t)g.dims[1] * dy;
    const uint32_t len = (uint32_t)(b.hi[2] + 1 - b.lo[2]);
    // every bound is loaded, those of columns outside from the box's last column: a load under a
    // condition is waited for before the next one goes out, up to nine round trips instead of one
    // (with the same in group_walk: nearest neighbours of a 424x240 frame 66 -> 45 us, normals of a
    // 640x480 frame at 1 cm 36 -> 31, outlier flags 27 -> 20)
    uint32_t s0[A * A], s1[A * A];
#pragma unroll
    for (int r = 0; r < A * A; ++r) {
        const uint32_t x = (uint32_t)min(x0 + r / A, b.hi[0]), y = (uint32_t)min(y0 + r % A, b.hi[1]);
        const uint32_t c = x * dx + y * dy + (uint32_t)b.lo[2];
        s0[r] = *(const uint32_t *)((const char *)start + 4u * c);
        s1[r] = *(const uint32_t *)((const char *)start + 4u * (c + len));
    }
#pragma unroll
    for (int r = 0; r < A * A; ++r) {
        keep_loaded(s0[r]);
        keep_loaded(s1[r]);
    }
#pragma unroll
    for (int r = 0; r < A * A; ++r) {
        const int x = x0 + r / A, y = y0 + r % A;
        const bool in = x <= b.hi[0] && y <= b.hi[1] && !(x == sx && y == sy);
        off[r] = s0[r];
        s1[r] = min(s1[r], limit);
        cum[r + 1] = in && s1[r] > s0[r] ? s1[r] - s0[r] : 0u;
    }
    cum[0] = 0;
#pragma unroll
    for (int r = 0; r < A * A; ++r) {
        off[r] -= cum[r];
        cum[r + 1] += cum[r];
    }
}

// The candidates [0, total) at slots slot(f) by a group of gs lanes (a power of two, lanes g = 0 ..
// gs - 1 of one wavefront), U loads in flight per lane: calls f(slot, point, valid) U times per
// round on every lane of the group (valid: the lane has a candidate), then more(): false ends the
// walk (the same answer on the group's lanes).  Returns whether it went to the end.  With IDS, ids[slot]
// is loaded with the point and goes to f as well.
template <int U, bool IDS = false, class S, class F, class M>
__device__ __forceinline__ bool group_walk(const float4 *__restrict__ sxyzi, uint32_t total, int g, int gs, S &&slot, F &&f,
                                           M &&more, const int32_t *__restrict__ ids = nullptr)
{
    for (uint32_t f0 = 0; f0 < total; f0 += gs * U) {
        float4 c[U];
        uint32_t sl[U];
        int32_t id[IDS ? U : 1];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            sl[u] = slot(min(f0 + u * gs + g, total - 1u));  // a lane past the end loads the last one
            c[u] = sxyzi[sl[u]];
            if constexpr (IDS) id[u] = ids[sl[u]];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            keep_loaded(c[u].x);
            keep_loaded(c[u].y);
            keep_loaded(c[u].z);
            if constexpr (IDS) keep_loaded(id[u]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if constexpr (IDS) f(sl[u], c[u], f0 + u * gs + g < total, id[u]);
            else f(sl[u], c[u], f0 + u * gs + g < total);
        }
        if (!more()) return false;
    }
    return true;
}

// The walk over box b (without column (sx, sy), and up to slot `limit`), a block of A x A columns as one
// flattened range.
template <int U, int A = 3, bool IDS = false, class F, class M>
__device__ __forceinline__ void group_walk_box(const GridView &v, const Box &b, int g, int gs, int sx, int sy, F &&f, M &&more,
                                               uint32_t limit = UINT_MAX, const int32_t *__restrict__ ids = nullptr)
{
    constexpr int kRuns = A * A;
    for (int x0 = b.lo[0]; x0 <= b.hi[0]; x0 += A)
        for (int y0 = b.lo[1]; y0 <= b.hi[1]; y0 += A) {
            uint32_t off[kRuns], cum[kRuns + 1];
            block_runs<A>(v.start, v.g, b, x0, y0, sx, sy, limit, off, cum);
            auto slot = [&](uint32_t fi) {
                uint32_t o = off[0];
#pragma unroll
                for (int r = 1; r < kRuns; ++r) {
                    const uint32_t next = off[r];  // read before the choice, so that off stays in registers
                    o = fi >= cum[r] ? next : o;
                }
                return o + fi;
            };
            if (!group_walk<U, IDS>(v.sxyzi, cum[kRuns], g, gs, slot, f, more, ids)) return;
        }
}

template <int U, class F>
__device__ __forceinline__ void group_walk_box(const GridView &v, const Box &b, int g, int gs, F &&f)
{
    group_walk_box<U>(v, b, g, gs, -1, -1, f, [] { return true; });
}

// The query's own column of cells, kept within box b.
__device__ __forceinline__ void own_column(const GridDesc &g, float qx, float qy, const Box &b, int &ix, int &iy)
{
    ix = min(max(grid_cell(qx, g.origin[0], g.cell, g.dims[0]), b.lo[0]), b.hi[0]);
    iy = min(max(grid_cell(qy, g.origin[1], g.cell, g.dims[1]), b.lo[1]), b.hi[1]);
}

// The walk over box b's column (ix, iy).
template <int U, class F, class M>
__device__ __forceinline__ void group_walk_column(const GridView &v, const Box &b, int ix, int iy, int g, int gs, F &&f,
                                                  M &&more)
{
    const uint32_t row = ((uint32_t)ix * (uint32_t)v.g.dims[1] + (uint32_t)iy) * (uint32_t)v.g.dims[2];
    const uint32_t s0 = v.start[row + (uint32_t)b.lo[2]], s1 = v.start[row + (uint32_t)b.hi[2] + 1u];
    group_walk<U>(v.sxyzi, s1 > s0 ? s1 - s0 : 0u, g, gs, [&](uint32_t fi) { return s0 + fi; }, f, more);
}

// ---- the smallest keys ----------------------------------------------------------------------
// Searches for a threshold td with exactly `want` of m distances below it (0 < want < m, all in
// [0, r2)), given count(t), how many are below t, and next(t), the smallest at or above t.  Trials
// go to the place a uniform spread of squared distances (points on a surface) would give, every
// fourth to the middle; where one is missing, a step to the next distance itself ends the search.
// Three steps on average for 30 of 45, five for the slowest of eight groups.  An uneven spread
// takes more: from kGuesses on, steps to the next distance and halvings of the bits (non-negative
// doubles order as their bits) alternate, which bounds their number.  Returns false for a tie: td
// is then a distance that more than one has, with `below` < want of them below it and more than
// want not above.
template <class C, class N>
__device__ __forceinline__ bool find_threshold(int m, int want, double r2, double &td, int &below, C &&count, N &&next)
{
    constexpr int kGuesses = 12;
    double lo = 0.0, hi = r2;  // fewer than `want` below lo, more below hi
    int chi = m;
    below = 0;
    for (int step = 0;; ++step) {
        const long long bl = __double_as_longlong(lo), bh = __double_as_longlong(hi);
        const bool exact = step >= kGuesses ? (step & 1) == 0 : step >= 2 && want - below == 1;
        double v = lo, t;
        if (exact) {
            v = next(lo);
            t = __longlong_as_double(__double_as_longlong(v) + 1);
        } else {
            t = lo + (hi - lo) * ((step & 3) == 3 ? 0.5 : (double)((float)(want - below) / (float)(chi - below)));
            if (step >= kGuesses || !(t > lo && t < hi)) t = __longlong_as_double(bl + ((bh - bl) >> 1));
            if (!(t > lo)) continue;  // neighbours: an exact step decides
        }
        const int c = count(t);
        if (c == want) {
            td = t;
            return true;
        }
        if (c < want) {
            lo = t;
            below = c;
        } else if (exact) {
            td = v;
            return false;
        } else {
            hi = t;
            chi = c;
        }
    }
}

// A wavefront's buffer of keys: candidates within the radius, as (squared distance, original
// index) and (SLOTS) the sorted slot.
constexpr int kSelCap = 512;
constexpr int kSelPer = kSelCap / kWave;     // keys per lane
constexpr int kSelBlock = kSelCap - kWave;   // keys that one collection can keep

template <bool SLOTS>
struct SelBuf {
    double d2[kSelCap];
    int32_t idx[kSelCap];
    int32_t slot[SLOTS ? kSelCap : 1];
};

// Keeps the `want` smallest of the buffer's m keys (want < m) and sets (td, ti) so that exactly the
// kept keys are below it in (d2, index) order.  Run by a whole wavefront; every d2 is in [0, r2).
template <bool SLOTS>
__device__ __forceinline__ void wave_prune(SelBuf<SLOTS> &buf, int m, int want, double r2, double &td, int32_t &ti)
{
    const int lane = lane_id();
    double d[kSelPer];
    int32_t x[kSelPer], s[kSelPer];
#pragma unroll
    for (int j = 0; j < kSelPer; ++j) {
        const int e = lane + kWave * j;
        d[j] = e < m ? buf.d2[e] : DBL_MAX;
        x[j] = e < m ? buf.idx[e] : INT_MAX;
        s[j] = SLOTS && e < m ? buf.slot[e] : 0;
    }
    int below;
    ti = -1;  // everything below td, whatever its index
    const bool plain = find_threshold(
        m, want, r2, td, below,
        [&](double t) {
            int c = 0;
#pragma unroll
            for (int j = 0; j < kSelPer; ++j) c += __popcll(__ballot(d[j] < t));
            return c;
        },
        [&](double t) {
            double v = DBL_MAX;
#pragma unroll
            for (int j = 0; j < kSelPer; ++j) v = d[j] >= t ? fmin(v, d[j]) : v;
            for (int s = 1; s < kWave; s <<= 1) v = fmin(v, __shfl_xor(v, s, kWave));
            return v;
        });
    if (!plain) {
        // of the keys at td, those of the want - below lowest indices
        int a = -1, z = INT_MAX - 1;  // count(index <= a) < need <= count(index <= z)
        while (z - a > 1) {
            const int mid = a + (z - a) / 2;
            int c = 0;
#pragma unroll
            for (int j = 0; j < kSelPer; ++j) c += __popcll(__ballot(d[j] == td && x[j] <= mid));
            if (c < want - below) a = mid;
            else z = mid;
        }
        ti = z + 1;
    }
    int pos = 0;
    wave_lds_sync();
#pragma unroll
    for (int j = 0; j < kSelPer; ++j) {
        const bool keep = key_less(d[j], x[j], td, ti);
        const uint64_t k = __ballot(keep);
        if (keep) {
            const int e = pos + __popcll(k & ((1ull << lane) - 1ull));
            buf.d2[e] = d[j];
            buf.idx[e] = x[j];
            if (SLOTS) buf.slot[e] = s[j];
        }
        pos += __popcll(k);
    }
    wave_lds_sync();
}

// Collects into the buffer the `want` (<= kSelBlock) smallest keys after (ld, li) of the points
// within the radius of q, or all of them if fewer; returns their number.  One pass over the
// candidates whatever their number: when the buffer is nearly full only the `want` smallest stay,
// and later candidates above their threshold are dropped at once.  Run by a whole wavefront.
template <bool SLOTS>
__device__ __forceinline__ int wave_collect(const GridView &v, const Box &b, float4 q, double r2, int want, double ld,
                                            int32_t li, SelBuf<SLOTS> &buf)
{
    const int lane = lane_id();
    double td = DBL_MAX;  // keys at or above this are not among the `want` smallest
    int32_t ti = INT_MAX;
    int m = 0;
    wave_lds_sync();
    group_walk_box<4>(
        v, b, lane, kWave,
        [&](uint32_t s, float4 c, bool valid) {
            const double d2 = dist2(c.x, c.y, c.z, q.x, q.y, q.z);
            bool in = valid && d2 < r2 && d2 <= td && d2 >= ld;
            int32_t ix = 0;
            if (in) {
                ix = v.order[s];
                in = key_less(d2, ix, td, ti) && key_less(ld, li, d2, ix);
            }
            const uint64_t k = __ballot(in);
            if (in) {
                const int e = m + __popcll(k & ((1ull << lane) - 1ull));
                buf.d2[e] = d2;
                buf.idx[e] = ix;
                if (SLOTS) buf.slot[e] = (int32_t)s;
            }
            m += __popcll(k);
            if (m > kSelBlock) {  // the next 64 might not fit (m > want, too)
                wave_lds_sync();
                wave_prune(buf, m, want, r2, td, ti);
                m = want;
            }
        });
    wave_lds_sync();
    if (m > want) {
        wave_prune(buf, m, want, r2, td, ti);
        m = want;
    }
    return m;
}

}  // namespace gca
