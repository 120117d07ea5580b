// grid.hip -- uniform-grid neighbour search (K4/K5/K6) and radius outlier removal.
//
// Replaces the grid build + nn_search_functor + nn_search_radius_step1/2 +
// check_if_enough_radius_nn_functor of src/geometry/cuda_nn_search.cu:29-800.
//
// Grid build is a counting sort: count points per dense cell (atomics), exclusive scan of
// the counts, scatter (atomicSub hands out slots and leaves the counts at zero again).  The
// points are copied into cell order (sxyzi) so that neighbour scans read contiguous float4s:
// cells (ix, iy, lo_z..hi_z) are adjacent in the z-fastest linear order, so a query reads at
// most 9 contiguous runs.  The grid is built once per cloud and radius and cached, where the
// reference rebuilds it (including a sort) on every call.
//
// Results are canonical: neighbour set = { j : d2_fp64 < r^2 }, nearest = argmin (d2, index),
// K-cap = the K smallest (d2, index); so they do not depend on the order inside a cell.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <climits>

#include "gca_device.hpp"
#include "gca_internal.hpp"
#include "neighbours.hpp"

namespace gca {

struct CountArgs {
    const float4 *xyzi;
    const CloudHdr *hdr;
    GridDesc g;
    uint32_t *count, *cell_of;
};

template <int N>
__global__ __launch_bounds__(256) void k_grid_count(Jobs<CountArgs, N> J)
{
    const CountArgs &A = J.a[N == 1 ? 0 : blockIdx.y];
    const float4 *__restrict__ xyzi = A.xyzi;
    uint32_t *__restrict__ count = A.count;
    uint32_t *__restrict__ cell_of = A.cell_of;
    const GridDesc g = A.g;
    const int n = A.hdr->n;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        float4 p = xyzi[i];
        int32_t cx = grid_cell(p.x, g.origin[0], g.cell, g.dims[0]);
        int32_t cy = grid_cell(p.y, g.origin[1], g.cell, g.dims[1]);
        int32_t cz = grid_cell(p.z, g.origin[2], g.cell, g.dims[2]);
        uint32_t lin = (uint32_t)(((int64_t)cx * g.dims[1] + cy) * g.dims[2] + cz);
        cell_of[i] = lin;
        atomicAdd(&count[lin], 1u);
    }
}

struct ScatterArgs {
    const float4 *xyzi;
    const CloudHdr *hdr;
    uint32_t *count;
    const uint32_t *start, *cell_of;
    int32_t *order;
    float4 *sxyzi;
};

template <int N>
__global__ __launch_bounds__(256) void k_grid_scatter(Jobs<ScatterArgs, N> J)
{
    const ScatterArgs &A = J.a[N == 1 ? 0 : blockIdx.y];
    const float4 *__restrict__ xyzi = A.xyzi;
    uint32_t *__restrict__ count = A.count;
    const uint32_t *__restrict__ start = A.start;
    const uint32_t *__restrict__ cell_of = A.cell_of;
    int32_t *__restrict__ order = A.order;
    float4 *__restrict__ sxyzi = A.sxyzi;
    const int n = A.hdr->n;
    const int lane = lane_id();
    for (int b = blockIdx.x * blockDim.x; b < n; b += gridDim.x * blockDim.x) {  // block-uniform
        const int i = b + (int)threadIdx.x;
        const bool on = i < n;
        const uint32_t lin = on ? cell_of[i] : 0u;
        // a run of equal cells in the wavefront takes its slots with one atomic (the order of
        // points within a cell is free: every query breaks ties by original index)
        const int head = run_head(on ? (int64_t)lin : -1 - (int64_t)lane);
        const uint32_t len = run_reduce(on ? 1u : 0u, head, [](uint32_t x, uint32_t y) { return x + y; });
        uint32_t top = 0u;
        if (on && head == lane) top = atomicSub(&count[lin], len);
        top = __shfl(top, head, kWave);
        if (on) {
            const uint32_t pos = start[lin] + top - 1u - (uint32_t)(lane - head);
            order[pos] = i;
            sxyzi[pos] = xyzi[i];
        }
    }
}

void grid_free_cells(gca_ctx ctx, Grid &g, bool idle)
{
    dev_array_free(ctx, g.count, g.cap_cells, idle);
    dev_array_free(ctx, g.start, g.cap_cells + 1, idle);
    g.cap_cells = 0;
}

void grid_free_points(gca_ctx ctx, Grid &g, bool idle)
{
    dev_array_free(ctx, g.order, g.cap_pts, idle);
    dev_array_free(ctx, g.sxyzi, g.cap_pts, idle);
    dev_array_free(ctx, g.cell_of, g.cap_pts, idle);
    dev_array_free(ctx, g.snrm, g.cap_pts, idle);
    dev_array_free(ctx, g.sgrad, g.cap_pts, idle);
    g.cap_pts = 0;
}

int32_t grid_prepare(gca_ctx ctx, gca_cloud c, const GridDesc &d)
{
    Grid &G = c->grid;
    G.valid = false;
    if (G.cap_cells < d.ncells) {
        if (G.count) GCA_HIP(hipStreamSynchronize(ctx->stream));
        grid_free_cells(c->ctx, G, G.count && device_idle(c->ctx));
        int64_t want = std::min<int64_t>(kGridCellCap, d.ncells + d.ncells / 4 + 1024);
        GCA_TRY(dev_array(c->ctx, &G.count, want));
        GCA_TRY(dev_array(c->ctx, &G.start, want + 1));
        GCA_HIP(hipMemsetAsync(G.count, 0, sizeof(uint32_t) * want, ctx->stream));
        G.cap_cells = want;
    }
    if (G.cap_pts < c->cap) {
        if (G.order) GCA_HIP(hipStreamSynchronize(ctx->stream));
        grid_free_points(c->ctx, G, G.order && device_idle(c->ctx));
        GCA_TRY(dev_array(c->ctx, &G.order, c->cap));
        GCA_TRY(dev_array(c->ctx, &G.sxyzi, c->cap));
        GCA_TRY(dev_array(c->ctx, &G.cell_of, c->cap));
        G.cap_pts = c->cap;
    }
    return GCA_OK;
}

int32_t launch_grid_build(gca_ctx ctx, gca_cloud c, const GridDesc &d, bool counted)
{
    Grid &G = c->grid;
    GCA_TRY(grid_prepare(ctx, c, d));
    const unsigned nb = (unsigned)std::min<int64_t>(4096, std::max<int64_t>(1, (c->cap + 255) / 256));
    StageTimer timer(ctx, GCA_STAGE_GRID);
    if (!counted) {
        const Jobs<CountArgs, 1> ct{{{c->xyzi, c->hdr, d, G.count, G.cell_of}}};
        hipLaunchKernelGGL(k_grid_count<1>, dim3(nb), dim3(256), 0, ctx->stream, ct);
        GCA_HIP(hipGetLastError());
    }
    GCA_TRY(exclusive_scan_u32(ctx, G.count, G.start, d.ncells, nullptr));
    const Jobs<ScatterArgs, 1> sc{{{c->xyzi, c->hdr, G.count, G.start, G.cell_of, G.order, G.sxyzi}}};
    hipLaunchKernelGGL(k_grid_scatter<1>, dim3(nb), dim3(256), 0, ctx->stream, sc);
    GCA_HIP(hipGetLastError());
    G.desc = d;
    G.valid = true;
    G.attrs_valid = false;
    return GCA_OK;
}

int32_t launch_grid_levels(gca_ctx launch, const gca_ctx *ctxs, const gca_cloud *cs, const GridDesc *ds, int nj,
                           bool counted)
{
    if (nj < 1 || nj > kMaxJobs) return GCA_ERR_INVALID_VALUE;
    bool wide = false;
    for (int j = 0; j < nj; ++j) {
        GCA_TRY(grid_prepare(ctxs[j], cs[j], ds[j]));
        wide = wide || scan_wide(ds[j].ncells);
    }
    ScanJob scans[kMaxJobs];
    Jobs<CountArgs, kMaxJobs> ct{};
    Jobs<ScatterArgs, kMaxJobs> sc{};
    unsigned nb = 1;
    for (int j = 0; j < nj; ++j) {
        const Grid &G = cs[j]->grid;
        int lane = 0;  // a lane of its ctx's scratch each
        for (int k = 0; k < j; ++k) lane += ctxs[k] == ctxs[j];
        GCA_TRY(scan_job(ctxs[j], G.count, G.start, ds[j].ncells, nullptr, wide, &scans[j], lane));
        ct.a[j] = CountArgs{cs[j]->xyzi, cs[j]->hdr, ds[j], G.count, G.cell_of};
        sc.a[j] = ScatterArgs{cs[j]->xyzi, cs[j]->hdr, G.count, G.start, G.cell_of, G.order, G.sxyzi};
        nb = std::max(nb, (unsigned)std::min<int64_t>(4096, std::max<int64_t>(1, (cs[j]->cap + 255) / 256)));
    }
    {
        StageTimer timer(launch, GCA_STAGE_GRID);
        if (!counted) hipLaunchKernelGGL(k_grid_count<kMaxJobs>, dim3(nb, (unsigned)nj), dim3(256), 0, launch->stream, ct);
        GCA_TRY(scan_launch(launch->stream, scans, nj, false, wide));
        hipLaunchKernelGGL(k_grid_scatter<kMaxJobs>, dim3(nb, (unsigned)nj), dim3(256), 0, launch->stream, sc);
        GCA_HIP(hipGetLastError());
    }
    for (int j = 0; j < nj; ++j) {
        Grid &G = cs[j]->grid;
        G.desc = ds[j];
        G.valid = true;
        G.attrs_valid = false;
    }
    return GCA_OK;
}

__global__ __launch_bounds__(256) void k_gather_sorted(const CloudHdr *__restrict__ hdr,
                                                       const int32_t *__restrict__ order,
                                                       const float4 *__restrict__ nrm,
                                                       const float4 *__restrict__ grad,
                                                       float4 *__restrict__ snrm, float4 *__restrict__ sgrad)
{
    const int n = hdr->n;
    for (int s = blockIdx.x * blockDim.x + threadIdx.x; s < n; s += gridDim.x * blockDim.x) {
        const int32_t j = order[s];
        snrm[s] = nrm[j];
        sgrad[s] = grad[j];
    }
}

// The grid's copies of normals and gradients: a call that gets only the first leaves it for the next one.
int32_t grid_alloc_attributes(gca_cloud c)
{
    Grid &G = c->grid;
    if (!G.snrm) GCA_TRY(dev_array(c->ctx, &G.snrm, G.cap_pts));
    if (!G.sgrad) GCA_TRY(dev_array(c->ctx, &G.sgrad, G.cap_pts));
    return GCA_OK;
}

int32_t grid_gather_attributes(gca_ctx ctx, gca_cloud c)
{
    Grid &G = c->grid;
    if (!G.valid) return GCA_ERR_NOT_READY;
    if (G.attrs_valid) return GCA_OK;
    GCA_TRY(grid_alloc_attributes(c));
    const unsigned nb = (unsigned)std::min<int64_t>(4096, std::max<int64_t>(1, (c->cap + 255) / 256));
    hipLaunchKernelGGL(k_gather_sorted, dim3(nb), dim3(256), 0, ctx->stream, c->hdr, G.order, c->nrm, c->grad,
                       G.snrm, G.sgrad);
    GCA_HIP(hipGetLastError());
    G.attrs_valid = true;
    return GCA_OK;
}

// ---- queries ---------------------------------------------------------------------------------

constexpr int kQUnroll = 4;  // candidates in flight per lane

// Points within the radius of q, counted by a group of lanes (the count is on all of them); the
// walk begins with the query's own column, where most of them are, and ends once the count
// exceeds `limit`.
__device__ __forceinline__ uint32_t group_count(const GridView &v, float4 q, int g, int gs, uint32_t limit)
{
    Box b;
    int ix, iy;
    if (!grid_range(v.g, q.x, q.y, q.z, b.lo, b.hi)) return 0;
    const double r2 = (double)v.g.radius * (double)v.g.radius;
    uint32_t k = 0, all = 0;
    auto test = [&](uint32_t, float4 c, bool valid) {
        k += valid && dist2(c.x, c.y, c.z, q.x, q.y, q.z) < r2 ? 1u : 0u;
    };
    auto sum = [&]() {
        all = k;
        for (int m = 1; m < gs; m <<= 1) all += __shfl_xor(all, m, kWave);
        return all <= limit;
    };
    own_column(v.g, q.x, q.y, b, ix, iy);
    group_walk_column<kQUnroll>(v, b, ix, iy, g, gs, test, sum);
    if (all <= limit) group_walk_box<kQUnroll>(v, b, g, gs, ix, iy, test, sum);
    return all;
}

// ---- nearest neighbour ----------------------------------------------------------------------
// kNnLanes lanes per query.  The query's own column of cells is searched first; the distance found
// there bounds the box of the rest, which for clouds that overlap is a few cells instead of 27
// (kBoxRel / kBoxAbs cover the rounding of the distance and of the cell arithmetic, so the box
// holds every point at most that far away: the result is that of the full search).
// Bound by the candidates' load latency.  92k queries on 92k points of a 424x240 frame, 3 cm: 45 us
// (66 with each candidate's load waited for by itself and its index loaded at once);
// 359 us with one thread per query over the whole box.
constexpr int kNnLanes = 8;
constexpr double kBoxRel = 1e-9, kBoxAbs = 1e-9;

__global__ __launch_bounds__(256) void k_nn(const float4 *__restrict__ q, const CloudHdr *__restrict__ qh,
                                            GridDesc g, const uint32_t *__restrict__ start,
                                            const int32_t *__restrict__ order, const float4 *__restrict__ sxyzi,
                                            int32_t *__restrict__ out)
{
    const GridView v = make_view(g, start, order, sxyzi);
    const int n = qh->n;
    const int gl = (int)threadIdx.x & (kNnLanes - 1);
    const double r2 = (double)g.radius * (double)g.radius;
    for (int i = (int)((blockIdx.x * blockDim.x + threadIdx.x) / kNnLanes); i < n;
         i += (int)(gridDim.x * blockDim.x / kNnLanes)) {
        const float4 p = q[i];
        double bd = DBL_MAX;
        int32_t bs = -1;  // slot; the original indices are compared (and loaded) only for ties
        auto better = [&](double d2, int32_t slot) {
            if (d2 < bd || (d2 == bd && slot != bs && order[slot] < order[bs])) {
                bd = d2;
                bs = slot;
            }
        };
        auto test = [&](uint32_t s, float4 c, bool valid) {
            const double d2 = dist2(c.x, c.y, c.z, p.x, p.y, p.z);
            if (valid && d2 < r2) better(d2, (int32_t)s);
        };
        auto reduce = [&]() {
            for (int m = 1; m < kNnLanes; m <<= 1) {
                const double od = __shfl_xor(bd, m, kWave);
                const int32_t os = __shfl_xor(bs, m, kWave);
                if (os >= 0) better(od, os);
            }
        };
        auto go = [] { return true; };
        Box b;
        int ix, iy;
        if (grid_range(g, p.x, p.y, p.z, b.lo, b.hi)) {
            own_column(g, p.x, p.y, b, ix, iy);
            group_walk_column<kQUnroll>(v, b, ix, iy, gl, kNnLanes, test, go);
            reduce();
            // the column was searched over the full box's cells, a superset of what is left of it
            if (bs < 0 || grid_range_r(g, p.x, p.y, p.z, fmin((double)g.radius, sqrt(bd) * (1.0 + kBoxRel) + kBoxAbs),
                                       b.lo, b.hi)) {
                group_walk_box<kQUnroll>(v, b, gl, kNnLanes, ix, iy, test, go);
                reduce();
            }
        }
        if (gl == 0) out[i] = bs >= 0 ? order[bs] : -1;
    }
}

// Launch width for `items` queries of `lanes` lanes in 256-thread workgroups.
static unsigned group_blocks(int64_t items, int lanes)
{
    return (unsigned)std::min<int64_t>(65536, std::max<int64_t>(1, (items * lanes + 255) / 256));
}

int32_t launch_nn(gca_ctx ctx, gca_cloud q, gca_cloud ref, float radius, int32_t *out)
{
    const Grid &G = ref->grid;
    hipLaunchKernelGGL(k_nn, dim3(group_blocks(q->cap, kNnLanes)), dim3(256), 0, ctx->stream, q->xyzi, q->hdr,
                       query_desc(G, radius), G.start, G.order, G.sxyzi, out);
    GCA_HIP(hipGetLastError());
    return GCA_OK;
}

// ---- radius search ------------------------------------------------------------------------
// Two kernels: the count per query (capped at max_nn), whose scan gives the offsets, and the fill,
// one wavefront per query, which writes each query's list in (d2, index) order straight to its
// place.

constexpr int kCountLanes = 16;

__global__ __launch_bounds__(256) void k_radius_count(const float4 *__restrict__ q,
                                                      const CloudHdr *__restrict__ qh, GridDesc g,
                                                      const uint32_t *__restrict__ start,
                                                      const float4 *__restrict__ sxyzi, uint32_t max_nn,
                                                      uint32_t *__restrict__ cnt)
{
    const GridView v = make_view(g, start, nullptr, sxyzi);
    const int n = qh->n;
    const int gl = (int)threadIdx.x & (kCountLanes - 1);
    for (int i = (int)((blockIdx.x * blockDim.x + threadIdx.x) / kCountLanes); i < n;
         i += (int)(gridDim.x * blockDim.x / kCountLanes)) {
        const uint32_t k = group_count(v, q[i], gl, kCountLanes, max_nn ? max_nn - 1u : UINT_MAX);
        if (gl == 0) cnt[i] = max_nn ? min(k, max_nn) : k;
    }
}

// The fill collects a query's keys in LDS (wave_collect): one pass over the candidates whatever
// their number, where an insertion sort in global memory grew with the square of the neighbourhood
// (11k queries of a 424x240 frame, 3 cm, 30 nearest: 66 us, 134 ms before; the counts 10 us with 16
// lanes per query, 364 us with one).  A list longer than the buffer comes out in blocks of
// kSelBlock, each pass taking the keys after the last one written.
constexpr int kFillWaves = 4;
constexpr int kFillRank = 2 * kWave;  // up to here lists are ordered by counting ranks

// Writes the buffer's m keys' indices to out in (d2, index) order; the last key goes to (ld, li).
__device__ __forceinline__ void fill_write(SelBuf<false> &buf, int m, int32_t *__restrict__ out, double &ld, int32_t &li)
{
    const int lane = lane_id();
    if (m <= kFillRank) {
        const int e1 = lane + kWave;
        const double d0 = lane < m ? buf.d2[lane] : DBL_MAX, d1 = e1 < m ? buf.d2[e1] : DBL_MAX;
        const int32_t x0 = lane < m ? buf.idx[lane] : INT_MAX, x1 = e1 < m ? buf.idx[e1] : INT_MAX;
        int r0 = 0, r1 = 0;
        for (int j = 0; j < m; ++j) {
            const double dj = buf.d2[j];
            const int32_t xj = buf.idx[j];
            r0 += key_less(dj, xj, d0, x0) ? 1 : 0;
            r1 += key_less(dj, xj, d1, x1) ? 1 : 0;
        }
        if (lane < m) out[r0] = x0;
        if (e1 < m) out[r1] = x1;
        return;  // only a list's last block is this short
    }
    int n2 = kFillRank;
    while (n2 < m) n2 *= 2;
    for (int e = m + lane; e < n2; e += kWave) {
        buf.d2[e] = DBL_MAX;
        buf.idx[e] = INT_MAX;
    }
    wave_lds_sync();
    for (int k = 2; k <= n2; k *= 2)  // bitonic
        for (int j = k / 2; j > 0; j /= 2) {
            for (int t = lane; t < n2 / 2; t += kWave) {
                const int a = 2 * t - (t & (j - 1)), b = a + j;
                const double da = buf.d2[a], db = buf.d2[b];
                const int32_t xa = buf.idx[a], xb = buf.idx[b];
                if (key_less(db, xb, da, xa) == ((a & k) == 0)) {
                    buf.d2[a] = db;
                    buf.d2[b] = da;
                    buf.idx[a] = xb;
                    buf.idx[b] = xa;
                }
            }
            wave_lds_sync();
        }
    for (int e = lane; e < m; e += kWave) out[e] = buf.idx[e];
    ld = buf.d2[m - 1];
    li = buf.idx[m - 1];
}

__global__ __launch_bounds__(kWave *kFillWaves) void k_radius_fill(const float4 *__restrict__ q, int n, GridDesc g,
                                                                   const uint32_t *__restrict__ start,
                                                                   const int32_t *__restrict__ order,
                                                                   const float4 *__restrict__ sxyzi,
                                                                   const uint32_t *__restrict__ off,
                                                                   int32_t *__restrict__ out)
{
    __shared__ SelBuf<false> bufs[kFillWaves];
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
    SelBuf<false> &buf = bufs[w];
    const GridView v = make_view(g, start, order, sxyzi);
    const double r2 = (double)g.radius * (double)g.radius;
    for (int i = (int)blockIdx.x * kFillWaves + w; i < n; i += (int)gridDim.x * kFillWaves) {
        const uint32_t first = off[i];
        const int total = (int)(off[i + 1] - first);
        const float4 p = q[i];
        Box b;
        if (total == 0 || !grid_range(g, p.x, p.y, p.z, b.lo, b.hi)) continue;
        double ld = -1.0;  // the last key written
        int32_t li = -1;
        for (int done = 0; done < total;) {
            const int want = min(total - done, kSelBlock);
            const int m = wave_collect(v, b, p, r2, want, ld, li, buf);
            fill_write(buf, m, out + first + done, ld, li);
            done += want;
        }
    }
}

int32_t launch_radius(gca_ctx ctx, gca_cloud q, gca_cloud ref, float radius, int32_t max_nn, int32_t *offsets,
                      int32_t *idx, int64_t idx_cap, int64_t *total)
{
    GCA_TRY(cloud_sync_header(q));
    const int64_t nq = q->host_hdr.n;
    const Grid &G = ref->grid;
    const GridDesc d = query_desc(G, radius);
    uint32_t *cnt = (uint32_t *)ctx_scratch(ctx, 8, sizeof(uint32_t) * (nq + 1), false);
    uint32_t *tot_dev = (uint32_t *)ctx_scratch(ctx, 10, sizeof(uint32_t) * 4, false);
    if (!cnt || !tot_dev) return GCA_ERR_OUT_OF_MEMORY;
    hipLaunchKernelGGL(k_radius_count, dim3(group_blocks(nq, kCountLanes)), dim3(256), 0, ctx->stream, q->xyzi, q->hdr,
                       d, G.start, G.sxyzi, (uint32_t)max_nn, cnt);
    GCA_HIP(hipGetLastError());
    GCA_TRY(exclusive_scan_u32(ctx, cnt, (uint32_t *)offsets, nq, tot_dev));
    GCA_HIP(hipMemcpyAsync(ctx->pinned, tot_dev, sizeof(uint32_t), hipMemcpyDeviceToHost, ctx->stream));
    GCA_HIP(hipStreamSynchronize(ctx->stream));
    const uint32_t capped = *(const uint32_t *)ctx->pinned;
    *total = capped;
    if (!idx) return GCA_OK;  // count-only query
    if ((int64_t)capped > idx_cap) return GCA_ERR_INVALID_VALUE;
    hipLaunchKernelGGL(k_radius_fill, dim3(group_blocks(nq, kWave)), dim3(kWave * kFillWaves), 0, ctx->stream, q->xyzi,
                       (int)nq, d, G.start, G.order, G.sxyzi, (const uint32_t *)offsets, idx);
    GCA_HIP(hipGetLastError());
    return GCA_OK;
}

// ---- cell binning (exposed for parity checks) --------------------------------------------

__global__ __launch_bounds__(256) void k_cells(const float4 *__restrict__ xyzi, const CloudHdr *__restrict__ h,
                                               GridDesc g, int32_t *__restrict__ cells)
{
    const int n = h->n;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        float4 p = xyzi[i];
        cells[3 * i] = grid_cell(p.x, g.origin[0], g.cell, g.dims[0]);
        cells[3 * i + 1] = grid_cell(p.y, g.origin[1], g.cell, g.dims[1]);
        cells[3 * i + 2] = grid_cell(p.z, g.origin[2], g.cell, g.dims[2]);
    }
}

int32_t launch_grid_cells(gca_ctx ctx, gca_cloud c, int32_t *cells)
{
    const unsigned nb = (unsigned)std::min<int64_t>(4096, std::max<int64_t>(1, (c->cap + 255) / 256));
    hipLaunchKernelGGL(k_cells, dim3(nb), dim3(256), 0, ctx->stream, c->xyzi, c->hdr, c->grid.desc, cells);
    GCA_HIP(hipGetLastError());
    return GCA_OK;
}

// ---- radius outlier removal (cuda_nn_search.cu:416-542,725-800) ---------------------------
// keep iff (# points within radius, itself included) > min_nn; stable compaction.

// A 1024-thread workgroup flags the 256 points of one compaction block, kOutLanes lanes per point.
// A point in a dense place is settled by its own column's first candidates, so the lanes' loads in
// flight are what counts (92k points, 3 cm: 20 us, 161 us with one thread per point).
constexpr int kOutBlock = 1024;
constexpr int kOutLanes = 8;

__global__ __launch_bounds__(kOutBlock) void k_outlier_flag(const float4 *__restrict__ xyzi,
                                                            const CloudHdr *__restrict__ h, GridDesc g,
                                                            const uint32_t *__restrict__ start,
                                                            const float4 *__restrict__ sxyzi, int32_t min_nn,
                                                            uint8_t *__restrict__ keep, uint32_t *__restrict__ bcnt)
{
    __shared__ uint32_t total;
    const GridView v = make_view(g, start, nullptr, sxyzi);
    const int n = h->n;
    const int gl = (int)threadIdx.x & (kOutLanes - 1);
    if (threadIdx.x == 0) total = 0u;
    __syncthreads();
    uint32_t kept = 0;
    for (int t = (int)threadIdx.x / kOutLanes; t < 256; t += kOutBlock / kOutLanes) {
        const int i = (int)blockIdx.x * 256 + t;
        if (i >= n) break;  // whole groups leave together
        const bool k = min_nn < 0 || group_count(v, xyzi[i], gl, kOutLanes, (uint32_t)min_nn) > (uint32_t)min_nn;
        if (gl == 0) {
            keep[i] = k ? 1 : 0;
            kept += k ? 1u : 0u;
        }
    }
    if (kept) atomicAdd(&total, kept);
    __syncthreads();
    if (threadIdx.x == 0) bcnt[blockIdx.x] = total;
}

__global__ __launch_bounds__(256) void k_outlier_compact(const float4 *__restrict__ xyzi,
                                                         const float4 *__restrict__ rgb,
                                                         const CloudHdr *__restrict__ h,
                                                         const uint8_t *__restrict__ keep,
                                                         const uint32_t *__restrict__ boff,
                                                         float4 *__restrict__ oxyzi, float4 *__restrict__ orgb)
{
    __shared__ uint32_t wo[4];
    const int n = h->n;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    bool k = i < n && keep[i];
    uint64_t m = __ballot(k);
    const int w = threadIdx.x / kWave;
    if (lane_id() == 0) wo[w] = (uint32_t)__popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t a = wo[0], b = wo[1], c = wo[2];
        wo[0] = 0;
        wo[1] = a;
        wo[2] = a + b;
        wo[3] = a + b + c;
    }
    __syncthreads();
    if (k) {
        uint32_t dst = boff[blockIdx.x] + wo[w] + (uint32_t)__popcll(m & ((1ull << lane_id()) - 1ull));
        oxyzi[dst] = xyzi[i];
        orgb[dst] = rgb[i];
    }
}

int32_t launch_outlier(gca_ctx ctx, gca_cloud in, float radius, int32_t min_nn, gca_cloud out)
{
    GCA_TRY(cloud_reserve(out, in->cap));
    Grid G = in->grid;
    G.desc.radius = radius;
    const int64_t nblk = std::max<int64_t>(1, (in->cap + 255) / 256);
    uint8_t *keep = (uint8_t *)ctx_scratch(ctx, 2, (size_t)in->cap, false);
    uint32_t *bcnt = (uint32_t *)ctx_scratch(ctx, 3, sizeof(uint32_t) * (nblk + 1), false);
    uint32_t *boff = (uint32_t *)ctx_scratch(ctx, 4, sizeof(uint32_t) * (nblk + 1), false);
    if (!keep || !bcnt || !boff) return GCA_ERR_OUT_OF_MEMORY;
    hipLaunchKernelGGL(k_outlier_flag, dim3((unsigned)nblk), dim3(kOutBlock), 0, ctx->stream, in->xyzi, in->hdr, G.desc,
                       G.start, G.sxyzi, min_nn, keep, bcnt);
    GCA_HIP(hipGetLastError());
    GCA_TRY(exclusive_scan_u32(ctx, bcnt, boff, nblk, (uint32_t *)&out->hdr->n));
    hipLaunchKernelGGL(k_outlier_compact, dim3((unsigned)nblk), dim3(256), 0, ctx->stream, in->xyzi, in->rgb,
                       in->hdr, keep, boff, out->xyzi, out->rgb);
    GCA_HIP(hipGetLastError());
    GCA_TRY(launch_bounds(ctx, out));
    return GCA_OK;
}

}  // namespace gca
