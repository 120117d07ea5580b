// normals.hip -- PCA normals and colour gradient: neighbourhood moments, then per-point solves.
//
// Replaces cuda_estimate_normals (src/geometry/cuda_estimate_normals.cu:22-199) and
// cuda_compute_color_gradient (src/registration/cuda_compute_color_gradient.cu:13-127).
//
// The reference materialises every (query, neighbour) pair, reduces 36-byte raw-moment
// records by key in FP32 and solves the 3x3 eigenproblem with an FP32 trigonometric closed
// form.  Here a group of eight lanes walks the query's grid runs (all run bounds loaded first,
// then one flattened candidate walk), and the neighbourhood sums are accumulated in 2^-40 fixed
// point scaled by the radius, centred on the query point: integer adds are exact, so the order of
// the reduction does not change the result, which equals the FP64 oracle's.  The colour gradient's sums are the raw ones (sum u u^T, sum u dI); its
// tangent projection is applied to the sums in the solve, so they need no normal and can be
// gathered in the same walk as the normals' when the gradient radius is the smaller one.  Where
// the K nearest are wanted the walk keeps the in-radius candidates in LDS and a threshold with
// exactly K of them below it is bisected by the group; the few queries with more candidates than
// fit there are finished by one wavefront each.  The covariance is then diagonalised per point with
// a cyclic Jacobi iteration in FP64 (only +, -, *, /, sqrt: identical on host and device).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <climits>

#include "gca_device.hpp"
#include "gca_internal.hpp"
#include "neighbours.hpp"

namespace gca {

// Cyclic Jacobi for a symmetric 3x3 (same operation sequence as the oracle's orc_eigen3).
__host__ __device__ inline void jacobi3(double A[3][3], double v[3][3])
{
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) v[i][j] = (i == j) ? 1.0 : 0.0;
    for (int sweep = 0; sweep < 32; ++sweep) {
        double off = (A[0][1] * A[0][1] + A[0][2] * A[0][2]) + A[1][2] * A[1][2];
        double dg = (A[0][0] * A[0][0] + A[1][1] * A[1][1]) + A[2][2] * A[2][2];
        if (!(off > 1e-36 * dg)) break;
        for (int r = 0; r < 3; ++r) {
            const int p = r == 2 ? 1 : 0;
            const int q = r == 0 ? 1 : 2;
            double apq = A[p][q];
            if (apq == 0.0) continue;
            double theta = (A[q][q] - A[p][p]) / (2.0 * apq);
            double t = 1.0 / (fabs(theta) + sqrt(theta * theta + 1.0));
            if (theta < 0.0) t = -t;
            double c = 1.0 / sqrt(t * t + 1.0), s = t * c;
            for (int k = 0; k < 3; ++k) {
                double akp = A[k][p], akq = A[k][q];
                A[k][p] = c * akp - s * akq;
                A[k][q] = s * akp + c * akq;
            }
            for (int k = 0; k < 3; ++k) {
                double apk = A[p][k], aqk = A[q][k];
                A[p][k] = c * apk - s * aqk;
                A[q][k] = s * apk + c * aqk;
            }
            A[p][q] = 0.0;
            A[q][p] = 0.0;
            for (int k = 0; k < 3; ++k) {
                double vkp = v[k][p], vkq = v[k][q];
                v[k][p] = c * vkp - s * vkq;
                v[k][q] = s * vkp + c * vkq;
            }
        }
    }
}

__host__ __device__ inline float4 normal_from_moments(int32_t cnt, const long long S[9])
{
    float4 out = make_float4(0.f, 0.f, 0.f, 0.f);
    if (cnt < 3) return out;  // cuda_estimate_normals.cu:89-93
    const double n = (double)cnt;
    double m[3], A[3][3], V[3][3];
    for (int a = 0; a < 3; ++a) m[a] = ((double)S[a] / kFx40) / n;
    const int IA[6] = {0, 0, 0, 1, 1, 2}, IB[6] = {0, 1, 2, 1, 2, 2};
    for (int k = 0; k < 6; ++k) {
        double c = ((double)S[3 + k] / kFx40) / n - m[IA[k]] * m[IB[k]];
        A[IA[k]][IB[k]] = c;
        A[IB[k]][IA[k]] = c;
    }
    jacobi3(A, V);
    const double e0 = A[0][0], e1 = A[1][1], e2 = A[2][2];
    int sel;  // strict-< selection (cuda_estimate_normals.cu:116-125)
    if (e0 < e1 && e0 < e2) sel = 0;
    else if (e1 < e0 && e1 < e2) sel = 1;
    else sel = 2;
    double v[3] = {V[0][sel], V[1][sel], V[2][sel]};
    double len = sqrt((v[0] * v[0] + v[1] * v[1]) + v[2] * v[2]);
    if (!(len > 0.0)) return out;
    for (int a = 0; a < 3; ++a) v[a] /= len;
    if (-v[2] < 0.0)  // orient toward (0,0,-1) (cuda_estimate_normals.cu:131-151)
        for (int a = 0; a < 3; ++a) v[a] = -v[a];
    out.x = (float)v[0];
    out.y = (float)v[1];
    out.z = (float)v[2];
    return out;
}

// ---- neighbourhood sums ----------------------------------------------------------------------
constexpr int kNbBlock = 256;
constexpr int kNbLanes = 8;     // lanes per query
constexpr int kNbUnroll = 2;    // candidates in flight per lane
constexpr int kOvfWaves = 4;    // wavefronts per workgroup of the overflow kernel

struct Moments {
    long long S[9];
    int32_t cnt;
    int32_t pad;
};

// Neighbourhood sums (2^-40 fixed point) of the neighbours p of a query q, u = (p - q) / r:
//   KIND 0, normals:  sum u, sum u u^T (xx xy xz yy yz zz)
//   KIND 1, gradient: sum u u^T, sum u dI with dI = I_p - I_q (raw: the projection onto the query's
//                     tangent plane is applied to the sums, gradient_from_moments)
// The query itself contributes exactly zero to every sum (and one to the count).
// |u_a| <= 1 (to rounding), so the u and u u^T terms are integers up to 2^40, rounded to nearest
// even by one instruction, and sums of up to kExactTerms of them are exact in FP64: two operations
// a term, where the 64-bit integer path takes five.  The scale 2^40 is applied as 2^20 per factor:
// powers of two, so every rounding is that of the plain expressions.  The u dI terms have no such
// bound and use the general conversion and integer sums; so do all terms of larger neighbourhoods.
constexpr double kFx20 = 1048576.0;
constexpr int32_t kExactTerms = 4096;

template <int KIND>
struct MomentSum {
    static constexpr int ND = KIND == 0 ? 9 : 6;  // terms bounded by 2^40
    double d[ND];
    long long x[9 - ND + 1];  // the u dI terms
    __device__ __forceinline__ void zero()
    {
#pragma unroll
        for (int k = 0; k < ND; ++k) d[k] = 0.0;
#pragma unroll
        for (int k = 0; k < 9 - ND; ++k) x[k] = 0;
    }
    // inv: 2^20 / radius
    __device__ __forceinline__ void add(float4 q, float px, float py, float pz, float pw, double inv)
    {
        const double w0 = ((double)px - (double)q.x) * inv;
        const double w1 = ((double)py - (double)q.y) * inv;
        const double w2 = ((double)pz - (double)q.z) * inv;
        int k = 0;
        if constexpr (KIND == 0) {
            d[0] += __builtin_rint(w0 * kFx20);
            d[1] += __builtin_rint(w1 * kFx20);
            d[2] += __builtin_rint(w2 * kFx20);
            k = 3;
        }
        d[k] += __builtin_rint(w0 * w0);
        d[k + 1] += __builtin_rint(w0 * w1);
        d[k + 2] += __builtin_rint(w0 * w2);
        d[k + 3] += __builtin_rint(w1 * w1);
        d[k + 4] += __builtin_rint(w1 * w2);
        d[k + 5] += __builtin_rint(w2 * w2);
        if constexpr (KIND == 1) {
            const double dI = (double)pw - (double)q.w;
            x[0] += fx((w0 * dI) * kFx20);
            x[1] += fx((w1 * dI) * kFx20);
            x[2] += fx((w2 * dI) * kFx20);
        }
    }
    // The sums as integers.
    __device__ __forceinline__ void take(long long S[9]) const
    {
#pragma unroll
        for (int k = 0; k < ND; ++k) S[k] = (long long)d[k];
#pragma unroll
        for (int k = ND; k < 9; ++k) S[k] = x[k - ND];
    }
};

// The sums over all neighbours within the radius (no K cap) by the gs lanes of a group: the lane's
// part; returns its part of the count.
template <int KIND>
__device__ __forceinline__ int32_t walk_moments(const GridView &v, const Box &b, float4 q, int gl, int gs, double r2,
                                                double inv, MomentSum<KIND> &A)
{
    A.zero();
    int32_t cnt = 0;
    group_walk_box<kNbUnroll>(
        v, b, gl, gs,
        [&](uint32_t, float4 c, bool valid) {
            if (valid && dist2(c.x, c.y, c.z, q.x, q.y, q.z) < r2) {
                A.add(q, c.x, c.y, c.z, c.w, inv);
                ++cnt;
            }
        });
    return cnt;
}

// The same with integer sums, for neighbourhoods beyond kExactTerms: term by term.
template <int KIND>
__device__ __forceinline__ void walk_moments_wide(const GridView &v, const Box &b, float4 q, int gl, int gs, double r2,
                                                  double inv, long long S[9])
{
#pragma unroll
    for (int k = 0; k < 9; ++k) S[k] = 0;
    group_walk_box<1>(
        v, b, gl, gs,
        [&](uint32_t, float4 c, bool valid) {
            if (valid && dist2(c.x, c.y, c.z, q.x, q.y, q.z) < r2) {
                MomentSum<KIND> A;
                long long t[9];
                A.zero();
                A.add(q, c.x, c.y, c.z, c.w, inv);
                A.take(t);
#pragma unroll
                for (int k = 0; k < 9; ++k) S[k] += t[k];
            }
        });
}

// The wavefront's sums and a count, stored by its first lane.
__device__ __forceinline__ void wave_store(long long S[9], int32_t cnt, Moments &M)
{
#pragma unroll
    for (int c = 0; c < 9; ++c) S[c] = wave_sum(S[c]);
    if (lane_id() != 0) return;
#pragma unroll
    for (int c = 0; c < 9; ++c) M.S[c] = S[c];
    M.cnt = cnt;
}

// The group's sums and a count, stored by its first lane.
template <int KIND>
__device__ __forceinline__ void group_store(MomentSum<KIND> &A, int32_t cnt, int gl, Moments &M)
{
    constexpr int ND = MomentSum<KIND>::ND;
#pragma unroll
    for (int k = 0; k < ND; ++k) A.d[k] = group_sum<kNbLanes>(A.d[k]);
#pragma unroll
    for (int k = 0; k < 9 - ND; ++k) A.x[k] = group_sum<kNbLanes>(A.x[k]);
    if (gl != 0) return;
#pragma unroll
    for (int k = 0; k < ND; ++k) M.S[k] = (long long)A.d[k];
#pragma unroll
    for (int k = ND; k < 9; ++k) M.S[k] = A.x[k - ND];
    M.cnt = cnt;
}

// Sums without a K cap, or with one that the buffer of k_moments_sel does not reach (K >= kSelCandidates:
// it selects nothing then, and sends every larger neighbourhood to a wavefront of its own): queries with
// more than K neighbours go to the overflow list.  100k points of a surface, 200 neighbours each, K 500:
// 304 us, 756 by k_moments_sel.  24 us for the gradient of 110k points at 2 cm (30 us with 64-bit integer
// sums and a division per cell bound).  Eight lanes per query: 4 and 16 measured 1-2 % and 5 %
// slower on a 640x480 target at 1 cm, 2 and 4 % on the overlapped odometry of such frames.
template <int KIND>
__global__ __launch_bounds__(kNbBlock) void k_moments(const float4 *__restrict__ xyzi, const CloudHdr *__restrict__ hdr,
                                                      GridDesc g, const uint32_t *__restrict__ start,
                                                      const float4 *__restrict__ sxyzi, Moments *__restrict__ mom, int32_t K,
                                                      int32_t *__restrict__ ovf, uint32_t *__restrict__ ovf_n)
{
    const GridView v = make_view(g, start, nullptr, sxyzi);
    const int n = hdr->n;
    const int gl = (int)threadIdx.x & (kNbLanes - 1);
    const double r2 = (double)g.radius * (double)g.radius;
    const double inv = kFx20 * (1.0 / (double)g.radius);
    for (int i = (int)(blockIdx.x * kNbBlock + threadIdx.x) / kNbLanes; i < n; i += (int)(gridDim.x * kNbBlock) / kNbLanes) {
        const float4 q = xyzi[i];
        MomentSum<KIND> A;
        Box b;
        int32_t cnt = 0;
        A.zero();
        if (grid_range(g, q.x, q.y, q.z, b.lo, b.hi)) cnt = walk_moments<KIND>(v, b, q, gl, kNbLanes, r2, inv, A);
        cnt = (int32_t)group_sum<kNbLanes>((uint32_t)cnt);
        if (K > 0 && cnt > K) {
            if (gl == 0) ovf[atomicAdd(ovf_n, 1u)] = i;
        } else if (cnt <= kExactTerms) {
            group_store<KIND>(A, cnt, gl, mom[i]);
        } else {
            long long S[9];
            walk_moments_wide<KIND>(v, b, q, gl, kNbLanes, r2, inv, S);
#pragma unroll
            for (int k = 0; k < 9; ++k) S[k] = group_sum<kNbLanes>(S[k]);
            if (gl == 0) {
                Moments &M = mom[i];
#pragma unroll
                for (int k = 0; k < 9; ++k) M.S[k] = S[k];
                M.cnt = cnt;
            }
        }
    }
}

// Sums over the K > 0 nearest neighbours within the radius (KIND), and with PAIR (KIND 0) also the
// colour gradient's over all neighbours within rg <= the radius, from one walk.
//   1. the walk puts the in-radius candidates into the group's part of LDS, packed;
//   2. if there are more than K, the group bisects a threshold with exactly K distances below it:
//      each lane counts among its own candidates (in registers), the counts are added across the
//      group by data-parallel moves;
//   3. every lane adds its selected candidates: packed, so the lanes are busy, where adding in the
//      walk runs at the share of candidates that are in the radius (about a third).
// Ties at the threshold are settled by index.  A query with more than kSelCandidates in-radius
// candidates goes to the overflow list.  Bound half by instruction issue (the walk's tests), half by
// the latency of the cell bounds and candidates.  110k points of a raw 640x480 frame at 1 cm, the 30
// nearest of about 50 within 2.5 cm: 31 us and 5 us for the (empty) overflow launch, where adding in
// the walk and ranking every larger neighbourhood by a wavefront of its own took 81 and 75 us.
// LDS: 32 groups x 96 candidates x 12 bytes (36 KB, four workgroups per CU), 16 bytes with PAIR.
constexpr int kSelCandidates = 96;

struct SelArgs {
    const float4 *xyzi;
    const CloudHdr *hdr;
    GridDesc g;
    const uint32_t *start;
    const int32_t *order;
    const float4 *sxyzi;
    int32_t K, pad;
    double rg;  // PAIR
    Moments *mom, *mom_g;
    int32_t *ovf;
    uint32_t *ovf_n;
};

template <int KIND, bool PAIR, int N>
__global__ __launch_bounds__(kNbBlock) void k_moments_sel(Jobs<SelArgs, N> J)
{
    constexpr int PER = kSelCandidates / kNbLanes;
    constexpr int WORDS = KIND == 1 || PAIR ? 4 : 3;  // the gradient's candidates carry their intensity
    __shared__ float cand[kNbBlock / kNbLanes][WORDS][kSelCandidates];
    const SelArgs &A = J.a[N == 1 ? 0 : blockIdx.y];
    const GridDesc &g = A.g;
    const GridView v = make_view(g, A.start, nullptr, A.sxyzi);
    const int n = A.hdr->n;
    const int32_t K = A.K;
    const int gl = (int)threadIdx.x & (kNbLanes - 1);
    const int base = lane_id() & ~(kNbLanes - 1);  // the group's first lane in its wavefront
    auto &C = cand[(int)threadIdx.x / kNbLanes];
    const double r2 = (double)g.radius * (double)g.radius;
    const double inv = kFx20 * (1.0 / (double)g.radius);
    const double rg2 = PAIR ? A.rg * A.rg : 0.0, inv_g = PAIR ? kFx20 * (1.0 / A.rg) : 0.0;
    for (int i = (int)(blockIdx.x * kNbBlock + threadIdx.x) / kNbLanes; i < n; i += (int)(gridDim.x * kNbBlock) / kNbLanes) {
        const float4 q = A.xyzi[i];
        Box b;
        int32_t cnt = 0;
        const bool box = grid_range(g, q.x, q.y, q.z, b.lo, b.hi);
        wave_lds_sync();
        if (box)
            group_walk_box<kNbUnroll>(
                v, b, gl, kNbLanes,
                [&](uint32_t, float4 c, bool valid) {
                    const bool in = valid && dist2(c.x, c.y, c.z, q.x, q.y, q.z) < r2;
                    const uint32_t m = (uint32_t)(__ballot(in) >> base) & ((1u << kNbLanes) - 1u);
                    const int pos = cnt + __popc(m & ((1u << gl) - 1u));
                    if (in && pos < kSelCandidates) {
                        C[0][pos] = c.x;
                        C[1][pos] = c.y;
                        C[2][pos] = c.z;
                        if (WORDS == 4) C[WORDS - 1][pos] = c.w;
                    }
                    cnt += __popc(m);
                });
        wave_lds_sync();
        const bool over = cnt > kSelCandidates;
        if (!over) {
            double d[PER];
#pragma unroll
            for (int j = 0; j < PER; ++j) {
                const int e = gl + kNbLanes * j;
                d[j] = e < cnt ? dist2(C[0][e], C[1][e], C[2][e], q.x, q.y, q.z) : DBL_MAX;
            }
            double thr = r2;  // all of them
            int below = K;    // of the K, how many are below thr: fewer only for a tie at thr
            if (cnt > K) {
                const bool plain = find_threshold(
                    cnt, K, r2, thr, below,
                    [&](double t) {
                        uint32_t c = 0;
#pragma unroll
                        for (int j = 0; j < PER; ++j) c += d[j] < t ? 1u : 0u;
                        return (int)group_sum<kNbLanes>(c);
                    },
                    [&](double t) {
                        double v = DBL_MAX;
#pragma unroll
                        for (int j = 0; j < PER; ++j) v = d[j] >= t ? fmin(v, d[j]) : v;
                        return group_min<kNbLanes>(v);
                    });
                if (plain) below = K;
            }
            MomentSum<KIND> M;
            MomentSum<1> Mg;
            uint32_t cg = 0;
            M.zero();
            Mg.zero();
#pragma unroll
            for (int j = 0; j < PER; ++j) {
                const int e = gl + kNbLanes * j;
                if (!(d[j] < r2)) continue;
                const float x = C[0][e], y = C[1][e], z = C[2][e], w = WORDS == 4 ? C[WORDS - 1][e] : 0.f;
                if (d[j] < thr) M.add(q, x, y, z, w, inv);
                if (PAIR && d[j] < rg2) {
                    Mg.add(q, x, y, z, w, inv_g);
                    ++cg;
                }
            }
            // a tie: of the points at that distance, those of the lowest indices.  A second walk puts them
            // where the candidates were, and each finds its place among them (a walk for each of them in
            // turn took 8000 points of a cubic lattice, 18 to choose of 24 each, from 126 to 173 us).
            if (below < K) {
                int32_t *slots = reinterpret_cast<int32_t *>(C[0]), *index = reinterpret_cast<int32_t *>(C[1]);
                int nt = 0;
                wave_lds_sync();
                group_walk_box<kNbUnroll>(v, b, gl, kNbLanes, [&](uint32_t s, float4 c, bool valid) {
                    const bool in = valid && dist2(c.x, c.y, c.z, q.x, q.y, q.z) == thr;
                    const uint32_t m = (uint32_t)(__ballot(in) >> base) & ((1u << kNbLanes) - 1u);
                    if (in) {
                        const int pos = nt + __popc(m & ((1u << gl) - 1u));  // (no more than cnt of them)
                        slots[pos] = (int32_t)s;
                        index[pos] = A.order[s];
                    }
                    nt += __popc(m);
                });
                wave_lds_sync();
                for (int e = gl; e < nt; e += kNbLanes) {
                    const int32_t mine = index[e];
                    int lower = 0;
                    for (int o = 0; o < nt; ++o) lower += index[o] < mine ? 1 : 0;
                    if (lower >= K - below) continue;
                    const float4 p = v.sxyzi[slots[e]];
                    M.add(q, p.x, p.y, p.z, p.w, inv);
                }
            }
            group_store<KIND>(M, min(cnt, K), gl, A.mom[i]);
            if (PAIR) group_store<1>(Mg, (int32_t)group_sum<kNbLanes>(cg), gl, A.mom_g[i]);
        }
        if (over && gl == 0) A.ovf[atomicAdd(A.ovf_n, 1u)] = i;
    }
}

// The overflow queries, one wavefront each: the K smallest (d2, index) keys by wave_collect; with
// mom_g, then the gradient's sums over all neighbours within rg.
struct OvfArgs {
    const float4 *xyzi;
    const CloudHdr *hdr;
    GridDesc g;
    const uint32_t *start;
    const int32_t *order;
    const float4 *sxyzi;
    int32_t K, pad;
    const int32_t *ovf;
    const uint32_t *ovf_n;
    Moments *mom, *mom_g;
    double rg;
};

template <int KIND, int N>
__global__ __launch_bounds__(kWave *kOvfWaves) void k_moments_overflow(Jobs<OvfArgs, N> J)
{
    const OvfArgs &A = J.a[N == 1 ? 0 : blockIdx.y];
    const GridDesc &g = A.g;
    const int32_t K = A.K;
    __shared__ SelBuf<true> bufs[kOvfWaves];
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
    const int lane = lane_id();
    SelBuf<true> &buf = bufs[w];
    const GridView v = make_view(g, A.start, A.order, A.sxyzi);
    const int n = A.hdr->n;
    const uint32_t m = *A.ovf_n;
    const double r2 = (double)g.radius * (double)g.radius;
    const double inv = kFx20 * (1.0 / (double)g.radius);
    for (uint32_t e = blockIdx.x * kOvfWaves + w; e < m; e += gridDim.x * kOvfWaves) {
        const int qi = A.ovf[e];
        if (qi < 0 || qi >= n) continue;
        const float4 q = A.xyzi[qi];  // in reach of the grid, or it would have no candidates
        long long S[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, t[9];
        int32_t cnt = 0;
        Box b;
        if (!grid_range(g, q.x, q.y, q.z, b.lo, b.hi)) continue;
        {
            MomentSum<KIND> M;
            double ld = -1.0;  // the largest key taken (K beyond one collection: several)
            int32_t li = -1;
            while (cnt < K) {
                const int want = min(K - cnt, kSelBlock);
                const int got = wave_collect(v, b, q, r2, want, ld, li, buf);
                double md = -1.0;
                int32_t mi = -1;
                M.zero();
                for (int k = lane; k < got; k += kWave) {
                    const float4 p = v.sxyzi[buf.slot[k]];
                    M.add(q, p.x, p.y, p.z, p.w, inv);
                    if (key_less(md, mi, buf.d2[k], buf.idx[k])) {
                        md = buf.d2[k];
                        mi = buf.idx[k];
                    }
                }
                M.take(t);
#pragma unroll
                for (int k = 0; k < 9; ++k) S[k] += t[k];
                cnt += got;
                if (got < want || cnt >= K) break;
                for (int s = 1; s < kWave; s <<= 1) {
                    const double od = __shfl_xor(md, s, kWave);
                    const int32_t oi = __shfl_xor(mi, s, kWave);
                    if (key_less(md, mi, od, oi)) {
                        md = od;
                        mi = oi;
                    }
                }
                ld = md;
                li = mi;
            }
        }
        wave_store(S, cnt, A.mom[qi]);
        if (KIND == 0 && A.mom_g) {
            const double rg2 = A.rg * A.rg, inv_g = kFx20 * (1.0 / A.rg);
            MomentSum<1> M;
            const int32_t cg = wave_sum(walk_moments<1>(v, b, q, lane, kWave, rg2, inv_g, M));
            if (cg <= kExactTerms) M.take(S);
            else walk_moments_wide<1>(v, b, q, lane, kWave, rg2, inv_g, S);
            wave_store(S, cg, A.mom_g[qi]);
        }
    }
}

// Colour gradient from the tangent-plane moments: A = sum w w^T r^2 + (k-1)^2 n n^T + 1e-6 I,
// b = sum w dI r, solved by unpivoted LDL^T (cuda_compute_color_gradient.cu:41-90,
// little_3x3_ldlt_solve.cuh:11-60); fewer than 5 neighbours (query included) -> zero.
__device__ __forceinline__ float4 gradient_from_moments(int32_t k, const long long S[9], float4 nf, double radius)
{
    float4 out = make_float4(0.f, 0.f, 0.f, 0.f);
    if (k < 5) return out;  // cuda_compute_color_gradient.cu:41-44
    const double nv[3] = {(double)nf.x, (double)nf.y, (double)nf.z};
    const double rr = radius * radius;
    const double kk = (double)(k - 1) * (double)(k - 1);
    const int IA[6] = {0, 0, 0, 1, 1, 2}, IB[6] = {0, 1, 2, 1, 2, 2};
    // sum w w^T = P E P and sum w dI = P F for w = P u, P = I - n n^T (:48-60), E and F the raw
    // sums; the same expressions as the oracle's project_tangent
    double M[3][3], f[3], Mn[3];
    for (int c = 0; c < 6; ++c) {
        const double v = (double)S[c] / kFx40;
        M[IA[c]][IB[c]] = v;
        M[IB[c]][IA[c]] = v;
    }
    for (int a = 0; a < 3; ++a) f[a] = (double)S[6 + a] / kFx40;
    for (int a = 0; a < 3; ++a) Mn[a] = (M[a][0] * nv[0] + M[a][1] * nv[1]) + M[a][2] * nv[2];
    const double nMn = (nv[0] * Mn[0] + nv[1] * Mn[1]) + nv[2] * Mn[2];
    double A[3][3];
    for (int c = 0; c < 6; ++c) {
        const int a = IA[c], bb = IB[c];
        const double pmp = ((M[a][bb] - nv[a] * Mn[bb]) - Mn[a] * nv[bb]) + (nv[a] * nv[bb]) * nMn;
        double v = pmp * rr + kk * (nv[a] * nv[bb]);
        A[a][bb] = v;
        A[bb][a] = v;
    }
    for (int a = 0; a < 3; ++a) A[a][a] += 1.0e-6;
    const double fn = (f[0] * nv[0] + f[1] * nv[1]) + f[2] * nv[2];
    double b[3];
    for (int a = 0; a < 3; ++a) b[a] = (f[a] - fn * nv[a]) * radius;
    double D0 = A[0][0];
    double L10 = A[1][0] / D0, L20 = A[2][0] / D0;
    double D1 = A[1][1] - L10 * L10 * D0;
    double L21 = (A[2][1] - L10 * L20 * D0) / D1;
    double D2 = A[2][2] - L20 * L20 * D0 - L21 * L21 * D1;
    double x0 = b[0];
    double x1 = b[1] - L10 * x0;
    double x2 = b[2] - L20 * x0 - L21 * x1;
    x0 /= D0;
    x1 /= D1;
    x2 /= D2;
    x1 -= L21 * x2;
    x0 -= L10 * x1 + L20 * x2;
    return make_float4((float)x0, (float)x1, (float)x2, 0.0f);
}

// Pass 3: one thread per point (FP64 eigen / LDL^T solves keep every lane busy).  Re-arms the
// overflow counter for the next call.
template <int KIND>
__global__ __launch_bounds__(kNbBlock) void k_solve(const CloudHdr *__restrict__ hdr, const Moments *__restrict__ mom,
                                                    const float4 *__restrict__ nrm, double radius,
                                                    float4 *__restrict__ out, uint32_t *__restrict__ ovf_n)
{
    const int n = hdr->n;
    if (blockIdx.x == 0 && threadIdx.x == 0) *ovf_n = 0u;
    for (int i = blockIdx.x * kNbBlock + threadIdx.x; i < n; i += gridDim.x * kNbBlock) {
        const Moments &M = mom[i];
        long long S[9];
#pragma unroll
        for (int c = 0; c < 9; ++c) S[c] = M.S[c];
        out[i] = KIND == 0 ? normal_from_moments(M.cnt, S) : gradient_from_moments(M.cnt, S, nrm[i], radius);
    }
}

// Pass 3 of the joint walk: the normal, then the colour gradient on that normal (the value
// stored, as a separate gradient call would read it back).
// order != nullptr: thread s solves point order[s] (the grid's sorted slot s) and also writes
// its normal and gradient to snrm[s] / sgrad[s], the grid-ordered copies registration reads.
struct SolveArgs {
    const CloudHdr *hdr;
    const Moments *mom, *mom_g;
    double rg;
    float4 *nrm, *grad;
    const int32_t *order;
    float4 *snrm, *sgrad;
    uint32_t *ovf_n;
};

template <int N>
__global__ __launch_bounds__(kNbBlock) void k_solve_pair(Jobs<SolveArgs, N> J)
{
    const SolveArgs &A = J.a[N == 1 ? 0 : blockIdx.y];
    const Moments *__restrict__ mom = A.mom;
    const Moments *__restrict__ mom_g = A.mom_g;
    const double rg = A.rg;
    float4 *__restrict__ nrm = A.nrm;
    float4 *__restrict__ grad = A.grad;
    const int32_t *__restrict__ order = A.order;
    float4 *__restrict__ snrm = A.snrm;
    float4 *__restrict__ sgrad = A.sgrad;
    const int n = A.hdr->n;
    if (blockIdx.x == 0 && threadIdx.x == 0) *A.ovf_n = 0u;
    for (int s = blockIdx.x * kNbBlock + threadIdx.x; s < n; s += gridDim.x * kNbBlock) {
        const int i = order ? order[s] : s;
        long long S[9];
        const Moments &M = mom[i];
#pragma unroll
        for (int c = 0; c < 9; ++c) S[c] = M.S[c];
        const float4 nf = normal_from_moments(M.cnt, S);
        nrm[i] = nf;
        const Moments &Mg = mom_g[i];
#pragma unroll
        for (int c = 0; c < 9; ++c) S[c] = Mg.S[c];
        const float4 gv = gradient_from_moments(Mg.cnt, S, nf, rg);
        grad[i] = gv;
        if (order) {
            snrm[s] = nf;
            sgrad[s] = gv;
        }
    }
}

static unsigned grid_for(int64_t items, int per_block, int64_t cap)
{
    return (unsigned)std::min<int64_t>(cap, std::max<int64_t>(1, (items + per_block - 1) / per_block));
}

// The sums without selection of the cloud of A, on grid d (K: those with more neighbours go to A's overflow
// list).
template <int KIND>
static void launch_all(dim3 grid, hipStream_t stream, const SelArgs &A, const GridDesc &d, Moments *mom, int32_t K)
{
    hipLaunchKernelGGL(k_moments<KIND>, grid, dim3(kNbBlock), 0, stream, A.xyzi, A.hdr, d, A.start, A.sxyzi, mom, K, A.ovf,
                       A.ovf_n);
}

static bool selects(int32_t K) { return K > 0 && K < kSelCandidates; }

template <int KIND>
static int32_t launch_moments_pipeline(gca_ctx ctx, gca_cloud c, float radius, int32_t K, float4 *out)
{
    const Grid &G = c->grid;
    const int64_t cap = std::max<int64_t>(c->cap, 1);
    Moments *mom = (Moments *)ctx_scratch(ctx, 17, sizeof(Moments) * cap, false);
    int32_t *ovf = (int32_t *)ctx_scratch(ctx, 18, sizeof(int32_t) * cap, false);
    uint32_t *ovf_n = (uint32_t *)ctx_scratch(ctx, 19, 256, true);  // zero, re-armed by k_solve
    if (!mom || !ovf || !ovf_n) return GCA_ERR_OUT_OF_MEMORY;
    const GridDesc d = query_desc(G, radius);
    StageTimer timer(ctx, KIND == 0 ? GCA_STAGE_NORMALS : GCA_STAGE_GRADIENT);
    const dim3 grid(grid_for(cap, kNbBlock / kNbLanes, 4096));
    const Jobs<SelArgs, 1> sj{{{c->xyzi, c->hdr, d, G.start, G.order, G.sxyzi, K, 0, 0.0, mom, nullptr, ovf, ovf_n}}};
    if (selects(K)) hipLaunchKernelGGL((k_moments_sel<KIND, false, 1>), grid, dim3(kNbBlock), 0, ctx->stream, sj);
    else launch_all<KIND>(grid, ctx->stream, sj.a[0], d, mom, K);
    if (K > 0) {
        const Jobs<OvfArgs, 1> oj{{{c->xyzi, c->hdr, d, G.start, G.order, G.sxyzi, K, 0, ovf, ovf_n, mom, nullptr, 0.0}}};
        hipLaunchKernelGGL((k_moments_overflow<KIND, 1>), dim3(grid_for(cap, kOvfWaves, 1024)), dim3(kWave * kOvfWaves),
                           0, ctx->stream, oj);
    }
    hipLaunchKernelGGL(k_solve<KIND>, dim3(grid_for(cap, kNbBlock, 2048)), dim3(kNbBlock), 0, ctx->stream, c->hdr,
                       (const Moments *)mom, (const float4 *)c->nrm, (double)radius, out, ovf_n);
    GCA_HIP(hipGetLastError());
    return GCA_OK;
}

int32_t launch_normals(gca_ctx ctx, gca_cloud c, float radius, int32_t K)
{
    return launch_moments_pipeline<0>(ctx, c, radius, K, c->nrm);
}

int32_t launch_gradient(gca_ctx ctx, gca_cloud c, float radius, int32_t K)
{
    return launch_moments_pipeline<1>(ctx, c, radius, K, c->grad);
}

// The three kernels of one joint normals + gradient call, as jobs.
struct PairJobs {
    SelArgs pair;
    OvfArgs ovf;
    SolveArgs solve;
    unsigned nb_pair, nb_ovf, nb_solve;
};

static int32_t pair_prepare(gca_ctx ctx, gca_cloud c, float radius, int32_t K, float gradient_radius, bool grid_attrs,
                            int lane, int64_t n, PairJobs *pj)
{
    if (!(gradient_radius <= radius)) return GCA_ERR_INVALID_VALUE;
    Grid &G = c->grid;
    if (grid_attrs) GCA_TRY(grid_alloc_attributes(c));
    const int64_t cap = std::max<int64_t>(n > 0 ? n : c->cap, 1);
    Moments *mom = (Moments *)lane_scratch(ctx, lane, 17, sizeof(Moments) * cap, false);
    int32_t *ovf = (int32_t *)lane_scratch(ctx, lane, 18, sizeof(int32_t) * cap, false);
    uint32_t *ovf_n = (uint32_t *)lane_scratch(ctx, lane, 19, 256, true);  // zero, re-armed by k_solve_pair
    Moments *mom_g = (Moments *)lane_scratch(ctx, lane, 24, sizeof(Moments) * cap, false);
    if (!mom || !ovf || !ovf_n || !mom_g) return GCA_ERR_OUT_OF_MEMORY;
    const GridDesc d = query_desc(G, radius);
    const double rg = (double)gradient_radius;
    pj->pair = SelArgs{c->xyzi, c->hdr, d, G.start, G.order, G.sxyzi, K, 0, rg, mom, mom_g, ovf, ovf_n};
    pj->ovf = OvfArgs{c->xyzi, c->hdr, d, G.start, G.order, G.sxyzi, K, 0, ovf, ovf_n, mom, mom_g, rg};
    pj->solve = SolveArgs{c->hdr, mom, mom_g, rg, c->nrm, c->grad, grid_attrs ? (const int32_t *)G.order : nullptr,
                          grid_attrs ? G.snrm : nullptr, grid_attrs ? G.sgrad : nullptr, ovf_n};
    pj->nb_pair = grid_for(cap, kNbBlock / kNbLanes, 4096);
    pj->nb_ovf = grid_for(cap, kOvfWaves, 1024);
    pj->nb_solve = grid_for(cap, kNbBlock, 2048);
    return GCA_OK;
}

// moments, overflow K-selection, solve: each kernel once for all nj calls (blockIdx.y = call), on
// stream.  A call that selects nothing in its walk (no K cap, or one beyond the buffer) has nothing to
// share with the gradient's, so its two sums come from a walk each.
template <int N>
static int32_t pair_launch(hipStream_t stream, const PairJobs *pj, int nj)
{
    Jobs<SelArgs, N> pair{};
    Jobs<OvfArgs, N> ovf{};
    Jobs<SolveArgs, N> solve{};
    unsigned nb_pair = 1, nb_ovf = 1, nb_solve = 1, nsel = 0, novf = 0;
    for (int j = 0; j < nj; ++j) {
        const SelArgs &A = pj[j].pair;
        if (selects(A.K)) {
            pair.a[nsel++] = A;
            nb_pair = std::max(nb_pair, pj[j].nb_pair);
        } else {
            GridDesc dg = A.g;
            dg.radius = (float)A.rg;
            launch_all<0>(dim3(pj[j].nb_pair), stream, A, A.g, A.mom, A.K);
            launch_all<1>(dim3(pj[j].nb_pair), stream, A, dg, A.mom_g, 0);
        }
        if (A.K > 0) {
            ovf.a[novf] = pj[j].ovf;
            if (!selects(A.K)) ovf.a[novf].mom_g = nullptr;  // (the gradient's sums are complete)
            ++novf;
            nb_ovf = std::max(nb_ovf, pj[j].nb_ovf);
        }
        solve.a[j] = pj[j].solve;
        nb_solve = std::max(nb_solve, pj[j].nb_solve);
    }
    if (nsel > 0) hipLaunchKernelGGL((k_moments_sel<0, true, N>), dim3(nb_pair, nsel), dim3(kNbBlock), 0, stream, pair);
    if (novf > 0) hipLaunchKernelGGL((k_moments_overflow<0, N>), dim3(nb_ovf, novf), dim3(kWave * kOvfWaves), 0, stream, ovf);
    hipLaunchKernelGGL(k_solve_pair<N>, dim3(nb_solve, (unsigned)nj), dim3(kNbBlock), 0, stream, solve);
    GCA_HIP(hipGetLastError());
    return GCA_OK;
}

int32_t launch_normals_gradient(gca_ctx ctx, gca_cloud c, float radius, int32_t K, float gradient_radius,
                                bool grid_attrs)
{
    PairJobs pj;
    GCA_TRY(pair_prepare(ctx, c, radius, K, gradient_radius, grid_attrs, 0, 0, &pj));
    {
        StageTimer timer(ctx, GCA_STAGE_NORMALS);
        GCA_TRY(pair_launch<1>(ctx->stream, &pj, 1));
    }
    if (grid_attrs) c->grid.attrs_valid = true;
    return GCA_OK;
}

int32_t launch_normals_gradient_levels(gca_ctx launch, const NormalsLevelJob *jobs, int nj)
{
    if (nj < 1 || nj > kMaxJobs) return GCA_ERR_INVALID_VALUE;
    PairJobs pj[kMaxJobs];
    for (int j = 0; j < nj; ++j)
        GCA_TRY(pair_prepare(jobs[j].ctx, jobs[j].c, jobs[j].radius, jobs[j].max_nn, jobs[j].gradient_radius, true,
                             jobs[j].lane, jobs[j].n, &pj[j]));
    {
        StageTimer timer(launch, GCA_STAGE_NORMALS);
        GCA_TRY(pair_launch<kMaxJobs>(launch->stream, pj, nj));
    }
    for (int j = 0; j < nj; ++j) jobs[j].c->grid.attrs_valid = true;
    return GCA_OK;
}

}  // namespace gca
