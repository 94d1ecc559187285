// Normal estimation for an unoriented point cloud on the device: the step
// before the reconstruction, which the reference runs on the host with PCL
// (mesh/PoissonReconstruction.cpp:137-186: NormalEstimationOMP, k = 10
// nearest neighbours from a kd-tree, default viewpoint (0, 0, 0)).  PCL is a
// third-party library absent here; its published algorithm is restated:
//   * the k nearest neighbours of each point, the point itself included
//     (distance 0);
//   * their mean and covariance, the eigenvector of the smallest eigenvalue
//     as the normal and lambda_0 / (lambda_0 + lambda_1 + lambda_2) as the
//     curvature (computePointNormal, solvePlaneParameters);
//   * the normal flipped to face the viewpoint: n = -n when (vp - p) . n < 0
//     (flipNormalTowardsViewpoint).
// Nearest neighbours are exact: points are bucketed in a uniform grid, a point
// searches the (2r+1)^3 cells around its own, and r grows until the k-th
// distance lies within the searched box.  Ties go to the lower point index.
#include "psr_internal.h"
#include "psr_prims.h"

#include <cmath>
#include <stdexcept>
#include <type_traits>

namespace psr {
namespace {

constexpr int kThreads = 256;
constexpr int kMaxK = 16;
constexpr int kBoundsBlocks = 128;  // workgroups of the bounds pass
constexpr int kMailBounds = 46;     // mailbox slot: the points' bounds are not finite
static_assert(kMailBounds > kMailGeo + 2 && kMailBounds < kMailScanErr, "mailbox slot of the bounds");

// The search grid, computed on the device from the points' bounds.
struct GridSpec {
    float3 lo;
    float h, invH;
    float eps;  // bound of the rounding in a coordinate's cell assignment
    int G;      // cells per axis
    int ok;     // the bounds are finite
};

__device__ __forceinline__ int3 cell_of(float3 p, const GridSpec& g) {
    return make_int3(min(g.G - 1, max(0, int((p.x - g.lo.x) * g.invH))), min(g.G - 1, max(0, int((p.y - g.lo.y) * g.invH))),
                     min(g.G - 1, max(0, int((p.z - g.lo.z) * g.invH))));
}

__device__ __forceinline__ float3 load_point(const char* xyz, unsigned stride, int i) {
    const float* p = reinterpret_cast<const float*>(xyz + size_t(i) * stride);
    return make_float3(p[0], p[1], p[2]);
}

// Per-block bounds of the points.
__global__ void __launch_bounds__(kThreads) ne_bounds(const char* __restrict__ xyz, unsigned stride, int n,
                                                      float* __restrict__ part) {
    __shared__ float s[6][kThreads];
    float mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int i = blockIdx.x * kThreads + threadIdx.x; i < n; i += gridDim.x * kThreads) {
        const float3 p = load_point(xyz, stride, i);
        mn[0] = fminf(mn[0], p.x), mn[1] = fminf(mn[1], p.y), mn[2] = fminf(mn[2], p.z);
        mx[0] = fmaxf(mx[0], p.x), mx[1] = fmaxf(mx[1], p.y), mx[2] = fmaxf(mx[2], p.z);
    }
    for (int a = 0; a < 3; ++a) s[a][threadIdx.x] = mn[a], s[3 + a][threadIdx.x] = mx[a];
    __syncthreads();
    for (int st = kThreads / 2; st > 0; st >>= 1) {
        if (int(threadIdx.x) < st)
            for (int a = 0; a < 3; ++a) {
                s[a][threadIdx.x] = fminf(s[a][threadIdx.x], s[a][threadIdx.x + st]);
                s[3 + a][threadIdx.x] = fmaxf(s[3 + a][threadIdx.x], s[3 + a][threadIdx.x + st]);
            }
        __syncthreads();
    }
    if (threadIdx.x < 6) part[blockIdx.x * 6 + threadIdx.x] = s[threadIdx.x][0];
}

// The grid of G cells an axis over the nb block bounds, in every thread of
// the block (each workgroup of the next kernel reduces the few partials
// itself: no host round trip, no launch of its own).
__device__ __forceinline__ GridSpec grid_from_bounds(const float* __restrict__ part, int nb, int G) {
    __shared__ float s[6][2];
    __shared__ GridSpec sg;
    static_assert(kBoundsBlocks <= 2 * PSR_WAVE, "two waves reduce the partials");
    if (threadIdx.x < 2 * PSR_WAVE) {
        float v[6];
        for (int a = 0; a < 6; ++a) v[a] = int(threadIdx.x) < nb ? part[threadIdx.x * 6 + a] : (a < 3 ? INFINITY : -INFINITY);
        for (int off = PSR_WAVE / 2; off > 0; off >>= 1)
            for (int a = 0; a < 6; ++a) {
                const float o = __shfl_xor(v[a], off, PSR_WAVE);
                v[a] = a < 3 ? fminf(v[a], o) : fmaxf(v[a], o);
            }
        if (__lane_id() == 0)
            for (int a = 0; a < 6; ++a) s[a][threadIdx.x / PSR_WAVE] = v[a];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        float lo[3], hi[3], ext = 1e-30f, mag = 0.f;
        int ok = 1;
        for (int a = 0; a < 3; ++a) {
            lo[a] = fminf(s[a][0], s[a][1]);
            hi[a] = fmaxf(s[3 + a][0], s[3 + a][1]);
            if (!isfinite(lo[a]) || !isfinite(hi[a])) ok = 0;
            ext = fmaxf(ext, hi[a] - lo[a]);
            mag = fmaxf(mag, fmaxf(fabsf(lo[a]), fabsf(hi[a])));
        }
        GridSpec g;
        g.lo = make_float3(lo[0], lo[1], lo[2]);
        g.G = G;
        g.h = ext * 1.0001f / float(G);
        g.invH = 1.0f / g.h;
        g.eps = 8e-7f * (mag + ext);
        g.ok = ok;
        sg = g;
    }
    __syncthreads();
    return sg;
}

// Grid cell (x-major linear index) of every point, the identity values, the
// points as (x, y, z, index) for the sort's gather, and the first pass's
// histogram of this workgroup's sort tile; block 0 stores the grid and
// reports bounds that are not finite.
__global__ void __launch_bounds__(kThreads) ne_cells(const char* __restrict__ xyz, unsigned stride, int n,
                                                     const float* __restrict__ part, int nb, int G,
                                                     GridSpec* __restrict__ grid, int* __restrict__ mail,
                                                     unsigned* __restrict__ key, unsigned* __restrict__ val,
                                                     float4* __restrict__ pos, int tiles, int* __restrict__ hist,
                                                     unsigned digitMask) {
    __shared__ int lh[256];
    static_assert(kThreads == 256 && kSortTileKeys == 2 * kThreads, "one thread per digit, two keys each");
    lh[threadIdx.x] = 0;
    const GridSpec g = grid_from_bounds(part, nb, G);  // its barriers publish lh
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        *grid = g;
        if (!g.ok) *mail = 1;
    }
    for (int k = 0; k < 2; ++k) {
        const int i = blockIdx.x * kSortTileKeys + k * kThreads + threadIdx.x;
        if (i >= n) continue;
        const float3 p = load_point(xyz, stride, i);
        const int3 c = cell_of(p, g);
        const unsigned cell = (unsigned(c.x) * unsigned(g.G) + unsigned(c.y)) * unsigned(g.G) + unsigned(c.z);
        key[i] = cell;
        val[i] = unsigned(i);
        pos[i] = make_float4(p.x, p.y, p.z, __int_as_float(i));
        atomicAdd(&lh[cell & digitMask], 1);
    }
    __syncthreads();
    if (threadIdx.x <= digitMask) hist[threadIdx.x * tiles + blockIdx.x] = lh[threadIdx.x];
}

// First sorted position in [0, n) whose cell is >= c, found by a whole wave:
// 64 probes a step (3 round trips for 200k keys, where one lane halving the
// range takes 18).
__device__ __forceinline__ int wave_lower_bound(const unsigned* __restrict__ key, int n, unsigned c) {
    const int lane = int(__lane_id());
    int lo = 0, len = n;  // the answer lies in [lo, lo + len]
    while (len > 0) {
        const int step = (len + PSR_WAVE - 1) / PSR_WAVE;
        const int at = lo + min(len, (lane + 1) * step) - 1;  // last key of the lane's part
        const int below = __popcll(__ballot(key[at] < c));    // parts that lie below c: a prefix
        const int skip = min(len, below * step);
        lo += skip;
        len = below == PSR_WAVE ? 0 : min(len - skip, step - 1);  // the next part's last key is >= c
    }
    return lo;
}

// start[c] = first sorted position whose cell is >= c, for c in [0, cells].
// A workgroup takes 2048 consecutive cells: two waves find its range of sorted
// positions, every first point of a cell is marked, and a scan from the right
// carries the marks over the empty cells (most: a surface meets few of them).
// 200k points: 25 us for 2.1M cells with a search of all keys per cell, 6.6 us
// here for the 0.97M cells of the same cloud.
constexpr int kStartItems = 8, kStartCells = kStartItems * kThreads;
__global__ void __launch_bounds__(kThreads) ne_cell_starts(const unsigned* __restrict__ key, int n, unsigned cells,
                                                           int* __restrict__ start) {
    __shared__ int sRange[2], sWave[kThreads / PSR_WAVE];
    __shared__ int first[kStartCells];
    const unsigned c0 = blockIdx.x * unsigned(kStartCells);
    const int w = threadIdx.x / PSR_WAVE, lane = int(__lane_id());
    for (int k = threadIdx.x; k < kStartCells; k += kThreads) first[k] = n;  // no point
    if (w < 2) {
        const int r = wave_lower_bound(key, n, w == 0 ? c0 : c0 + kStartCells);
        if (lane == 0) sRange[w] = r;
    }
    __syncthreads();
    const int b = sRange[0], e = sRange[1];
    for (int i = b + int(threadIdx.x); i < e; i += kThreads) {
        const unsigned c = key[i];
        if (i == b || key[i - 1] != c) first[c - c0] = i;
    }
    __syncthreads();
    int v[kStartItems], run = n;
#pragma unroll
    for (int k = kStartItems - 1; k >= 0; --k) v[k] = run = min(run, first[threadIdx.x * kStartItems + k]);
    // the smallest mark of the threads to the right: within the wave, then the waves
    int inc = run;
#pragma unroll
    for (int off = 1; off < PSR_WAVE; off <<= 1) {
        const int o = __shfl_down(inc, off, PSR_WAVE);
        if (lane + off < PSR_WAVE) inc = min(inc, o);
    }
    if (lane == 0) sWave[w] = inc;
    int right = __shfl_down(inc, 1, PSR_WAVE);
    if (lane == PSR_WAVE - 1) right = n;
    __syncthreads();
    for (int k = w + 1; k < kThreads / PSR_WAVE; ++k) right = min(right, sWave[k]);
    right = min(right, e);  // past the workgroup's last point: its end
#pragma unroll
    for (int k = 0; k < kStartItems; ++k) first[threadIdx.x * kStartItems + k] = min(v[k], right);
    __syncthreads();
    for (int k = threadIdx.x; k < kStartCells; k += kThreads)
        if (c0 + k <= cells) start[c0 + k] = first[k];
}

// 1 / sqrt(x) and 1 / x to FP64's last bit or two: the hardware's estimate and
// two Newton steps.
__device__ __forceinline__ double rsqrt_newton(double x) {
    double r = __builtin_amdgcn_rsq(x);
    r = __fma_rn(0.5 * r, __fma_rn(-x * r, r, 1.0), r);
    return __fma_rn(0.5 * r, __fma_rn(-x * r, r, 1.0), r);
}
__device__ __forceinline__ double rcp_newton(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = __fma_rn(r, __fma_rn(-x, r, 1.0), r);
    return __fma_rn(r, __fma_rn(-x, r, 1.0), r);
}

// Cyclic Jacobi on a symmetric 3 x 3 matrix, in FP64: eigenvalues on the
// diagonal, eigenvectors in the columns of V.  With theta = (a_qq - a_pp) / (2
// a_pq), t = sign(theta) / (|theta| + sqrt(theta^2 + 1)) is formed without the
// quotient theta.  Roots and reciprocals by Newton steps in place of the
// library's correctly rounded ones, whose instructions were three quarters of a
// rotation's.
template <int P, int Q>
__device__ __forceinline__ void jacobi_rotate(double (&A)[3][3], double (&V)[3][3]) {
    constexpr int R = 3 - P - Q;
    if (A[P][Q] == 0.0) return;
    const double dif = A[Q][Q] - A[P][P], h = 2.0 * A[P][Q], x = __fma_rn(dif, dif, h * h);
    if (x == 0.0) return;  // the squares underflow: nothing to rotate beside the entries that do not
    const double t = dif == 0.0 ? 1.0 : (dif > 0.0 ? h : -h) * rcp_newton(fabs(dif) + x * rsqrt_newton(x));
    const double cs = rsqrt_newton(__fma_rn(t, t, 1.0));
    const double sn = t * cs;
    const double app = A[P][P], aqq = A[Q][Q], apq = A[P][Q], arp = A[R][P], arq = A[R][Q];
    const double cc = cs * cs, ss = sn * sn, sc = sn * cs;
    A[P][P] = __fma_rn(cc, app, __fma_rn(ss, aqq, -2.0 * sc * apq));
    A[Q][Q] = __fma_rn(ss, app, __fma_rn(cc, aqq, 2.0 * sc * apq));
    A[P][Q] = A[Q][P] = __fma_rn(sc, app - aqq, (cc - ss) * apq);
    A[R][P] = A[P][R] = __fma_rn(cs, arp, -sn * arq);
    A[R][Q] = A[Q][R] = __fma_rn(sn, arp, cs * arq);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const double vp = V[k][P], vq = V[k][Q];
        V[k][P] = __fma_rn(cs, vp, -sn * vq);
        V[k][Q] = __fma_rn(sn, vp, cs * vq);
    }
}
__device__ __forceinline__ void jacobi3(double (&A)[3][3], double (&V)[3][3]) {
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) V[i][j] = i == j ? 1.0 : 0.0;
    for (int sweep = 0; sweep < 32; ++sweep) {
        const double off = A[0][1] * A[0][1] + A[0][2] * A[0][2] + A[1][2] * A[1][2];
        const double diag = A[0][0] * A[0][0] + A[1][1] * A[1][1] + A[2][2] * A[2][2];
        if (off <= 1e-30 * diag || off == 0.0) break;
        jacobi_rotate<0, 1>(A, V);
        jacobi_rotate<0, 2>(A, V);
        jacobi_rotate<1, 2>(A, V);
    }
}

// A candidate as one ordered word: its squared distance (never negative, so
// its bits order as it does) above its point index, so the smaller word is the
// closer point, ties to the lower index.
typedef unsigned long long Cand;
constexpr unsigned kNoPoint = 0x7fffffffu;  // the index of a place without a point

__device__ __forceinline__ int cand_index(Cand c) { return int(unsigned(c)); }

// Squared distance of grid point o (its index in w) from p, the same bits
// wherever it is formed.
__device__ __forceinline__ float dist2(float4 o, float3 p) {
    const float dx = o.x - p.x, dy = o.y - p.y, dz = o.z - p.z;
    return __fmaf_rn(dz, dz, __fmaf_rn(dx, dx, __fmul_rn(dy, dy)));
}
__device__ __forceinline__ Cand candidate(float4 o, float3 p) {
    return (Cand(__float_as_uint(dist2(o, p))) << 32) | unsigned(__float_as_int(o.w));
}

// d into the ascending list of the K smallest distances: one median a place.
template <int K>
__device__ __forceinline__ void dist_insert(float (&best)[K], float d) {
#pragma unroll
    for (int j = K - 1; j > 0; --j) best[j] = __builtin_amdgcn_fmed3f(best[j - 1], best[j], d);
    best[0] = fminf(best[0], d);
}

// x into the ascending list of the K lowest indices.
template <int K>
__device__ __forceinline__ void index_insert(unsigned (&low)[K], unsigned x) {
#pragma unroll
    for (int j = K - 1; j > 0; --j) low[j] = max(low[j - 1], min(low[j], x));
    low[0] = min(low[0], x);
}

// Orders a wave's LDS writes before its later reads of other lanes' values.
__device__ __forceinline__ void wave_publish() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// The cells searched around p.
struct Box {
    int x0, x1, y0, y1, z0, z1;
};

// Calls f on every LANES-th point of the box's cells, this lane's share of the
// box.  A row of cells along z is one range of sorted points.  Nearly every
// search ends at radius 1: its nine rows' ranges are read together.
template <int LANES, class F>
__device__ __forceinline__ void for_points(const Box& o, int r, int3 c, int sub, int G, const float4* __restrict__ spos,
                                           const int* __restrict__ start, F f) {
    auto scan_row = [&](int b, int e) {
        for (int s = b + sub; s < e; s += 2 * LANES) {  // two loads in flight
            const float4 p0 = spos[s], p1 = spos[min(s + LANES, e - 1)];
            f(p0);
            if (s + LANES < e) f(p1);
        }
    };
    auto row_of = [&](int x, int y) { return (unsigned(x) * unsigned(G) + unsigned(y)) * unsigned(G); };
    if (r == 1) {
        int b[9], e[9];
#pragma unroll
        for (int q = 0; q < 9; ++q) {
            const int x = c.x + q / 3 - 1, y = c.y + q % 3 - 1;
            const bool in = x >= o.x0 && x <= o.x1 && y >= o.y0 && y <= o.y1;
            const unsigned row = row_of(in ? x : c.x, in ? y : c.y);
            b[q] = start[row + unsigned(o.z0)];
            e[q] = in ? start[row + unsigned(o.z1) + 1] : 0;
        }
#pragma unroll
        for (int q = 0; q < 9; ++q) scan_row(b[q], e[q]);
        return;
    }
    for (int x = o.x0; x <= o.x1; ++x)
        for (int y = o.y0; y <= o.y1; ++y) {
            const unsigned row = row_of(x, y);
            scan_row(start[row + unsigned(o.z0)], start[row + unsigned(o.z1) + 1]);
        }
}

// Exact kk <= K nearest of the grid's points to p, ties to the lower index:
// their indices, ascending by (distance, index), to found[0..kk) (stride
// `stride`).  The (2r+1)^3 cells around p's cell are searched, r growing until
// the kk-th distance lies inside the box; p may lie anywhere (its cell is
// clamped into the grid).  A first pass keeps the K smallest distances only
// (one median instruction a place, where an ordered list of distances with
// indices costs five), a second collects the points within the kk-th, and
// their ranks order them.  LANES consecutive lanes share one p, each taking
// every LANES-th point; list holds kListCap candidates of p, *cnt (zero at the
// call) their count.
constexpr int kListCap = 20;
template <int K, int LANES>
__device__ __forceinline__ void knn_search(float3 p, int sub, int kk, const GridSpec& g, const float4* __restrict__ spos,
                                           const int* __restrict__ start, int* cnt, Cand* list, int* found,
                                           int stride) {
    static_assert(K <= kListCap, "room for the nearest");
    const int3 c = cell_of(p, g);
    Box o;
    float dk;
    // a p that is not finite has no nearest cells: the whole grid at once
    int r = isfinite(p.x) && isfinite(p.y) && isfinite(p.z) ? 1 : g.G;
    for (;; ++r) {
        o = Box{max(0, c.x - r), min(g.G - 1, c.x + r), max(0, c.y - r), min(g.G - 1, c.y + r),
                max(0, c.z - r), min(g.G - 1, c.z + r)};
        float best[K];
#pragma unroll
        for (int j = 0; j < K; ++j) best[j] = INFINITY;
        for_points<LANES>(o, r, c, sub, g.G, spos, start, [&](float4 q) {
            dist_insert<K>(best, fminf(dist2(q, p), INFINITY));  // NaN: none
        });
#pragma unroll
        for (int m = 1; m < LANES; m <<= 1) {
            float other[K];
#pragma unroll
            for (int j = 0; j < K; ++j) other[j] = __shfl_xor(best[j], m, PSR_WAVE);
#pragma unroll
            for (int j = 0; j < K; ++j) dist_insert<K>(best, other[j]);
        }
        // every point outside the box lies at least cover - eps from p (eps:
        // the rounding of the cell assignment), so the k found are the nearest
        const bool all = o.x0 == 0 && o.y0 == 0 && o.z0 == 0 && o.x1 == g.G - 1 && o.y1 == g.G - 1 && o.z1 == g.G - 1;
        float cover = INFINITY;
        if (o.x0 > 0) cover = fminf(cover, p.x - (g.lo.x + o.x0 * g.h));
        if (o.y0 > 0) cover = fminf(cover, p.y - (g.lo.y + o.y0 * g.h));
        if (o.z0 > 0) cover = fminf(cover, p.z - (g.lo.z + o.z0 * g.h));
        if (o.x1 < g.G - 1) cover = fminf(cover, g.lo.x + (o.x1 + 1) * g.h - p.x);
        if (o.y1 < g.G - 1) cover = fminf(cover, g.lo.y + (o.y1 + 1) * g.h - p.y);
        if (o.z1 < g.G - 1) cover = fminf(cover, g.lo.z + (o.z1 + 1) * g.h - p.z);
        dk = INFINITY;
#pragma unroll
        for (int j = 0; j < K; ++j)
            if (j == kk - 1) dk = best[j];
        if (all || (dk < INFINITY && sqrtf(dk) * (1.0f + 1e-6f) + g.eps < cover)) break;
    }
    int added = 0;
    for_points<LANES>(o, r, c, sub, g.G, spos, start, [&](float4 q) {
        const Cand e = candidate(q, p);
        if (!(__uint_as_float(unsigned(e >> 32)) <= dk) || added > kListCap) return;
        const int at = atomicAdd(cnt, 1);
        ++added;
        if (at < kListCap) list[at] = e;
    });
    wave_publish();  // the lanes of p read each other's entries
    int m = *cnt;
    const bool ties = m > kListCap;
    unsigned tie[K];
#pragma unroll
    for (int j = 0; j < K; ++j) tie[j] = kNoPoint;
    if (ties) {
        // more points at the kk-th distance than the list holds: once more, the
        // nearer ones (fewer than kk) to the list and of those at the kk-th
        // distance the lowest indices, a median a place as for the distances
        wave_publish();
        if (sub == 0) *cnt = 0;
        wave_publish();
        for_points<LANES>(o, r, c, sub, g.G, spos, start, [&](float4 q) {
            const Cand e = candidate(q, p);
            const float d = __uint_as_float(unsigned(e >> 32));
            if (d < dk) list[atomicAdd(cnt, 1)] = e;
            else if (d == dk) index_insert<K>(tie, unsigned(e));
        });
#pragma unroll
        for (int w = 1; w < LANES; w <<= 1) {
            unsigned other[K];
#pragma unroll
            for (int j = 0; j < K; ++j) other[j] = __shfl_xor(tie[j], w, PSR_WAVE);
#pragma unroll
            for (int j = 0; j < K; ++j) index_insert<K>(tie, other[j]);
        }
        wave_publish();
        m = *cnt;
    }
    for (int j = sub; j < m; j += LANES) {
        const Cand e = list[j];
        int rank = 0;
        for (int i = 0; i < m; ++i) rank += list[i] < e ? 1 : 0;
        if (rank < kk) found[rank * stride] = cand_index(e);
    }
    // the places that are left: the ties, or no point (fewer than kk have a distance)
    if (m < kk && sub == 0) {
#pragma unroll
        for (int j = 0; j < K; ++j)
            if (m + j < kk) found[(m + j) * stride] = int(tie[j]);
    }
}

// The k nearest neighbours of each point, then the plane fit.  The points are
// taken in cell order, so a wave's searches read the same few cells, LANES
// lanes to a point; the fits (a serial FP64 chain each) are then made by
// kThreads / LANES threads of the workgroup, one a point.  Bound by the scan's
// instructions and the latency of its dependent loads (cell ranges, points).
// 200k points, k = 10: 319 us with a thread per point in input order (every
// lane in cells of its own), 89 us here, of which the fits take about 20.
// Lanes to a point, us a call at 30k / 200k / 700k points: 115 / 203 / 765
// with 2, 100 / 180 / 688 with 4.
constexpr int kFitLanes = 4;
template <int K, int LANES>
__global__ void __launch_bounds__(kThreads) ne_estimate(const char* __restrict__ xyz, unsigned stride, int n, int k,
                                                        const GridSpec* __restrict__ grid,
                                                        const float4* __restrict__ spos,
                                                        const int* __restrict__ start, float3 vp,
                                                        float* __restrict__ normals, float* __restrict__ curvature,
                                                        int* __restrict__ knn) {
    constexpr int Q = kThreads / LANES;  // points of a workgroup
    __shared__ int found[K][Q], cnt[Q];
    __shared__ Cand list[Q][kListCap + 1];  // an odd stride: the lanes' entries on different banks
    const GridSpec g = *grid;
    if (!g.ok) return;  // the call fails
    const int kk = min(k, n);
    {
        const int q = threadIdx.x / LANES, sub = threadIdx.x % LANES;
        const int at = blockIdx.x * Q + q;
        const float4 p4 = spos[min(at, n - 1)];
        if (sub == 0) cnt[q] = 0;
        knn_search<K, LANES>(make_float3(p4.x, p4.y, p4.z), sub, kk, g, spos, start, &cnt[q], list[q], &found[0][q], Q);
    }
    __syncthreads();
    const int at = blockIdx.x * Q + int(threadIdx.x);
    if (int(threadIdx.x) >= Q || at >= n) return;
    const float4 p4 = spos[at];
    const float3 p = make_float3(p4.x, p4.y, p4.z);
    const int i = __float_as_int(p4.w);
    // kNoPoint (fewer than kk points have a distance: NaN coordinates) reads as NaN
    auto point = [&](int q) {
        return q < n ? load_point(xyz, stride, q) : make_float3(NAN, NAN, NAN);
    };
    // mean and covariance of the neighbours in FP64
    double m[3] = {0, 0, 0};
    float3 nb[K];
#pragma unroll
    for (int j = 0; j < K; ++j) {
        if (j >= kk) continue;
        const int q = found[j][threadIdx.x];
        nb[j] = point(q);
        m[0] += nb[j].x, m[1] += nb[j].y, m[2] += nb[j].z;
        if (knn) knn[size_t(i) * k + j] = q;
    }
    for (int a = 0; a < 3; ++a) m[a] /= kk;
    double A[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
#pragma unroll
    for (int j = 0; j < K; ++j) {
        if (j >= kk) continue;
        const double d[3] = {nb[j].x - m[0], nb[j].y - m[1], nb[j].z - m[2]};
        for (int a = 0; a < 3; ++a)
            for (int b = a; b < 3; ++b) A[a][b] += d[a] * d[b];
    }
    for (int a = 0; a < 3; ++a)
        for (int b = a; b < 3; ++b) A[a][b] /= kk, A[b][a] = A[a][b];
    double V[3][3];
    jacobi3(A, V);
    int s = 0;
    if (A[1][1] < A[s][s]) s = 1;
    if (A[2][2] < A[s][s]) s = 2;
    double nx = V[0][s], ny = V[1][s], nz = V[2][s];
    const double len = sqrt(nx * nx + ny * ny + nz * nz);
    nx /= len, ny /= len, nz /= len;
    if ((vp.x - p.x) * nx + (vp.y - p.y) * ny + (vp.z - p.z) * nz < 0) nx = -nx, ny = -ny, nz = -nz;
    normals[3 * size_t(i)] = float(nx);
    normals[3 * size_t(i) + 1] = float(ny);
    normals[3 * size_t(i) + 2] = float(nz);
    if (curvature) {
        const double tr = A[0][0] + A[1][1] + A[2][2];
        curvature[i] = tr != 0.0 ? float(A[s][s] / tr) : 0.f;
    }
}

// --- vertex colours (DrawMesh.cu:35-79, 179-211) ---
// The colour of a mesh vertex from its 4 nearest points, weighted as the
// reference weights them: each squared distance over their sum (the farther
// point weighs more), colour = sum of weight x point colour.  Where all four
// distances are zero the weights are equal (the reference divides by zero).
// LANES lanes search for one vertex: a mesh has far fewer vertices than the
// GPU has lanes, and one lane's scan is a chain of dependent loads.  28k
// vertices of 200k points: 308 us with a thread a vertex over the points in
// input order, 44 us here (with 8 lanes the call takes 112 us, with 16 103;
// 66k vertices 127 and 131).
constexpr int kColorLanes = 16;
template <int LANES>
__global__ void __launch_bounds__(kThreads) vc_colors(const float* __restrict__ V, int nv,
                                                      const char* __restrict__ xyz, unsigned stride, int n,
                                                      const float* __restrict__ pc, const GridSpec* __restrict__ grid,
                                                      const float4* __restrict__ spos,
                                                      const int* __restrict__ start, float* __restrict__ out) {
    const GridSpec g = *grid;
    if (!g.ok) return;  // the call fails
    const int i = blockIdx.x * (kThreads / LANES) + threadIdx.x / LANES, sub = threadIdx.x % LANES;
    const size_t at = size_t(min(i, nv - 1));
    const float3 p = make_float3(V[3 * at], V[3 * at + 1], V[3 * at + 2]);
    const int kk = min(4, n);
    constexpr int Q = kThreads / LANES;
    __shared__ int found[Q][5], cnt[Q];
    __shared__ Cand list[Q][kListCap + 1];
    const int q = threadIdx.x / LANES;
    if (sub == 0) cnt[q] = 0;
    knn_search<4, LANES>(p, sub, kk, g, spos, start, &cnt[q], list[q], found[q], 1);
    wave_publish();  // the lanes of a vertex are one wave's
    if (i >= nv || sub != 0) return;
    int idx[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) idx[j] = j < kk ? min(found[q][j], n - 1) : 0;  // NaN coordinates: any point of the cloud
    float d[4] = {0.f, 0.f, 0.f, 0.f}, sum = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (j >= kk) continue;
        const float3 q = load_point(xyz, stride, idx[j]);
        const float tx = __fsub_rn(p.x, q.x), ty = __fsub_rn(p.y, q.y), tz = __fsub_rn(p.z, q.z);
        d[j] = __fadd_rn(__fadd_rn(__fmul_rn(tx, tx), __fmul_rn(ty, ty)), __fmul_rn(tz, tz));
        sum = __fadd_rn(sum, d[j]);
    }
    float w[4];
    const float inv = sum > 0.f ? __fdiv_rn(1.0f, sum) : 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = j >= kk ? 0.f : (sum > 0.f ? __fmul_rn(d[j], inv) : __fdiv_rn(1.0f, float(kk)));
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (j < kk) acc = __fadd_rn(acc, __fmul_rn(pc[3 * size_t(idx[j]) + a], w[j]));
        out[3 * size_t(i) + a] = acc;
    }
}

// Grid of the n points for exact nearest-neighbour searches: cell size from
// about k points per occupied surface cell; the points sorted by cell, with
// their indices (spos), and each cell's first sorted position (start, G^3 + 1
// entries).  Waits for nothing: the grid is computed on the device, and bounds
// that are not finite are reported through the mailbox (check_bounds).
void build_knn_grid(Ctx& c, const char* base, unsigned stride, int n, int k, GridSpec*& grid, float4*& spos,
                    int*& start) {
    hipStream_t s = c.stream;
    const int nb = std::min<int>(kBoundsBlocks, int(div_up(n, kThreads)));
    // Cells per axis: on a closed surface of area about 2-3 times the square of
    // its extent, 0.7 sqrt(n / k) makes the k-th distance about 0.55-0.7 of a
    // cell, so that the 27 cells nearly always hold the k nearest and not many
    // more.  At 200k points, k = 10 (torus / sphere): 230 / 206 us a call at
    // 0.6 sqrt(n / k), 188 / 190 at 0.7, 202 / 247 at 0.9 (searches repeat with
    // 125 cells), 222 / 284 at 1.  256 at most: 64 MB of cell starts.
    const int G = std::min(256, std::max(2, int(std::lround(0.7 * std::sqrt(double(n) / double(k))))));
    const unsigned cells = unsigned(G) * unsigned(G) * unsigned(G);
    int bits = 1;
    while ((cells - 1) >> bits) ++bits;
    // one block of the arena: a context's first call allocates once
    BlockParts parts;
    auto part_of = [&](size_t bytes) { return parts.add(bytes); };
    const size_t oPart = part_of(sizeof(float) * 6 * nb), oGrid = part_of(sizeof(GridSpec)), oKey = part_of(4 * size_t(n)),
                 oVal = part_of(4 * size_t(n)), oKt = part_of(4 * size_t(n)), oVt = part_of(4 * size_t(n)),
                 oPos = part_of(16 * size_t(n)), oSpos = part_of(16 * size_t(n)),
                 oStart = part_of(4 * (size_t(cells) + 1));
    char* block = c.buf<char>("ne_grid", parts.bytes);
    float* part = reinterpret_cast<float*>(block + oPart);
    grid = reinterpret_cast<GridSpec*>(block + oGrid);
    unsigned* key = reinterpret_cast<unsigned*>(block + oKey);
    unsigned* val = reinterpret_cast<unsigned*>(block + oVal);
    unsigned* kt = reinterpret_cast<unsigned*>(block + oKt);
    unsigned* vt = reinterpret_cast<unsigned*>(block + oVt);
    float4* pos = reinterpret_cast<float4*>(block + oPos);
    spos = reinterpret_cast<float4*>(block + oSpos);
    start = reinterpret_cast<int*>(block + oStart);
    c.hostPinned[kMailBounds] = 0;
    ne_bounds<<<nb, kThreads, 0, s>>>(base, stride, n, part);
    int* scratch = c.scratch_for(sort_scratch_ints(size_t(n)));
    const int tiles = int(div_up(n, kSortTileKeys));
    ne_cells<<<tiles, kThreads, 0, s>>>(base, stride, n, part, nb, G, grid, c.mail + kMailBounds, key, val, pos, tiles,
                                        scratch, (1u << sort_digit_bits(bits)) - 1u);
    radix_sort_pairs(key, val, kt, vt, n, bits, scratch, true, c.scan_for(sort_scan_elems(size_t(n))),
                     SortGather{pos, nullptr, spos, nullptr}, s);
    ne_cell_starts<<<div_up(size_t(cells) + 1, kStartCells), kThreads, 0, s>>>(key, n, cells, start);
}

// After the wait: the grid's points had finite bounds.
void check_bounds(const Ctx& c) {
    if (c.hostPinned[kMailBounds]) throw std::invalid_argument("non-finite point coordinates");
}

}  // namespace

void estimate_normals(Ctx& c, const float* xyz, int n, unsigned stride, int k, float3 vp, float* normals,
                      float* curvature, int* knn) {
    if (k < 1 || k > kMaxK) throw std::invalid_argument("k must lie in 1..16");
    if (n <= 0) return;
    const char* base = reinterpret_cast<const char*>(xyz);
    GridSpec* grid = nullptr;
    float4* spos = nullptr;
    int* start = nullptr;
    build_knn_grid(c, base, stride, n, k, grid, spos, start);
    // the list of distances is as long as k needs, in three lengths
    auto launch = [&](auto kernel) {
        kernel<<<div_up(n, kThreads / kFitLanes), kThreads, 0, c.stream>>>(base, stride, n, k, grid, spos, start, vp,
                                                                           normals, curvature, knn);
    };
    if (k <= 8) launch(ne_estimate<8, kFitLanes>);
    else if (k <= 10) launch(ne_estimate<10, kFitLanes>);
    else launch(ne_estimate<kMaxK, kFitLanes>);
    c.wait();
    PSR_HIP_CHECK(hipGetLastError());
    check_bounds(c);
}

void vertex_colors(Ctx& c, const float* V, int nv, const float* xyz, unsigned stride, const float* pc, int n,
                   float* out) {
    if (nv <= 0) return;
    if (n <= 0) throw std::invalid_argument("no points to colour from");
    const char* base = reinterpret_cast<const char*>(xyz);
    GridSpec* grid = nullptr;
    float4* spos = nullptr;
    int* start = nullptr;
    build_knn_grid(c, base, stride, n, 10, grid, spos, start);  // cells sized as for 10 (the search is exact for 4)
    vc_colors<kColorLanes><<<div_up(nv, kThreads / kColorLanes), kThreads, 0, c.stream>>>(V, nv, base, stride, n, pc,
                                                                                           grid, spos, start, out);
    c.wait();
    PSR_HIP_CHECK(hipGetLastError());
    check_bounds(c);
}

}  // namespace psr
