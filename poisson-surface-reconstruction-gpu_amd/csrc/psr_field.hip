// Basis inner-product tables, vector-field splat and divergence.
#include "psr_internal.h"

#include <hip/hip_fp16.h>

#include <algorithm>
#include <cmath>
#include <vector>

namespace psr {

namespace {

// --- 1-D tables (FunctionData::setDotTables, mesh/FunctionData.h:134-190) ---
// Exact FP64 integrals over the real line of products of the scaled/shifted
// quadratic B-spline and its derivative, one thread per (a, b) entry:
//   dot[a + res b]   = <F_a,  F_b>
//   ddot[a + res b]  = <F_a', F_b>
//   d2dot[a + res b] = <F_a', F_b'>
// and ddotT, ddot transposed: the divergence of a node reads one row of it.
// Each product is a polynomial of degree <= 4 between breakpoints; 3-point
// Gauss-Legendre per piece integrates it exactly.
__device__ double bsp_d(double u) {
    u = fabs(u);
    if (u < 0.5) return 1.0 - (4.0 / 3.0) * u * u;
    if (u < 1.5) return (2.0 / 3.0) * (1.5 - u) * (1.5 - u);
    return 0.0;
}
__device__ double bsp_deriv(double u) {
    if (u <= -1.5 || u >= 1.5) return 0.0;
    if (u < -0.5) return (4.0 / 3.0) * (1.5 + u);
    if (u < 0.5) return -(8.0 / 3.0) * u;
    return -(4.0 / 3.0) * (1.5 - u);
}
__device__ void cw_of(int idx, double& c, double& w) {
    int depth = 31 - __clz(idx + 1);
    int off = idx + 1 - (1 << depth);
    w = 1.0 / double(1 << depth);
    c = (0.5 + off) * w;
}

__global__ void __launch_bounds__(256) build_tables_kernel(int res, double* __restrict__ dot,
                                                           double* __restrict__ ddot, double* __restrict__ ddotT,
                                                           double* __restrict__ d2dot) {
    long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    if (t >= (long long)res * res) return;
    int a = int(t % res), b = int(t / res);
    double ca, wa, cb, wb;
    cw_of(a, ca, wa);
    cw_of(b, cb, wb);
    double lo = fmax(ca - 1.5 * wa, cb - 1.5 * wb), hi = fmin(ca + 1.5 * wa, cb + 1.5 * wb);
    double r0 = 0, r1 = 0, r2 = 0;
    if (lo < hi) {
        double br[6];
        int nb = 0;
        br[nb++] = lo;
        double cand[4] = {ca - 0.5 * wa, ca + 0.5 * wa, cb - 0.5 * wb, cb + 0.5 * wb};
        for (int k = 0; k < 4; ++k)
            if (cand[k] > lo && cand[k] < hi) br[nb++] = cand[k];
        br[nb++] = hi;
        for (int i = 1; i < nb; ++i)  // insertion sort, <= 6 entries
            for (int j = i; j > 0 && br[j - 1] > br[j]; --j) {
                double x = br[j];
                br[j] = br[j - 1];
                br[j - 1] = x;
            }
        const double gx[3] = {-0.77459666924148337704, 0.0, 0.77459666924148337704};
        const double gw[3] = {5.0 / 9.0, 8.0 / 9.0, 5.0 / 9.0};
        for (int k = 0; k + 1 < nb; ++k) {
            double x0 = br[k], x1 = br[k + 1];
            if (!(x1 > x0)) continue;
            double h = 0.5 * (x1 - x0), m = 0.5 * (x1 + x0);
            for (int g = 0; g < 3; ++g) {
                double x = m + h * gx[g];
                double ua = (x - ca) / wa, ub = (x - cb) / wb;
                double fa = bsp_d(ua), fb = bsp_d(ub);
                double da = bsp_deriv(ua) / wa, db = bsp_deriv(ub) / wb;
                double wg = gw[g] * h;
                r0 += wg * fa * fb;
                r1 += wg * da * fb;
                r2 += wg * da * db;
            }
        }
        if (fabs(r0) < 1e-15) r0 = r1 = r2 = 0;  // FunctionData.h:172
    }
    dot[t] = r0;
    ddot[t] = r1;
    ddotT[size_t(a) * res + b] = r1;
    d2dot[t] = r2;
}

// band[k * res + f] = (dot, d2dot) of functions f and f + k - 1, where both
// belong to one depth.
__global__ void __launch_bounds__(256) gather_band(int res, int D, const double* __restrict__ dot,
                                                   const double* __restrict__ d2dot, double2* __restrict__ band) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= 3 * res) return;
    const int k = t / res, f = t - k * res, g = f + k - 1;
    const int d = 31 - __clz(f + 1);
    const bool in = g >= (1 << d) - 1 && g < (2 << d) - 1;
    const size_t at = size_t(f) * res + size_t(in ? g : f);
    band[t] = in ? make_double2(dot[at], d2dot[at]) : make_double2(0.0, 0.0);
}

// Concatenated ranges of the 27 neighbours of a node, held in LDS per wave.
struct NbRanges {
    int start[28];
    int first[27];
};

// Fills r for node o with range (first, len) per neighbour; returns total.
template <class LenFn>
__device__ __forceinline__ int wave_ranges(NbRanges& r, const int* __restrict__ neigh, int M, int o, int lane,
                                           LenFn fn) {
    int nb = -1, len = 0, first = 0;
    if (lane < 27) {
        nb = neigh[lane * M + o];
        if (nb != -1) fn(nb, first, len);
    }
    int inc = len;
    for (int off = 1; off < PSR_WAVE; off <<= 1) {
        int t = __shfl_up(inc, off, PSR_WAVE);
        if (lane >= off) inc += t;
    }
    if (lane < 27) {
        r.start[lane] = inc - len;
        r.first[lane] = first;
    }
    int total = __shfl(inc, 26, PSR_WAVE);
    if (lane == 0) r.start[27] = total;
    return total;
}

// wave_ranges for two nodes, one per half-wave (hl: the lane within the half;
// an invalid node has no range).
template <class LenFn>
__device__ __forceinline__ int half_ranges(NbRanges& r, const int* __restrict__ neigh, int M, int o, int hl,
                                           bool valid, LenFn fn) {
    constexpr int kHalf = PSR_WAVE / 2;
    int len = 0, first = 0;
    if (valid && hl < 27) {
        const int nb = neigh[hl * M + o];
        if (nb != -1) fn(nb, first, len);
    }
    int inc = len;
    for (int off = 1; off < kHalf; off <<= 1) {
        const int t = __shfl_up(inc, off, kHalf);
        if (hl >= off) inc += t;
    }
    if (hl < 27) {
        r.start[hl] = inc - len;
        r.first[hl] = first;
    }
    const int total = __shfl(inc, 26, kHalf);
    if (hl == 0) r.start[27] = total;
    return total;
}

__device__ __forceinline__ int range_of(const NbRanges& r, int t) {
    int i = 0;
    for (int step = 16; step > 0; step >>= 1)
        if (i + step < 28 && r.start[i + step] <= t) i += step;
    return i;
}

// --- vector field (ComputeVectorField.cu:61-100) ---------------------------
// V(o) = sum over the 27 neighbours' points p of F_o(x)F_o(y)F_o(z) n_p,
// two depth-D nodes per wave, one per half: a node's chain of dependent loads
// (neighbours, their point ranges, the points) is latency-bound, and the two
// chains of a wave overlap.
// Field storage, a vector per node: FP32, or FP16 holding V * 2^-(D+1) (the
// normals' scale, an exact power of two, so the stored value is the FP16
// rounding of the sum of weighted unit normals); the divergence reads a vector
// with one load (FieldHalf, float4: the fourth component is unused).
__device__ __forceinline__ void store_field(float4* p, float3 v, float) { *p = make_float4(v.x, v.y, v.z, 0.f); }
__device__ __forceinline__ void store_field(FieldHalf* p, float3 v, float invScale) {
    *p = FieldHalf{__float2half_rn(v.x * invScale), __float2half_rn(v.y * invScale), __float2half_rn(v.z * invScale),
                   __half(0.f)};
}
__device__ __forceinline__ float3 load_field(const float4* p, float) {
    const float4 v = *p;
    return make_float3(v.x, v.y, v.z);
}
__device__ __forceinline__ float3 load_field(const FieldHalf* p, float scale) {
    const FieldHalf v = *p;
    return make_float3(__half2float(v.x) * scale, __half2float(v.y) * scale, __half2float(v.z) * scale);
}

constexpr int kVfWaves = 4;
template <class FieldT>
__device__ __forceinline__ void vector_field_kernel_body(int psr_bid, int psr_nbid, 
    int nD, int offD, int M, int D, const int* __restrict__ neigh, const int* __restrict__ pidx,
    const int* __restrict__ pnum, const int* __restrict__ key, const float4* __restrict__ pos,
    const float4* __restrict__ nrm, FieldT* __restrict__ vf, int* __restrict__ clear) {
    // the operator's per-depth entry counts and slot masks, which the
    // divergence launch's assembly adds to, and the CG error flag between
    // them in the results block
    if (psr_bid == 0 && threadIdx.x < kResultsClearWords) clear[threadIdx.x] = 0;
    __shared__ NbRanges R[kVfWaves][2];
    constexpr int kHalf = PSR_WAVE / 2;
    const int wid = threadIdx.x / PSR_WAVE, lane = __lane_id(), half = lane / kHalf, hl = lane % kHalf;
    const int node0 = (psr_bid * kVfWaves + wid) * 2;
    if (node0 >= nD) return;
    const int node = node0 + half;
    const bool valid = node < nD;
    const int o = offD + (valid ? node : node0);
    NbRanges& r = R[wid][half];
    const int total = half_ranges(r, neigh, M, o, hl, valid, [&](int nb, int& first, int& len) {
        first = pidx[nb];
        len = pnum[nb];
    });
    __builtin_amdgcn_wave_barrier();
    int3 f = key_func_index(key[o], D, D);
    float cx, cy, cz, invw;
    func_center_invw(f.x, cx, invw);
    func_center_invw(f.y, cy, invw);
    func_center_invw(f.z, cz, invw);
    float ax = 0.f, ay = 0.f, az = 0.f;
    for (int t = hl; t < total; t += kHalf) {
        int i = range_of(r, t);
        int p = r.first[i] + (t - r.start[i]);
        float4 q = pos[p];
        float4 n = nrm[p];
        float w = bspline((q.x - cx) * invw) * bspline((q.y - cy) * invw) * bspline((q.z - cz) * invw);
        ax += w * n.x;
        ay += w * n.y;
        az += w * n.z;
    }
    ax = half_sum_f32(ax, half);
    ay = half_sum_f32(ay, half);
    az = half_sum_f32(az, half);
    if (hl == 0 && valid) {
        store_field(&vf[node], make_float3(ax, ay, az), 1.0f / float(2 << D));
    }
}
template <class FieldT>
__global__ void __launch_bounds__(kVfWaves * PSR_WAVE) vector_field_kernel(
    int nD, int offD, int M, int D, const int* __restrict__ neigh, const int* __restrict__ pidx,
    const int* __restrict__ pnum, const int* __restrict__ key, const float4* __restrict__ pos,
    const float4* __restrict__ nrm, FieldT* __restrict__ vf, int* __restrict__ clear) {
    vector_field_kernel_body<FieldT>(xcd_block(blockIdx.x, gridDim.x), gridDim.x, nD, offD, M, D, neigh, pidx, pnum, key, pos, nrm, vf, clear);
}
template <class FieldT>
struct vector_field_kernel_k {
    static constexpr int kBlock = kVfWaves * PSR_WAVE;
    template <class... A>
    __device__ __forceinline__ static void run(int bid, int nbid, const A&... a) { vector_field_kernel_body<FieldT>(bid, nbid, a...); }
};


// --- divergence (ComputeNodesDivergence.cu:25-136) -------------------------
// b(o) = sum over the 27 neighbours' depth-D descendants j of
//        V_j . (<F'_ox, F_jx>, <F'_oy, F_jy>, <F'_oz, F_jz>)     (reference Q3)
// The rows of ddotT of a node's three functions: F_j's values lie beside those of
// its neighbours, where a column of ddot has a cache line for each.
struct DivRows {
    const double *x, *y, *z;
    __device__ __forceinline__ DivRows(const double* ddotT, int res, int3 fo)
        : x(ddotT + size_t(fo.x) * res), y(ddotT + size_t(fo.y) * res), z(ddotT + size_t(fo.z) * res) {}
};
template <class FieldT>
__device__ __forceinline__ double div_term(int j, int offD, int D, const DivRows& rows, const int* __restrict__ enc,
                                           const FieldT* __restrict__ vf) {
    const int3 fj = decode_func_index(enc[offD + j], D);
    const float3 v = load_field(&vf[j], float(2 << D));
    double s = double(v.x) * rows.x[fj.x];
    s += double(v.y) * rows.y[fj.y];
    s += double(v.z) * rows.z[fj.z];
    return s;
}

constexpr int kDivWaves = 4;
// The wave's three rows are copied to LDS where they are short (a term's table
// values are three scattered 8-byte reads, which bound the kernel from the cache;
// its vector and index are contiguous).  The launch with this, one load a vector
// and the leaves' 9 table values: 200k torus at depth 7 51 -> 38 us, 20k sphere at
// depth 6 25 -> 16 us, 300k points at depth 8 163 -> 141 us, 32 clouds 1141 -> 980.
constexpr int kDivRow = 96;  // functions an axis kept in LDS: up to 5 levels above depth D
template <class FieldT>
__device__ __forceinline__ void divergence_fine_body(int psr_bid, int psr_nbid, 
    int begin, int count, int M, int offD, int nD, int res, int D, const int* __restrict__ neigh,
    const int* __restrict__ didx, const int* __restrict__ dnum, const int* __restrict__ enc,
    const FieldT* __restrict__ vf, const double* __restrict__ ddotT, const int* __restrict__ q1Fired,
    float* __restrict__ div) {
    // (two nodes per wave, as the vector field splats them, measured 64%
    // slower here: a node at depth 4 or 5 has hundreds to thousands of terms)
    __shared__ NbRanges ranges[kDivWaves];
    __shared__ double rowStore[kDivWaves][3 * kDivRow];
    int wid = threadIdx.x / PSR_WAVE, lane = __lane_id();
    int node = psr_bid * kDivWaves + wid;
    if (node >= count) return;
    int o = begin + node;
    NbRanges& r = ranges[wid];
    double* tab = rowStore[wid];
    int total = wave_ranges(r, neigh, M, o, lane, [&](int nb, int& first, int& len) {
        first = didx[nb];
        len = dnum[nb];
    });
    __builtin_amdgcn_wave_barrier();
    const int3 fo = decode_func_index(enc[o], D);
    const DivRows rows(ddotT, res, fo);
    double acc = 0;
    // on the regular grid the descendants' functions are those of the node's cell
    // and the cells beside it, 3 2^(D - d) an axis
    const int d = 31 - __clz(fo.x + 1), k = D - d, R = 3 << k;
    if (*q1Fired == 0 && R <= kDivRow) {
        int f0[3];
        const int f[3] = {fo.x, fo.y, fo.z};
        const double* g[3] = {rows.x, rows.y, rows.z};
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            f0[a] = (1 << D) - 1 + (f[a] - (1 << d)) * (1 << k);  // the first of the cell below
            for (int u = lane; u < R; u += PSR_WAVE) tab[a * kDivRow + u] = g[a][min(max(f0[a] + u, 0), res - 1)];
        }
        __builtin_amdgcn_wave_barrier();
        for (int t = lane; t < total; t += PSR_WAVE) {
            const int i = range_of(r, t), j = r.first[i] + (t - r.start[i]);
            const int3 fj = decode_func_index(enc[offD + j], D);
            const float3 v = load_field(&vf[j], float(2 << D));
            double s = double(v.x) * tab[fj.x - f0[0]];
            s += double(v.y) * tab[kDivRow + fj.y - f0[1]];
            s += double(v.z) * tab[2 * kDivRow + fj.z - f0[2]];
            acc += s;
        }
    } else {
        for (int t = lane; t < total; t += PSR_WAVE) {
            int i = range_of(r, t);
            acc += div_term(r.first[i] + (t - r.start[i]), offD, D, rows, enc, vf);
        }
    }
    acc = wave_sum_f64(acc);
    if (lane == 0) div[o] = float(acc);
}


// A coarse node's share of workgroup `part` (CoarsePlan; folded by divergence_fold).
constexpr int kDivCoarseThreads = 256;
template <class FieldT>
__device__ __forceinline__ void divergence_coarse_body(int psr_bid, int psr_nbid, 
    const CoarsePlan& P, int M, int offD, int nD, int res, int D, const int* __restrict__ neigh,
    const int* __restrict__ didx, const int* __restrict__ dnum, const int* __restrict__ enc,
    const FieldT* __restrict__ vf, const double* __restrict__ ddotT, double* __restrict__ partial) {
    int d = 0;
    while (d + 1 < P.depths && int(psr_bid) >= P.blockStart[d + 1]) ++d;
    const int parts = P.parts[d];
    const int rel = psr_bid - P.blockStart[d];
    const int node = rel / parts, part = rel - node * parts;
    const int o = P.base[d] + node;
    __shared__ int start[28], first[27];
    __shared__ double red[kDivCoarseThreads / PSR_WAVE];
    if (threadIdx.x == 0) {
        int s = 0;
        for (int i = 0; i < 27; ++i) {
            int nb = neigh[i * M + o];
            start[i] = s;
            first[i] = nb != -1 ? didx[nb] : 0;
            s += nb != -1 ? dnum[nb] : 0;
        }
        start[27] = s;
    }
    __syncthreads();
    const int total = start[27];
    const DivRows rows(ddotT, res, decode_func_index(enc[o], D));
    double acc = 0;
    int i = 0;
    for (int t = part * kDivCoarseThreads + threadIdx.x; t < total; t += parts * kDivCoarseThreads) {
        while (start[i + 1] <= t) ++i;
        acc += div_term(first[i] + (t - start[i]), offD, D, rows, enc, vf);
    }
    acc = wave_sum_f64(acc);
    if (__lane_id() == 0) red[threadIdx.x / PSR_WAVE] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0;
        for (int w = 0; w < kDivCoarseThreads / PSR_WAVE; ++w) s += red[w];
        partial[psr_bid] = s;
    }
}
// Depth-D nodes: their neighbours are depth-D nodes, each its own only
// descendant, so a thread sums the 27 terms of its node.  On the regular grid
// neighbour i's functions are the node's own shifted by its offset, so that the
// 81 table values are 9 and no neighbour's index is read.
template <class FieldT>
__device__ __forceinline__ void divergence_leaf_nodes(int block, int offD, int nD, int M, int res, int D,
                                                      const int* __restrict__ neigh, const int* __restrict__ enc,
                                                      const FieldT* __restrict__ vf,
                                                      const double* __restrict__ ddotT,
                                                      const int* __restrict__ q1Fired, float* __restrict__ div) {
    const int t = block * 256 + threadIdx.x;
    if (t >= nD) return;
    const int o = offD + t;
    const int3 fo = decode_func_index(enc[o], D);
    const DivRows rows(ddotT, res, fo);
    double acc = 0;
    if (*q1Fired == 0 && neigh[13 * M + o] == o) {
        const float sc = float(2 << D);
        double wy[3], wz[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {  // past the domain: not used
            wy[k] = rows.y[min(max(fo.y + k - 1, 0), res - 1)];
            wz[k] = rows.z[min(max(fo.z + k - 1, 0), res - 1)];
        }
#pragma unroll 1
        for (int x = 0; x < 3; ++x) {  // nine neighbours' loads in flight (27 take 12 more registers)
            const double wx = rows.x[min(max(fo.x + x - 1, 0), res - 1)];
            int nb[9];
            float3 v[9];
#pragma unroll
            for (int i = 0; i < 9; ++i) nb[i] = neigh[(9 * x + i) * M + o];
#pragma unroll
            for (int i = 0; i < 9; ++i) v[i] = load_field(&vf[nb[i] != -1 ? nb[i] - offD : 0], sc);
#pragma unroll
            for (int i = 0; i < 9; ++i) {
                // rounded as div_term rounds it: y's product by itself, the other two fused onto it (here the
                // compiler would choose x's, and one value in 170k differ in its last bit)
                double p = double(v[i].y) * wy[i / 3];
                asm("" : "+v"(p));
                double s = p + double(v[i].x) * wx;
                s += double(v[i].z) * wz[i % 3];
                if (nb[i] != -1) acc += s;
            }
        }
    } else {
#pragma unroll 1
        for (int x = 0; x < 3; ++x) {
            int nb[9];
#pragma unroll
            for (int i = 0; i < 9; ++i) nb[i] = neigh[(9 * x + i) * M + o];
#pragma unroll
            for (int i = 0; i < 9; ++i)
                if (nb[i] != -1) acc += div_term(nb[i] - offD, offD, D, rows, enc, vf);
        }
    }
    div[o] = float(acc);
}

// Every depth in one launch, each role a range of 256-thread workgroups: the
// coarse nodes' shares, a middle-depth node per wave, a depth-D node per
// thread, and the operator's assembly (assemble_rows).  They read only the
// vector field, the octree and the tables and write disjoint outputs, so the
// roles fill the GPU side by side instead of one launch after another; the
// coarse shares are folded by divergence_fold.
struct DivRoles {
    int coarseBlocks, midBlocks, leafBlocks;
};
static_assert(kDivCoarseThreads == kDivWaves * PSR_WAVE && kAssembleThreads == kDivCoarseThreads,
              "one block size for every role");
template <class FieldT>
__device__ __forceinline__ void divergence_all_body(int psr_bid, int psr_nbid, const CoarsePlan& P, const DivRoles& R,
                                                    int begin, int count, int M, int offD, int nD, int res, int D,
                                                    const int* __restrict__ neigh, const int* __restrict__ didx,
                                                    const int* __restrict__ dnum, const int* __restrict__ enc,
                                                    const FieldT* __restrict__ vf, const double* __restrict__ ddotT,
                                                    double* __restrict__ partial, float* __restrict__ div,
                                                    const AssembleArgs& aa) {
    int b = psr_bid;
    if (b < R.coarseBlocks) {
        divergence_coarse_body<FieldT>(b, R.coarseBlocks, P, M, offD, nD, res, D, neigh, didx, dnum, enc, vf, ddotT,
                                       partial);
        return;
    }
    b -= R.coarseBlocks;
    if (b < R.midBlocks) {
        divergence_fine_body<FieldT>(b, R.midBlocks, begin, count, M, offD, nD, res, D, neigh, didx, dnum, enc, vf,
                                     ddotT, aa.q1Fired, div);
        return;
    }
    b -= R.midBlocks;
    if (b < R.leafBlocks) {
        divergence_leaf_nodes<FieldT>(b, offD, nD, M, res, D, neigh, enc, vf, ddotT, aa.q1Fired, div);
        return;
    }
    assemble_rows(aa, b - R.leafBlocks);
}
template <class FieldT>
__global__ void __launch_bounds__(kDivCoarseThreads) divergence_all(
    CoarsePlan P, DivRoles R, int begin, int count, int M, int offD, int nD, int res, int D,
    const int* __restrict__ neigh, const int* __restrict__ didx, const int* __restrict__ dnum,
    const int* __restrict__ enc, const FieldT* __restrict__ vf, const double* __restrict__ ddotT,
    double* __restrict__ partial, float* __restrict__ div, AssembleArgs aa) {
    divergence_all_body<FieldT>(blockIdx.x, gridDim.x, P, R, begin, count, M, offD, nD, res, D, neigh, didx, dnum, enc,
                                vf, ddotT, partial, div, aa);
}
template <class FieldT>
struct divergence_all_k {
    static constexpr int kBlock = kDivCoarseThreads;
    template <class... A>
    __device__ __forceinline__ static void run(int bid, int nbid, const A&... a) { divergence_all_body<FieldT>(bid, nbid, a...); }
};

}  // namespace

void build_tables(Ctx& c) {
    const int D = c.cfg.depth;
    const int res = (1 << (D + 1)) - 1;
    Tables& t = c.tables;
    t.res = res;
    size_t n = size_t(res) * res;
    const int functions = res;  // of all depths
    std::vector<float> weights(27 * size_t(D + 1), 0.f);
    BlockParts parts;
    const size_t oDot = parts.add(sizeof(double) * n), oDdot = parts.add(sizeof(double) * n), oDdotT = parts.add(sizeof(double) * n),
                 oD2dot = parts.add(sizeof(double) * n), oBand = parts.add(sizeof(double2) * 3 * functions),
                 oWeights = parts.add(sizeof(float) * weights.size());
    char* block = c.buf<char>("tables", parts.bytes);
    t.dot = reinterpret_cast<double*>(block + oDot);
    t.ddot = reinterpret_cast<double*>(block + oDdot);
    t.ddotT = reinterpret_cast<double*>(block + oDdotT);
    t.d2dot = reinterpret_cast<double*>(block + oD2dot);
    build_tables_kernel<<<div_up(n, 256), 256, 0, c.stream>>>(res, t.dot, t.ddot, t.ddotT, t.d2dot);
    PSR_HIP_CHECK(hipGetLastError());
    // The inner products of each depth's functions with those at offsets -1, 0
    // and 1 (a depth's functions are consecutive), copied out in one piece.
    double2* band = reinterpret_cast<double2*>(block + oBand);
    gather_band<<<div_up(size_t(3) * functions, 256), 256, 0, c.stream>>>(res, D, t.dot, t.d2dot, band);
    std::vector<double2> hb(size_t(3) * functions);
    PSR_HIP_CHECK(hipMemcpyAsync(hb.data(), band, sizeof(double2) * hb.size(), hipMemcpyDeviceToHost, c.stream));
    PSR_HIP_CHECK(hipStreamSynchronize(c.stream));
    // The operator's entry of every depth and offset: the inner products at one
    // offset differ from function to function in their last bits only, and the
    // entry rounds to one float for every triple of them or the depth has no
    // table of entries.
    bool unique = true;
    for (int d = 0; d <= D; ++d) {
        std::vector<double2> distinct[3];
        for (int k = 0; k < 3; ++k) {
            for (int f = (1 << d) - 1; f < (2 << d) - 1; ++f) {
                const int g = f + k - 1;
                if (g < (1 << d) - 1 || g >= (2 << d) - 1) continue;
                const double2 v = hb[size_t(k) * functions + f];
                bool seen = false;
                for (const double2& q : distinct[k]) seen = seen || (q.x == v.x && q.y == v.y);
                if (!seen) distinct[k].push_back(v);
            }
        }
        for (int q = 0; q < 27; ++q) {
            bool first = true;
            for (const double2& x : distinct[q / 9])
                for (const double2& y : distinct[(q / 3) % 3])
                    for (const double2& z : distinct[q % 3]) {
                        const float e = operator_entry(x.x, y.x, z.x, x.y, y.y, z.y);
                        if (first) weights[27 * size_t(d) + q] = e;
                        else unique = unique && e == weights[27 * size_t(d) + q];
                        first = false;
                    }
        }
    }
    if (unique) {
        t.weights = reinterpret_cast<float*>(block + oWeights);
        PSR_HIP_CHECK(hipMemcpyAsync(t.weights, weights.data(), sizeof(float) * weights.size(), hipMemcpyHostToDevice, c.stream));
        PSR_HIP_CHECK(hipStreamSynchronize(c.stream));
    }
    // Which depths' operators are indefinite once entries with |L| <= 1e-6 are
    // dropped (LaplacianSolver.cu:62).  An entry depends only on the neighbour
    // offset (the inner products are shift-invariant inside the domain), so a
    // depth's operator is a constant 27-point stencil; its symbol
    // sum_o L_o cos(theta . o), sampled over [0, pi]^3, takes both signs
    // exactly when the operator has eigenvalues of both signs on large
    // interiors.  At depth 9 only the diagonal and the six face entries
    // survive and the symbol at (pi, pi, pi) is negative.
    for (int d = 2; d <= D; ++d) {
        const int f = (1 << d) - 1 + (1 << (d - 1));  // an interior function of depth d
        double dt[2], d2[2];
        for (int k = 0; k < 2; ++k) {
            dt[k] = hb[size_t(1 + k) * functions + f].x;
            d2[k] = hb[size_t(1 + k) * functions + f].y;
        }
        double L[2][2][2];  // by |offset| per axis
        for (int a = 0; a < 2; ++a)
            for (int b = 0; b < 2; ++b)
                for (int e = 0; e < 2; ++e) {
                    const double v = dt[a] * dt[b] * dt[e] * (d2[a] + d2[b] + d2[e]);
                    L[a][b][e] = std::fabs(v) > double(1e-6f) ? v : 0.0;
                }
        constexpr int S = 32;
        double lo = 1e300;
        for (int i = 0; i <= S; ++i)
            for (int j = 0; j <= S; ++j)
                for (int k = 0; k <= S; ++k) {
                    // cos(theta o) summed over o = -1, 0, 1 per axis: 1 for |o| = 0, 2 cos theta for |o| = 1
                    const double cx[2] = {1.0, 2.0 * std::cos(M_PI * i / S)};
                    const double cy[2] = {1.0, 2.0 * std::cos(M_PI * j / S)};
                    const double cz[2] = {1.0, 2.0 * std::cos(M_PI * k / S)};
                    double sym = 0;
                    for (int a = 0; a < 2; ++a)
                        for (int b = 0; b < 2; ++b)
                            for (int e = 0; e < 2; ++e) sym += L[a][b][e] * cx[a] * cy[b] * cz[e];
                    lo = std::min(lo, sym);
                }
        c.indefinite[d] = lo < 0;
    }
}

namespace {

template <class FieldT>
void field_stages(Ctx& c, FieldT* vf) {
    Octree& o = c.oct;
    const Levels& L = o.L;
    const int D = L.D, nD = L.count[D], offD = L.base[D], M = o.M;
    hipStream_t s = c.stream;
    PSR_LAUNCH_K(vector_field_kernel<FieldT>, vector_field_kernel_k<FieldT>,
        std::max<size_t>(1, div_up(nD, 2 * kVfWaves)), 0, s,
        nD, offD, M, D, o.neigh, o.pidx, o.pnum, o.key, o.spos, o.snrm, vf, c.results()->cgNnz);
    // depths 0..kCoarse: several workgroups per node, per depth as many as the
    // node's expected share of depth D asks for; depth D: a thread per node;
    // between: a wave per node
    const int kCoarse = D >= 5 ? kMaxCoarse - 1 : 1;
    const int coarseCount = L.base[kCoarse + 1];
    CoarsePlan P{};
    double* partial = nullptr;
    {
        P.depths = kCoarse + 1;
        int blocks = 0;
        for (int d = 0; d <= kCoarse; ++d) {
            const double share = std::min(double(nD), 27.0 * nD / std::max(1, L.count[d]));
            P.parts[d] = std::max(1, std::min(64, int(share / 2048.0)));
            P.blockStart[d] = blocks;
            P.base[d] = L.base[d];
            blocks += P.parts[d] * L.count[d];
        }
        P.blockStart[kCoarse + 1] = blocks;
        P.base[kCoarse + 1] = L.base[kCoarse + 1];
        partial = c.buf<double>("div_partial", blocks);
    }
    // every depth's divergence and the operator's assembly (it needs only the
    // octree and the tables) in one launch
    const int midCount = std::max(offD - coarseCount, 0);
    const DivRoles R{P.blockStart[kCoarse + 1], int(div_up(midCount, kDivWaves)), int(div_up(nD, 256))};
    const AssembleArgs aa{L,     M,     o.neigh, o.encIdx, c.tables.dot, c.tables.d2dot, c.tables.res,
                          c.buf<float>("lap_val", size_t(27) * M), c.results()->cgNnz, c.results()->cgSlotMask,
                          c.tables.weights, o.q1Fired};
    const int assembleBlocks = int(div_up(size_t(3) * M, kAssembleThreads));
    PSR_LAUNCH_K(divergence_all<FieldT>, divergence_all_k<FieldT>,
                 R.coarseBlocks + R.midBlocks + R.leafBlocks + assembleBlocks, 0, s, P, R, coarseCount, midCount, M,
                 offD, nD, c.tables.res, D, o.neigh, o.didx, o.dnum, o.encIdx, vf, c.tables.ddotT, partial, c.fld.div,
                 aa);
    c.fld.foldArgs = DivFoldArgs{P, partial, c.fld.div};  // run by the solve's first kernel (solve_depths)
    PSR_HIP_CHECK(hipGetLastError());
}

}  // namespace

void compute_field(Ctx& c) {
    const Levels& L = c.oct.L;
    const int nD = L.count[L.D];
    c.fld.div = c.buf<float>("divergence", c.oct.M);
    if (c.cfg.precision == PSR_PRECISION_MIXED) {
        c.fld.vfield = nullptr;
        c.fld.vhalf = c.buf<FieldHalf>("vfield_half", nD);
        field_stages(c, c.fld.vhalf);
    } else {
        c.fld.vhalf = nullptr;
        c.fld.vfield = c.buf<float4>("vfield", nD);
        field_stages(c, c.fld.vfield);
    }
}

}  // namespace psr
