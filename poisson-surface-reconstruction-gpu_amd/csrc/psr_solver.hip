// Per-depth Laplacian, concurrent CG over all depths, implicit function at the
// input points and the iso-value.
#include "psr_internal.h"

#include <algorithm>
#include <mutex>
#include <chrono>
#include <stdexcept>
#include <thread>
#include <type_traits>
#include <vector>

namespace psr {

namespace {

constexpr int kThreads = 256;

// --- concurrent CG (CGAlgorithm.cu:10-147, 296-408) -------------------------
// Work item = a range of rows of one depth.  All work items of a depth form a
// group that iterates in lock step through a bounded-spin group barrier; a
// group of one workgroup uses __syncthreads only.
struct CgGroup {
    int depth;
    int rowBegin;   // global node index of the depth's first row
    int rows;
    int firstWg;    // first workgroup of the group
    int wgs;        // workgroups in the group
    int rowsPerWg;
    int indef;      // mixed form: the depth's operator is indefinite, solved with MINRES
};

struct CgParams {
    int ngroups;
    CgGroup g[PSR_MAX_DEPTH + 1];
    int M;
    float tolSq;     // reference: r1 > tol * tol with float tol (CGAlgorithm.cu:36)
    int maxIter;
    unsigned spinLimit;
    double relTol;   // mixed form: target ||b - A x|| / ||b|| per depth
    int maxOuter;    // mixed form: refinement steps
};

constexpr int kCgThreads = 256;
constexpr int kCgWaves = kCgThreads / PSR_WAVE;
// The FP32 generic form is compiled for 4 waves per SIMD (its persistent
// launch's resident budget follows from that occupancy; 21% faster sweeps at
// depth 9 than at 2), the mixed generic CG for 3.
constexpr int kCgFp32GenericWaves = 4, kCgMixedGenericWaves = 3;
// The MINRES kernel (indefinite depths of the mixed form) carries only its
// own path and is compiled for 4 waves per SIMD.  Its occupancy (5) also sets
// the row blocks of the on-chip form, whose sums follow them.
constexpr int kCgMinresWaves = 4;
// The mixed form's inner CG ends when its residual has not reached a new
// minimum for this many iterations, and its solution goes back to the
// iterate of the smallest residual.  A definite depth converges long before
// (20-70 iterations here); an operator that the reference's neighbour rules
// leave nonsymmetric or singular at a coarse depth (seen on ellipsoids of the
// 64-cloud batch) lets CG wander without converging, and the FP64 oracle's
// own CG diverges there.
constexpr int kCgStall = 128;

// Vectors read by other workgroups (r, p) and the reduction partials are
// accessed with agent-scope relaxed atomics, which are coherent across the
// XCDs without flushing or invalidating the L2; the barrier then only has to
// order them (s_waitcnt) before the arrival.
__device__ __forceinline__ float ld_shared(const float* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_shared(float* p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Orders a wave's LDS and memory writes before its later reads of other
// lanes' values: the steps of a group that fits one wave need no workgroup
// barrier.
__device__ __forceinline__ void wave_sync_memory() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

__device__ __forceinline__ double block_sum_double(double v, double* sh) {
    v = wave_sum_f64(v);
    int w = threadIdx.x / PSR_WAVE;
    if (__lane_id() == 0) sh[w] = v;
    __syncthreads();
    double s = 0;
    for (int k = 0; k < kCgWaves; ++k) s += sh[k];
    __syncthreads();
    return s;
}

// Per-group control block; each group's counters sit on their own cache lines.
struct GroupCtl {
    unsigned cnt;         // arrivals, monotonic: phase p is complete at p * workgroups
    unsigned pad0[31];
    unsigned gen;         // last phase whose total has been published
    unsigned pad1[31];
    unsigned res[2][32];  // published totals by phase parity
};
static_assert(sizeof(GroupCtl) == 512, "GroupCtl layout");

template <class T>
__device__ __forceinline__ void st_agent(T* p, const T& v) {
    static_assert(sizeof(T) % 4 == 0, "word-sized values");
    const unsigned* s = reinterpret_cast<const unsigned*>(&v);
    unsigned* d = reinterpret_cast<unsigned*>(p);
#pragma unroll
    for (int k = 0; k < int(sizeof(T) / 4); ++k) __hip_atomic_store(&d[k], s[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ T ld_agent(const T* p) {
    T v;
    unsigned* d = reinterpret_cast<unsigned*>(&v);
    const unsigned* s = reinterpret_cast<const unsigned*>(p);
#pragma unroll
    for (int k = 0; k < int(sizeof(T) / 4); ++k) d[k] = __hip_atomic_load(&s[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return v;
}

// Group all-reduce and barrier in one.  Every workgroup of the group stores its
// block total `mine` and arrives; the last to arrive folds the partials in a
// fixed order (fold(parts, n), called by the whole block, returns the same
// value in every thread), publishes the total and the phase; the others wait
// for the phase and read the total.  Every workgroup therefore sees the same
// bits.  The wait is bounded by spinLimit; on expiry (or when another
// workgroup has failed) the error flag is set and false returned.
template <class T, class Fold>
__device__ __forceinline__ bool group_allreduce(const T& mine, T& out, T* partial, GroupCtl* ctl, unsigned& phase,
                                                int G, int local, unsigned spinLimit, int* errFlag, int* shInt,
                                                T* shT, Fold fold) {
    ++phase;
    T* half = partial + (phase & 1u) * unsigned(G);
    if (threadIdx.x == 0) st_agent(&half[local], mine);
    __builtin_amdgcn_s_waitcnt(0);  // this wave's agent-scope stores have completed
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned old = __hip_atomic_fetch_add(&ctl->cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *shInt = (old == phase * unsigned(G) - 1u) ? 1 : 0;
    }
    __syncthreads();
    T* res = reinterpret_cast<T*>(ctl->res[phase & 1u]);
    if (*shInt) {
        T t = fold(half, G);
        if (threadIdx.x == 0) {
            st_agent(res, t);
            __builtin_amdgcn_s_waitcnt(0);
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            __hip_atomic_store(&ctl->gen, phase, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        out = t;
        __syncthreads();
        return true;
    }
    if (threadIdx.x == 0) {
        unsigned spins = 0;
        int ok = 1;
        while (__hip_atomic_load(&ctl->gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < phase) {
            if (++spins > spinLimit || __hip_atomic_load(errFlag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                ok = 0;
                __hip_atomic_store(errFlag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        if (ok) *shT = ld_agent(res);
        *shInt = ok;
    }
    __syncthreads();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    const bool ok = *shInt != 0;
    out = *shT;
    __syncthreads();
    return ok;
}

__device__ __forceinline__ double fold_double(const double* parts, int n, double* sh) {
    double t = 0;
    for (int k = threadIdx.x; k < n; k += blockDim.x) t += ld_agent(&parts[k]);
    return block_sum_double(t, sh);
}

__device__ __forceinline__ float p_next(float r, float beta, float p) { return r + beta * p; }

// The stored entries of row i in slot order, acc = term(acc, v, j) for each:
// the N slots of `mask` (the slots some row of the depth stores, assembled
// with the operator).  Every weight and column load of the row is issued
// before the gathers that term makes; an entry this row does not store
// (v = 0: dropped or missing) gathers row i itself with weight zero, which
// adds exactly nothing.
template <int N, class T, class F>
__device__ __forceinline__ T row_product_n(unsigned mask, int i, int M, const float* __restrict__ val,
                                           const int* __restrict__ neigh, T acc, F term) {
    // in chunks of at most 9 slots, so that the loads in flight stay within
    // the register budget of the occupancy the CG launch is sized for
    constexpr int C = N < 9 ? N : 9;
    static_assert(N % C == 0, "whole chunks");
    unsigned m = mask;
#pragma unroll
    for (int c0 = 0; c0 < N; c0 += C) {
        float vv[C];
        int jj[C];
#pragma unroll
        for (int k = 0; k < C; ++k) {
            const int q = N == 27 ? c0 + k : __builtin_ctz(m);
            m &= m - 1;
            vv[k] = val[q * M + i];
            jj[k] = neigh[q * M + i];
        }
#pragma unroll
        for (int k = 0; k < C; ++k) acc = term(acc, vv[k], vv[k] != 0.f ? jj[k] : i);
    }
    return acc;
}
// Depths whose operator keeps only the diagonal and the six face entries
// (seven slots: depth 9 and finer after the 1e-6 drop) read those slots only;
// every other depth reads all 27.
template <class T, class F>
__device__ __forceinline__ T row_product(unsigned mask, int i, int M, const float* __restrict__ val,
                                         const int* __restrict__ neigh, T acc, F term) {
    if (__popc(mask) == 7) return row_product_n<7>(mask, i, M, val, neigh, acc, term);
    return row_product_n<27>(0x7ffffffu, i, M, val, neigh, acc, term);
}

// Vectors that other workgroups read are exchanged as packed 8- or 16-byte
// records through buffer loads and stores with the cache policy of the
// agent-scope atomics (sc1), so one load brings all of a neighbour's values.
constexpr int kCoherent = 16;  // cache-policy bits: sc1
__device__ __forceinline__ __amdgpu_buffer_rsrc_t vec_rsrc(const void* base, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), short(0), int(bytes), 0x00020000);
}
__device__ __forceinline__ float2 ld_vec2(__amdgpu_buffer_rsrc_t r, int idx) {
    return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, idx * 8, 0, kCoherent));
}
__device__ __forceinline__ void st_vec2(__amdgpu_buffer_rsrc_t r, int idx, float2 v) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(__attribute__((ext_vector_type(2))) unsigned, v), r,
                                          idx * 8, 0, kCoherent);
}
__device__ __forceinline__ float4 ld_vec4(__amdgpu_buffer_rsrc_t r, int idx) {
    return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, idx * 16, 0, kCoherent));
}
__device__ __forceinline__ void st_vec4(__amdgpu_buffer_rsrc_t r, int idx, float4 v) {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(__attribute__((ext_vector_type(4))) unsigned, v), r,
                                           idx * 16, 0, kCoherent);
}

// --- one row per thread -------------------------------------------------------
// Both forms' kernels for depths whose rows all have a thread (to about 390k
// rows in all): a workgroup takes kRowThreads rows, the row's vectors stay in
// registers, and what its neighbours read of it (p, or the next residual) is
// formed once, in LDS.  A workgroup's rows are a patch of the surface (Morton
// order), so 87% of their stored entries lie inside it; each row outside that
// some entry names (a ghost: about half as many as rows) is read once per
// sweep, as one record, and its value formed beside the own rows'.  The
// weights are one constant per slot (the operator depends on the offset only;
// checked row by row), held in scalar registers; a row's columns are 26 16-bit
// places in LDS.  Only rows with a neighbour outside write records.
// Where the level-local child 0 rule changed the neighbour tables a row may lack
// its own entry, and in a tenth of such clouds a slot's weights differ from row
// to row: such a workgroup reads each row's own (RowHead::kOwnWeights), a group
// of one wave from LDS.  Neighbours outside that the ghost list cannot hold are
// read from memory (RowHead::kMemoryPlaces).
// Bound by the reductions' memory round trips (about 2 us each) and the
// ghosts' (1 us).  Whole solves with 256 rows a workgroup, the stencil per row
// and a record gathered per entry, and here: torus at depth 7 (71k rows) 146 ->
// 107 us mixed, 582 -> 293 us FP32 (whose two sums per iteration went through
// an arrival counter); ellipsoid at depth 8 (263k rows, several rows a thread
// before) 638 -> 195 us and 1398 -> 458 us; sphere at depth 5 (7k rows) 327 ->
// 209 us FP32.  Of these the maps take 14-30 us.
constexpr int kRowThreads = 512, kRowWaves = kRowThreads / PSR_WAVE;
// The sums' blocks: 256 rows, whatever the workgroup holds, so that they do not
// depend on it.
constexpr int kRowBlock = 256, kRowBlockWaves = kRowBlock / PSR_WAVE, kRowBlocks = kRowThreads / kRowBlock;
constexpr int kRowMaxBlocks = 4 * kRowThreads;  // blocks of a group
constexpr int kSlotStride = 2;                  // slots of a block and parity, whatever a sum uses
constexpr int kGhostTable = 2048, kGhostMax = kRowThreads * 2;
// Places are byte offsets into RowShared::v, two to a word; the top bit of the
// last word marks a boundary row.
constexpr int kPlaceGhosts = 4 * kRowThreads, kPlaceZero = 4 * (kRowThreads + kGhostMax), kPlaceMemory = 0x7ffc;
static_assert(kPlaceZero < kPlaceMemory, "place range");
constexpr unsigned kBoundaryBit = 1u << 31;
// Waves per SIMD: four workgroups a CU (524k rows resident) in the FP32 form,
// three (393k rows) in the mixed form, whose state is larger.
constexpr int kRowFp32Waves = 8, kRowMixedWaves = 6;

// What row_maps leaves for a workgroup of the row form (its ghosts' rows in a
// list of kGhostMax, its rows' places in a table [13][M]).
struct RowHead {
    int ghosts;
    int form;     // 0: what follows suffices
    float w[27];  // the slots' weights
    int pad[3];
    static constexpr int kOwnWeights = 1, kMemoryPlaces = 2;  // bits of form
};
struct RowMapArgs {
    const int* neigh;
    const float* val;
    const float* weights;  // the operator's entries by depth and slot on the regular grid, or null
    const int* q1Fired;
    unsigned* places;
    int* ghosts;
    RowHead* heads;
};

// The maps of the row form's workgroups, a workgroup each (ahead of the CG
// kernel: inside it the table costs registers that its sweeps then lack; beside
// the coarse divergence's fold, which leaves the GPU idle).  Every stored neighbour inside the workgroup gets its row's place.  Those
// outside (13% of the entries) are listed, shared out over the threads and
// entered into a hash table, whose used positions are numbered and become the
// ghosts' places.
__device__ __forceinline__ void row_maps_body(int psr_bid, int psr_nbid, const CgParams& P, const RowMapArgs& a) {
    __shared__ unsigned short place[26][kRowThreads];       // kGhostMark | table position until the ghosts are numbered
    __shared__ unsigned short list[26 * kRowThreads];       // entries outside: row << 5 | slot
    __shared__ int key[kGhostTable];                        // ghost rows by hash, -1: free
    __shared__ unsigned short number[kGhostTable];
    __shared__ unsigned weight[27];
    __shared__ int entries, ghosts, form;
    constexpr unsigned kGhostMark = 0x8000u;
    static_assert(kRowThreads == 512, "nine bits of row, five of slot");
    int gi = 0;
    while (gi + 1 < P.ngroups && int(psr_bid) >= P.g[gi + 1].firstWg) ++gi;
    const CgGroup& G = P.g[gi];
    const int t = int(threadIdx.x), M = P.M;
    const int r0 = G.rowBegin + (psr_bid - G.firstWg) * G.rowsPerWg;
    const int rows = min(G.rowBegin + G.rows, r0 + G.rowsPerWg) - r0;
    const bool own = t < rows;
    const int i = r0 + min(t, rows - 1);
    // on the regular grid an entry is its slot's constant where the neighbour exists
    const bool regular = a.weights && *a.q1Fired == 0;
    float v[27];
    int j[27];
#pragma unroll
    for (int q = 0; q < 27; ++q) j[q] = a.neigh[size_t(q) * M + i];
    if (regular) {
#pragma unroll
        for (int q = 0; q < 27; ++q) v[q] = j[q] >= 0 ? a.weights[27 * G.depth + q] : 0.f;
    } else {
#pragma unroll
        for (int q = 0; q < 27; ++q) v[q] = a.val[size_t(q) * M + i];
    }
    for (int k = t; k < kGhostTable; k += kRowThreads) key[k] = -1;
    if (t < 27) weight[t] = regular ? __float_as_uint(a.weights[27 * G.depth + t]) : 0u;
    if (t == 0) entries = 0, ghosts = 0, form = 0;
    __syncthreads();
    int needs = 0;
    unsigned outside = 0u, ghost = 0u;  // ghost: slots with a stored neighbour outside
#pragma unroll
    for (int q = 0; q < 27; ++q) {
        const int l = j[q] - r0;
        const bool inside = unsigned(l) < unsigned(rows), stored = own && v[q] != 0.f;
        if (!regular && stored) weight[q] = __float_as_uint(v[q]);  // any row's
        if (q == 13) {  // the row itself or, below a parent the child 0 rule changed, nothing
            if (own && !stored) needs |= RowHead::kOwnWeights;
            continue;
        }
        const bool away = own && j[q] >= 0 && !inside;
        if (away) outside = 1u;
        if (away && stored) ghost |= 1u << q;
        place[q < 13 ? q : q - 1][t] =
            static_cast<unsigned short>(!stored ? kPlaceZero : (inside ? 4 * l : kPlaceMemory));
    }
    // the entries outside, listed: a wave's at consecutive positions
    const int count = __popc(ghost);
    int inc = count;
#pragma unroll
    for (int off = 1; off < PSR_WAVE; off <<= 1) {
        const int o = __shfl_up(inc, off, PSR_WAVE);
        if (int(__lane_id()) >= off) inc += o;
    }
    int base = 0;
    if (__lane_id() == PSR_WAVE - 1 && inc) base = atomicAdd(&entries, inc);
    int at = __builtin_amdgcn_readlane(base, PSR_WAVE - 1) + inc - count;
    for (unsigned m = ghost; m; m &= m - 1) list[at++] = static_cast<unsigned short>(t << 5 | __builtin_ctz(m));
    __syncthreads();
    for (int e = t; e < entries; e += kRowThreads) {
        const int row = list[e] >> 5, q = list[e] & 31;
        const int n = a.neigh[size_t(q) * M + r0 + row];
        static_assert(kGhostTable == 1 << 11, "hash bits");
        unsigned h = (unsigned(n) * 2654435761u) >> 21;
        for (int tries = 0; tries < kGhostTable; ++tries, h = (h + 1) & (kGhostTable - 1)) {
            const int old = atomicCAS(&key[h], -1, n);
            if (old != -1 && old != n) continue;
            place[q < 13 ? q : q - 1][row] = static_cast<unsigned short>(kGhostMark | h);
            break;  // (a full table leaves kPlaceMemory)
        }
    }
    __syncthreads();
    // the positions in use are numbered wave by wave, and listed
    int* rowsOf = a.ghosts + size_t(psr_bid) * kGhostMax;
    for (int h = t; h < kGhostTable; h += kRowThreads) {
        const int row = key[h];
        const unsigned long long mask = __ballot(row >= 0);
        int n = 0;
        if (__lane_id() == 0 && mask) n = atomicAdd(&ghosts, __popcll(mask));
        n = __builtin_amdgcn_readfirstlane(n) + __popcll(mask & ((1ull << __lane_id()) - 1ull));
        number[h] = static_cast<unsigned short>(n);
        if (row >= 0 && n < kGhostMax) rowsOf[n] = row;
    }
    __syncthreads();
    // more ghosts than the list holds: every neighbour outside is read from memory
    const bool overflow = ghosts > kGhostMax;
    auto final_place = [&](int e) {
        unsigned p = place[e][t];
        if (p & kGhostMark) p = overflow ? unsigned(kPlaceMemory) : unsigned(kPlaceGhosts) + 4u * number[p & (kGhostTable - 1)];
        if (own && p == unsigned(kPlaceMemory)) needs |= RowHead::kMemoryPlaces;
        return p;
    };
    unsigned word = 0u;
#pragma unroll
    for (int e = 0; e < 26; e += 2) {
        word = final_place(e) | final_place(e + 1) << 16;
        if (own && e < 24) a.places[size_t(e / 2) * M + i] = word;
    }
    if (!regular) {
#pragma unroll
        for (int q = 0; q < 27; ++q)
            if (own && v[q] != 0.f && __float_as_uint(v[q]) != weight[q]) needs |= RowHead::kOwnWeights;
    }
    if (needs) atomicOr(&form, needs);
    __syncthreads();
    // readers of a row outside its workgroup: symmetric where the tables are regular
    const bool boundary = outside != 0u || *a.q1Fired != 0 || form != 0;
    if (own) a.places[size_t(12) * M + i] = word | (boundary ? kBoundaryBit : 0u);
    RowHead& head = a.heads[psr_bid];
    if (t < 27) head.w[t] = __uint_as_float(weight[t]);
    if (t == 0) head.ghosts = overflow ? 0 : ghosts, head.form = form;
}
// The solve's first kernel: the fold of the coarse nodes' divergence, and the
// row form's maps (mapBlocks of them; none for the other forms) beside it.  Both
// are chains of loads in a few workgroups, 4 and 13 us as a launch each on a small
// cloud and 14 us together.  On the regular grid the maps leave the entries unread
// (a row's are its slots' constants where the neighbour exists): a batch of 32
// depth-7 clouds, whose maps and assembly this and assemble_rows shorten, 11.7 ->
// 10.3 ms a call.
__device__ __forceinline__ void solve_prepare_body(int psr_bid, int psr_nbid, const CgParams& P, const RowMapArgs& a,
                                                   int mapBlocks, const DivFoldArgs& fold) {
    if (psr_bid < mapBlocks) row_maps_body(psr_bid, psr_nbid, P, a);
    else divergence_fold(fold, (psr_bid - mapBlocks) * kRowThreads + int(threadIdx.x));
}
__global__ void __launch_bounds__(kRowThreads) solve_prepare(CgParams P, RowMapArgs a, int mapBlocks, DivFoldArgs fold) {
    solve_prepare_body(blockIdx.x, gridDim.x, P, a, mapBlocks, fold);
}
PSR_BATCHABLE(solve_prepare, kRowThreads)

// A value that is the same in every lane, in scalar registers: the rows' state
// needs the vector ones (a spilled one's reload would wait for the records'
// stores ahead of it).
__device__ __forceinline__ float uniform(float v) {
    return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v)));
}
__device__ __forceinline__ double uniform(double v) {
    const long long b = __double_as_longlong(v);
    return __hiloint2double(__builtin_amdgcn_readfirstlane(int(b >> 32)), __builtin_amdgcn_readfirstlane(int(b)));
}
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
// The group of workgroup `bid` (a batch's workgroups take bid and the arguments from memory).
__device__ __forceinline__ CgGroup uniform_group(const CgParams& P, int bid) {
    int gi = 0;
    while (gi + 1 < P.ngroups && bid >= P.g[gi + 1].firstWg) ++gi;
    const CgGroup& g = P.g[gi];
    return CgGroup{uniform(g.depth),   uniform(g.rowBegin),  uniform(g.rows), uniform(g.firstWg),
                   uniform(g.wgs),     uniform(g.rowsPerWg), uniform(g.indef)};
}

struct RowShared {
    // the rows' places; or, in a one-wave group with own weights, lane t's 27
    // weights and 13 words of places as chunks of four, [11][PSR_WAVE]
    alignas(16) unsigned place[13][kRowThreads];
    float v[kRowThreads + kGhostMax + 1];  // the rows' values, the ghosts', a zero
    double sum[2][kRowWaves][2];           // wave sums, by the parity of the sum
    double fold[kRowWaves][2];
    int fail;
};
constexpr int kLaneChunks = 11, kLanePlaces = 28;  // words: 27 weights and a pad, then the places
static_assert(kLaneChunks * 4 >= kLanePlaces + 13 && kLaneChunks * 4 * PSR_WAVE <= 13 * kRowThreads, "a lane's words fit");
__device__ __forceinline__ unsigned& lane_word(RowShared& sh, int k, int t) {
    return (&sh.place[0][0])[4 * (k / 4 * PSR_WAVE + t) + k % 4];
}

// A row's place in its group and what it needs of the stencil.
struct RowMap {
    int ghostRow[2];     // this thread's ghosts (places t and t + kRowThreads of them): row, or -1
    bool boundary;       // another workgroup may read this row
    int form;            // RowHead::form, the same in the whole workgroup
    bool lanes;          // the weights and places are in lane_word
};

__device__ __forceinline__ RowMap row_map(RowShared& sh, const RowMapArgs& a, int bid, int r0, int rows, int M, bool multi,
                                          bool oneWave) {
    RowMap m;
    const int t = int(threadIdx.x), i = r0 + min(t, rows - 1);
    const bool own = t < rows;
    const RowHead& head = a.heads[bid];
    const int ghosts = __builtin_amdgcn_readfirstlane(head.ghosts);
    m.form = __builtin_amdgcn_readfirstlane(head.form);
    m.lanes = oneWave && m.form == RowHead::kOwnWeights;
#pragma unroll
    for (int e = 0; e < 13; ++e) {
        unsigned p = a.places[size_t(e) * M + i];
        if (e == 12) {
            m.boundary = multi && own && (p & kBoundaryBit) != 0u;
            p &= ~kBoundaryBit;
        }
        // the other waves of a one-wave group have no rows, and write none of its words
        if (m.lanes && t < PSR_WAVE) lane_word(sh, kLanePlaces + e, t) = p;
        else if (!oneWave || t < PSR_WAVE) sh.place[e][t] = p;
    }
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        const int e = t + g * kRowThreads;
        m.ghostRow[g] = e < ghosts ? a.ghosts[size_t(bid) * kGhostMax + e] : -1;
    }
    if (m.lanes && t < PSR_WAVE) {
#pragma unroll 1
        for (int q = 0; q < 27; ++q) lane_word(sh, q, t) = own ? __float_as_uint(a.val[size_t(q) * M + i]) : 0u;
    }
    if (t == 0) sh.fail = 0, sh.v[kPlaceZero / 4] = 0.f;
    __syncthreads();
    return m;
}

// The solves are compiled twice, for workgroups of form 0 (OWN false: the slots'
// weights) and for the others (OWN: each row's own), so that what the others need
// costs the first no registers: a spilled one is read back every sweep (300k
// points at depth 8, mixed, 242 us a solve, 324 with one loop for both).
// The others have missing entries and, where they are one wave at a coarse depth,
// thousands of sweeps: solves of four bent clouds in the FP32 form with weights
// and places in LDS by computed address and two branches an entry 41-52 ms, in
// this straight line 7.3-18.5 ms; mixed 2.0-4.7 and 0.4-1.6 ms.
template <bool OWN>
__device__ __forceinline__ void slot_weights(const RowHead& head, float (&w)[27]) {
#pragma unroll
    for (int q = 0; q < 27; ++q) w[q] = OWN ? 0.f : uniform(head.w[q]);
}

// sum over the slots in order of weight x value, acc = term(acc, weight, value),
// the values from LDS (`self`: the row's own); a thread without a row gets
// something, which it must not use.  An entry that is not stored adds zero times
// zero.  memory(e): the value of the neighbour in entry e of the table where it
// has no place.
template <bool OWN, class T, class Term, class Memory>
__device__ __forceinline__ T row_product(const RowMap& m, const RowMapArgs& a, RowShared& sh, const float (&w)[27],
                                         float self, bool own, int i, int M, T acc, Term term, Memory memory) {
    const int t = int(threadIdx.x);
    auto placed = [&](unsigned p) { return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(sh.v) + p); };
    if constexpr (!OWN) {
        // half of the neighbours' values are read together, then summed
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const int first = half ? 14 : 0, count = half ? 12 : 14;
            float n[14];
#pragma unroll
            for (int e = 0; e < count; e += 2) {
                const unsigned p = sh.place[(first + e) / 2][t];
                n[e] = placed(p & 0xffffu);
                n[e + 1] = placed(p >> 16);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < count; ++e) {
                if (first + e == 13) acc = term(acc, w[13], self);  // slot 13, the row itself, comes before entry 13
                acc = term(acc, w[first + e < 13 ? first + e : first + e + 1], n[e]);
            }
        }
        return acc;
    }
    // slots 0-14 (entries 0-13 and the row itself), then 15-26: the values of a
    // part are read together, then summed.  words(k, p): words k.. of the row's
    // places; weights(q, v): the weights of slots q..
    auto in_parts = [&](auto words, auto weights) {
#pragma unroll
        for (int part = 0; part < 2; ++part) {
            const int count = part ? 12 : 14;
            unsigned p[7];
            float v[15], n[14];
            words(part * 7, p);
            weights(part * 15, v);
#pragma unroll
            for (int e = 0; e < count; ++e) n[e] = placed(e % 2 ? p[e / 2] >> 16 : p[e / 2] & 0xffffu);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < (part ? 12 : 15); ++k)
                acc = term(acc, v[k], part ? n[k] : (k < 13 ? n[k] : (k == 13 ? self : n[13])));
        }
    };
    if (m.lanes) {
        // such a group may take thousands of sweeps: its words come four at a time
        const uint4* words = reinterpret_cast<const uint4*>(&sh.place[0][0]) + t;
        auto word = [](const uint4& u, int k) { return k == 0 ? u.x : (k == 1 ? u.y : (k == 2 ? u.z : u.w)); };
        in_parts(
            [&](int first, unsigned (&p)[7]) {
                const int k0 = kLanePlaces + first, c0 = k0 / 4;
                uint4 u[3];
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    if (c0 + c < kLaneChunks) u[c] = words[(c0 + c) * PSR_WAVE];
#pragma unroll
                for (int k = 0; k < 7; ++k)
                    if (first + k < 13) p[k] = word(u[(k0 + k) / 4 - c0], (k0 + k) % 4);
            },
            [&](int first, float (&v)[15]) {
                const int c0 = first / 4;
                uint4 u[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) u[c] = words[(c0 + c) * PSR_WAVE];
#pragma unroll
                for (int k = 0; k < 15; ++k)
                    if (first + k < 27) v[k] = __uint_as_float(word(u[(first + k) / 4 - c0], (first + k) % 4));
            });
        return acc;
    }
    if (!own) return acc;
    asm volatile("" : "+v"(i));  // addresses are formed anew, not kept from sweep to sweep
    if (m.form == RowHead::kOwnWeights) {
        auto place_words = [&](int first, unsigned (&p)[7]) {
#pragma unroll
            for (int k = 0; k < 7; ++k)
                if (first + k < 13) p[k] = sh.place[first + k][t];
        };
        float rowWeights[27];  // all on their way at once
#pragma unroll
        for (int q = 0; q < 27; ++q) rowWeights[q] = (a.val + size_t(q) * M)[unsigned(i)];
        in_parts(place_words, [&](int first, float (&v)[15]) {
#pragma unroll
            for (int k = 0; k < 15; ++k)
                if (first + k < 27) v[k] = rowWeights[first + k];
        });
        return acc;
    }
#pragma unroll 1
    for (int c = 0; c < 27; c += 9) {
        float v[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) v[k] = (a.val + size_t(c + k) * M)[unsigned(i)];
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            const int q = c + k;
            if (v[k] == 0.f) continue;  // adds nothing
            float n = self;
            if (q != 13) {
                const int e = q < 13 ? q : q - 1;
                const unsigned p = (sh.place[e / 2][t] >> (e & 1 ? 16 : 0)) & 0xffffu;
                n = p == unsigned(kPlaceMemory) ? memory(size_t(q) * M + i) : placed(p);
            }
            acc = term(acc, v[k], n);
        }
    }
    return acc;
}

// One group's sums: where its slots lie and how far it is.
struct RowGroup {
    float4* region;    // [2 parities][blocks][kSlotStride] slots
    int blocks;        // of the group
    int firstBlock;    // this workgroup's first
    int ownBlocks;     // and how many it has
    bool multi, oneWave;
    unsigned phase, parity;
    unsigned spinLimit;
    int* errFlag;
};

// Sums v[n] over the group's rows, the same bits in every thread of every
// workgroup: wave sums, blocks of four waves, then the blocks in the order of
// 64 a wave.  A block's total goes to its slot(s), 8 bytes of payload stamped
// with the phase in one 16-byte store; every workgroup reads all blocks' slots,
// one lane a slot, each wave until its own have come, and folds them: no
// atomics, one memory round trip after the last workgroup's store.  Slots
// alternate with the parity of the phase (a workgroup runs at most one phase
// ahead of the slowest) and start at zero (phases start at 1).  Every store of
// the workgroup before the call completes before its slots are stored: whoever
// has seen a phase's slots reads that phase's records.
template <int N>
__device__ __forceinline__ bool row_group_sum(double (&v)[N], RowShared& sh, RowGroup& g) {
#pragma unroll
    for (int n = 0; n < N; ++n) v[n] = wave_sum_f64(v[n]);
    if (g.oneWave) {
#pragma unroll
        for (int n = 0; n < N; ++n) v[n] = uniform(v[n]);
        wave_sync_memory();
        return true;
    }
    int t = int(threadIdx.x);
    asm volatile("" : "+v"(t));  // lane, wave and addresses are formed anew, not spilled from sum to sum
    const int lane = t % PSR_WAVE, wave = t / PSR_WAVE;
    g.parity ^= 1u;
    if (g.multi) __builtin_amdgcn_s_waitcnt(0);
    if (lane == 0) {
#pragma unroll
        for (int n = 0; n < N; ++n) sh.sum[g.parity][wave][n] = v[n];
    }
    __syncthreads();
    auto block_total = [&](int b, int n) {
        double s = 0;
        for (int k = 0; k < kRowBlockWaves; ++k) s += sh.sum[g.parity][b * kRowBlockWaves + k][n];
        return s;
    };
    if (!g.multi) {
#pragma unroll
        for (int n = 0; n < N; ++n) {
            double s = block_total(0, n);
            for (int b = 1; b < kRowBlocks; ++b) s += block_total(b, n);
            v[n] = uniform(s);
        }
        return true;
    }
    ++g.phase;
    const __amdgpu_buffer_rsrc_t rs = vec_rsrc(g.region + size_t(g.phase & 1u) * g.blocks * kSlotStride,
                                               sizeof(float4) * size_t(g.blocks) * kSlotStride);
    const float stamp = __uint_as_float(g.phase);
    if (t < N * g.ownBlocks) {
        const int b = t / N, n = t % N;
        const unsigned long long u = static_cast<unsigned long long>(__double_as_longlong(block_total(b, n)));
        st_vec4(rs, (g.firstBlock + b) * kSlotStride + n,
                make_float4(__uint_as_float(unsigned(u)), __uint_as_float(unsigned(u >> 32)), stamp, 0.f));
    }
    double part[N];
#pragma unroll
    for (int n = 0; n < N; ++n) part[n] = 0.0;
    for (int k = t; k - t < g.blocks; k += kRowThreads) {
        const bool mine = k < g.blocks;
        float4 got[N];
        for (unsigned spins = 0;; ++spins) {
            bool ready = true;
            if (mine) {
#pragma unroll
                for (int n = 0; n < N; ++n) {
                    got[n] = ld_vec4(rs, k * kSlotStride + n);
                    ready = ready && __float_as_uint(got[n].z) == g.phase;
                }
            }
            if (__ballot(!ready) == 0) break;
            if (spins >= g.spinLimit || ((spins & 63u) == 63u && __hip_atomic_load(g.errFlag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
                __hip_atomic_store(g.errFlag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                sh.fail = 1;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        if (mine) {
#pragma unroll
            for (int n = 0; n < N; ++n) part[n] += __hiloint2double(__float_as_int(got[n].y), __float_as_int(got[n].x));
        }
    }
#pragma unroll
    for (int n = 0; n < N; ++n) {
        part[n] = wave_sum_f64(part[n]);
        if (lane == 0) sh.fold[wave][n] = part[n];
    }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < N; ++n) {
        double s = 0;
        for (int k = 0; k < kRowWaves; ++k) s += sh.fold[k][n];
        v[n] = uniform(s);
    }
    return __builtin_amdgcn_readfirstlane(sh.fail) == 0;
}

__device__ __forceinline__ RowGroup row_group(const CgParams& P, const CgGroup& G, int local, float4* slots, int* errFlag) {
    RowGroup g;
    const int per = G.rowsPerWg > kRowBlock ? kRowBlocks : 1;  // blocks of a full workgroup
    const int last = G.rows - (G.wgs - 1) * G.rowsPerWg;       // rows of the last
    g.blocks = (G.wgs - 1) * per + (last > kRowBlock ? 2 : 1);
    g.firstBlock = local * per;
    g.ownBlocks = local + 1 < G.wgs ? per : g.blocks - g.firstBlock;
    g.region = slots + size_t(2) * kRowBlocks * kSlotStride * G.firstWg;
    g.multi = G.wgs > 1;
    // a group of at most one wave of rows (the coarsest depths) iterates in
    // wave 0 alone, with no workgroup barrier (a wave's sum equals the block's,
    // whose other waves add exact zeros)
    g.oneWave = !g.multi && G.rows <= PSR_WAVE;
    g.phase = g.parity = 0u;
    g.spinLimit = unsigned(uniform(int(P.spinLimit)));
    g.errFlag = errFlag;
    return g;
}
__device__ __forceinline__ void row_sync(const RowGroup& g) {
    if (g.oneWave) wave_sync_memory();
    else __syncthreads();
}

// The reference's CG (CGAlgorithm.cu:10-80), one launch for all depths.  Per
// iteration k the record of row i in buffer k & 1 holds {r_k, p_{k-1}}; a
// ghost's p_k = r_k + beta p_{k-1} is formed from it, so the update of p and
// the product A p need no group barrier in between (CGAlgorithm.cu:37-53).
template <bool OWN>
__device__ __forceinline__ void cg_fp32_row_solve(int psr_bid, const CgParams& P, const CgGroup& G, const RowMapArgs& maps,
                                                  const RowMap& m, RowGroup& g, RowShared& sh, int r0, int rows,
                                                  const float* __restrict__ b, float* __restrict__ x, float2* state,
                                                  int* __restrict__ iters, double* __restrict__ resid) {
    const int local = psr_bid - G.firstWg, t = int(threadIdx.x), M = uniform(P.M), i = r0 + t;
    const bool own = t < rows;
    const int* __restrict__ neigh = maps.neigh;
    float w[27];
    slot_weights<OWN>(maps.heads[psr_bid], w);
    const __amdgpu_buffer_rsrc_t st = vec_rsrc(state, sizeof(float2) * 2 * size_t(M));
    // x = 0, r = b, rr = r.r  (CGAlgorithm.cu:21-33 with x0 = 0)
    float xi = 0.f, ri = own ? b[i] : 0.f, pi = 0.f;
    if (m.boundary) st_vec2(st, i, make_float2(ri, 0.f));
    double sum[1] = {double(ri * ri)};
    if (!row_group_sum<1>(sum, sh, g)) return;
    float rr = uniform(float(sum[0])), rrOld = 1.f;
    int k = 1;
    while (rr > P.tolSq && k <= P.maxIter) {
        const float beta = uniform((k > 1) ? rr / rrOld : 0.f);
        const int cur = ((k - 1) & 1) * M, nxt = M - cur;
        // p = r + beta p (CGAlgorithm.cu:37-43), Ap = A p (:47), p.Ap (:53)
        float2 n[2];
#pragma unroll
        for (int e = 0; e < 2; ++e)
            if (m.ghostRow[e] >= 0) n[e] = ld_vec2(st, cur + m.ghostRow[e]);
        pi = p_next(ri, beta, pi);
        sh.v[t] = pi;
#pragma unroll
        for (int e = 0; e < 2; ++e)
            if (m.ghostRow[e] >= 0) sh.v[kRowThreads + e * kRowThreads + t] = p_next(n[e].x, beta, n[e].y);
        row_sync(g);
        auto term = [](float a, float wq, float v) { return __fmaf_rn(wq, v, a); };
        auto memory = [&](size_t e) {
            const float2 r = ld_vec2(st, cur + neigh[e]);
            return p_next(r.x, beta, r.y);
        };
        const float api = row_product<OWN>(m, maps, sh, w, pi, own, i, M, 0.f, term, memory);
        sum[0] = own ? double(pi * api) : 0.0;
        if (!row_group_sum<1>(sum, sh, g)) return;
        const float alpha = uniform(float(double(rr) / sum[0]));
        xi = __fmaf_rn(alpha, pi, xi);
        ri = own ? __fmaf_rn(-alpha, api, ri) : 0.f;
        if (m.boundary) st_vec2(st, nxt + i, make_float2(ri, pi));
        sum[0] = double(ri * ri);
        rrOld = rr;
        if (!row_group_sum<1>(sum, sh, g)) return;
        rr = uniform(float(sum[0]));
        ++k;
    }
    if (own) x[i] = xi;
    if (local == 0 && t == 0) {
        iters[G.depth] = k - 1;
        iters[PSR_MAX_DEPTH + 1 + G.depth] = 1;
        resid[G.depth] = sqrt(double(rr));
    }
}
__device__ __forceinline__ void cg_fp32_row_body(int psr_bid, int psr_nbid, const CgParams& P, const RowMapArgs& maps,
                                                 const float* __restrict__ b, float* __restrict__ x, float2* state,
                                                 float4* slots, int* __restrict__ iters, double* __restrict__ resid,
                                                 int* errFlag) {
    __shared__ RowShared sh;
    psr_bid = uniform(psr_bid);
    const CgGroup G = uniform_group(P, psr_bid);
    const int local = psr_bid - G.firstWg, r0 = G.rowBegin + local * G.rowsPerWg;
    const int rows = min(G.rowBegin + G.rows, r0 + G.rowsPerWg) - r0;
    RowGroup g = row_group(P, G, local, slots, errFlag);
    const RowMap m = row_map(sh, maps, psr_bid, r0, rows, P.M, g.multi, g.oneWave);
    if (g.oneWave && int(threadIdx.x) >= PSR_WAVE) return;
    if (m.form == 0) cg_fp32_row_solve<false>(psr_bid, P, G, maps, m, g, sh, r0, rows, b, x, state, iters, resid);
    else cg_fp32_row_solve<true>(psr_bid, P, G, maps, m, g, sh, r0, rows, b, x, state, iters, resid);
}
__global__ void __launch_bounds__(kRowThreads) __attribute__((amdgpu_waves_per_eu(kRowFp32Waves))) cg_fp32_row(
    CgParams P, RowMapArgs maps, const float* __restrict__ b, float* __restrict__ x, float2* state, float4* slots,
    int* __restrict__ iters, double* __restrict__ resid, int* errFlag) {
    cg_fp32_row_body(blockIdx.x, gridDim.x, P, maps, b, x, state, slots, iters, resid, errFlag);
}
PSR_BATCHABLE_WAVES(cg_fp32_row, kRowThreads, kRowFp32Waves)


// A group of one workgroup with at most one row a thread (the coarse depths,
// and a batch's small clouds), solved by that workgroup alone with its
// vectors in LDS: cg_all_depths' arithmetic without a memory round trip per
// sweep.
// Makes p opaque to the compiler: loads through it are repeated after this
// point instead of being kept in registers from an earlier sweep.
template <class T>
__device__ __forceinline__ void opaque(const T*& p) {
    asm volatile("" : "+v"(p));
}

__device__ __forceinline__ void cg_small_fp32(const CgParams& P, const CgGroup& G, const int* __restrict__ neigh,
                                              const float* __restrict__ val, const float* __restrict__ b,
                                              float* __restrict__ x, int* __restrict__ iters,
                                              double* __restrict__ resid, double* sh) {
    // the small groups' stencil is re-read every sweep (it stays in cache) rather than
    // held in registers: this path shares its kernel with the large-depth sweeps
    const float* vs = val;
    const int* ns = neigh;
    __shared__ float lr[kCgThreads], lp[2][kCgThreads];
    const int M = P.M, t = int(threadIdx.x), i = G.rowBegin + t, rb = G.rowBegin;
    const bool own = t < G.rows;
    float xi = 0.f, ri = 0.f, pi = 0.f, api = 0.f;
    double loc = 0;
    if (own) {
        ri = b[i];
        lr[t] = ri;
        lp[0][t] = 0.f;
        loc = double(ri * ri);
    }
    float rr = float(block_sum_double(loc, sh)), rrOld = 1.f;
    int k = 1;
    while (rr > P.tolSq && k <= P.maxIter) {
        const float beta = (k > 1) ? rr / rrOld : 0.f;
        const int cur = (k - 1) & 1;
        double lpAp = 0;
        if (own) {
            float s = 0.f;
            opaque(vs);
            opaque(ns);
            s = row_product_n<27>(0x7ffffffu, i, M, vs, ns, s, [&](float a, float v, int j) {
                return a + v * p_next(lr[j - rb], beta, lp[cur][j - rb]);
            });
            pi = p_next(ri, beta, lp[cur][t]);
            lp[cur ^ 1][t] = pi;
            api = s;
            lpAp = double(pi * s);
        }
        const double pAp = block_sum_double(lpAp, sh);
        const float alpha = float(double(rr) / pAp);
        double lrr = 0;
        if (own) {
            xi = xi + alpha * pi;
            ri = ri + (-alpha) * api;
            lr[t] = ri;
            lrr = double(ri * ri);
        }
        rrOld = rr;
        rr = float(block_sum_double(lrr, sh));
        ++k;
    }
    if (own) x[i] = xi;
    if (threadIdx.x == 0) {
        iters[G.depth] = k - 1;
        iters[PSR_MAX_DEPTH + 1 + G.depth] = 1;
        resid[G.depth] = sqrt(double(rr));
    }
}

// The same iteration with several rows per thread (large depths): vectors in
// memory, the stencil read every sweep.
__device__ __forceinline__ void cg_all_depths_body(int psr_bid, int psr_nbid, const CgParams& P, const int* __restrict__ neigh,
                                                            const float* __restrict__ val,
                                                            const float* __restrict__ b, float* __restrict__ x,
                                                            float* r, float* pA, float* pB,
                                                            float* __restrict__ Ap, double* partial,
                                                            GroupCtl* ctlAll, int* __restrict__ iters,
                                                            double* __restrict__ resid, int* errFlag,
                                                            const unsigned* __restrict__ slotMasks) {
    __shared__ double sh[kCgWaves];
    __shared__ int shFlag;
    __shared__ double shRes;
    int gi = 0;
    while (gi + 1 < P.ngroups && int(psr_bid) >= P.g[gi + 1].firstWg) ++gi;
    const CgGroup G = P.g[gi];
    const int local = psr_bid - G.firstWg;
    const int r0 = G.rowBegin + local * G.rowsPerWg;
    const int r1 = min(G.rowBegin + G.rows, r0 + G.rowsPerWg);
    const int M = P.M;
    double* part = partial + 2 * G.firstWg;
    GroupCtl* ctl = ctlAll + gi;
    unsigned phase = 0;
    const bool multi = G.wgs > 1;
    if (!multi && G.rows <= kCgThreads) {
        cg_small_fp32(P, G, neigh, val, b, x, iters, resid, sh);
        return;
    }
    const unsigned slotMask = slotMasks[G.depth];

    // Sum over the group (partials double-buffered by phase parity).
    auto group_sum = [&](double v, double& out) -> bool {
        double s = block_sum_double(v, sh);
        if (!multi) {
            out = s;
            return true;
        }
        return group_allreduce(s, out, part, ctl, phase, G.wgs, local, P.spinLimit, errFlag, &shFlag, &shRes,
                               [&](const double* parts, int n) { return fold_double(parts, n, sh); });
    };

    // x = 0, r = b, rr = r.r  (CGAlgorithm.cu:21-33 with x0 = 0)
    double loc = 0;
    for (int i = r0 + threadIdx.x; i < r1; i += kCgThreads) {
        float bi = b[i];
        x[i] = 0.f;
        st_shared(&r[i], bi);
        st_shared(&pA[i], 0.f);
        loc += double(bi * bi);
    }
    double rrD;
    if (!group_sum(loc, rrD)) return;
    float rr = float(rrD), rrOld = 1.f;
    int k = 1;
    float* pOld = pA;
    float* pNew = pB;
    while (rr > P.tolSq && k <= P.maxIter) {
        const float beta = (k > 1) ? rr / rrOld : 0.f;
        // p = r + beta p (CGAlgorithm.cu:37-43), Ap = A p (:47), p.Ap (:53).  The
        // neighbours' p entries are formed from the previous r and p, so no
        // barrier is needed between the update and the product.
        double lpAp = 0;
        for (int i = r0 + threadIdx.x; i < r1; i += kCgThreads) {
            float s = 0.f;
            s = row_product(slotMask, i, M, val, neigh, s, [&](float a, float v, int j) {
                return a + v * p_next(ld_shared(&r[j]), beta, ld_shared(&pOld[j]));
            });
            float pi = p_next(ld_shared(&r[i]), beta, ld_shared(&pOld[i]));
            st_shared(&pNew[i], pi);
            Ap[i] = s;
            lpAp += double(pi * s);
        }
        double pAp;
        if (!group_sum(lpAp, pAp)) return;
        const float alpha = float(double(rr) / pAp);
        double lrr = 0;
        for (int i = r0 + threadIdx.x; i < r1; i += kCgThreads) {
            float pi = ld_shared(&pNew[i]);
            x[i] = x[i] + alpha * pi;
            float ri = ld_shared(&r[i]) + (-alpha) * Ap[i];
            st_shared(&r[i], ri);
            lrr += double(ri * ri);
        }
        rrOld = rr;
        double rrNew;
        if (!group_sum(lrr, rrNew)) return;
        rr = float(rrNew);
        float* t = pOld;
        pOld = pNew;
        pNew = t;
        ++k;
    }
    if (local == 0 && threadIdx.x == 0) {
        iters[G.depth] = k - 1;
        iters[PSR_MAX_DEPTH + 1 + G.depth] = 1;
        resid[G.depth] = sqrt(double(rr));
    }
}
__global__ void __launch_bounds__(kCgThreads) __attribute__((amdgpu_waves_per_eu(kCgFp32GenericWaves))) cg_all_depths(CgParams P, const int* __restrict__ neigh,
                                                            const float* __restrict__ val,
                                                            const float* __restrict__ b, float* __restrict__ x,
                                                            float* r, float* pA, float* pB,
                                                            float* __restrict__ Ap, double* partial,
                                                            GroupCtl* ctlAll, int* __restrict__ iters,
                                                            double* __restrict__ resid, int* errFlag,
                                                            const unsigned* __restrict__ slotMasks) {
    cg_all_depths_body(blockIdx.x, gridDim.x, P, neigh, val, b, x, r, pA, pB, Ap, partial, ctlAll, iters, resid, errFlag,
                       slotMasks);
}
PSR_BATCHABLE_WAVES(cg_all_depths, kCgThreads, kCgFp32GenericWaves)


// --- mixed-precision CG ------------------------------------------------------
// Same system per depth, solved to a true relative residual:
//   outer (FP64): r = b - A x accumulated in double, ||r|| / ||b|| in double;
//   inner (FP32): Chronopoulos-Gear CG on A e = r, one group reduction per
//                 iteration, dot products as compensated FP32 sums (Dot2:
//                 TwoProduct by fma, TwoSum accumulation).
// One barrier per inner iteration is possible because every value a row
// reads from its neighbours was written before the previous barrier: the
// neighbour's next residual is formed on the fly as
//   r_{k+1} = r_k - alpha_k (w_k + beta_k s_{k-1}),  w = A r,  s = A p,
// with r, w and s double-buffered by iteration parity.

__device__ __forceinline__ void two_sum_acc(float& s, float& c, float v) {
#pragma clang fp contract(off)
    float t = s + v;
    float bv = t - s;
    float e = (s - (t - bv)) + (v - bv);
    s = t;
    c += e;
}
__device__ __forceinline__ void dot2_acc(float& s, float& c, float a, float b) {
#pragma clang fp contract(off)
    float p = a * b;
    float e = __fmaf_rn(a, b, -p);
    two_sum_acc(s, c, p);
    c += e;
}
__device__ __forceinline__ void comp_merge(float& s, float& c, float s2, float c2) {
#pragma clang fp contract(off)
    two_sum_acc(s, c, s2);
    c += c2;
}
// s_k = w_k + beta s_{k-1};  r_{k+1} = r_k - alpha s_k (owner and neighbours use the same operations)
__device__ __forceinline__ float s_next(float w, float beta, float sPrev) { return __fmaf_rn(beta, sPrev, w); }
__device__ __forceinline__ float r_next(float r, float alpha, float s) { return __fmaf_rn(-alpha, s, r); }

struct Comp2 {
    float gs, gc, ds, dc;  // gamma = gs + gc, delta = ds + dc
};

__device__ __forceinline__ void comp2_merge(Comp2& a, const Comp2& b) {
    comp_merge(a.gs, a.gc, b.gs, b.gc);
    comp_merge(a.ds, a.dc, b.ds, b.dc);
}

// Block-wide merge in a fixed order; every thread returns the same value.
template <int CTRL>
__device__ __forceinline__ void comp2_dpp_step(Comp2& v) {
    const Comp2 o{dpp_f32<CTRL>(v.gs), dpp_f32<CTRL>(v.gc), dpp_f32<CTRL>(v.ds), dpp_f32<CTRL>(v.dc)};
    comp2_merge(v, o);
}
__device__ __forceinline__ Comp2 readlane_comp2(const Comp2& v, int lane) {
    return Comp2{readlane_f32(v.gs, lane), readlane_f32(v.gc, lane), readlane_f32(v.ds, lane), readlane_f32(v.dc, lane)};
}
// The wave's merge through DPP (psr_common.h: rows of 16, then the four rows
// in a fixed order); every lane returns the same value.
__device__ __forceinline__ Comp2 wave_comp2(Comp2 v) {
    comp2_dpp_step<kDppSwap1>(v);
    comp2_dpp_step<kDppSwap2>(v);
    comp2_dpp_step<kDppHalfMirror>(v);
    comp2_dpp_step<kDppMirror>(v);
    Comp2 r = readlane_comp2(v, 0);
    comp2_merge(r, readlane_comp2(v, 16));
    comp2_merge(r, readlane_comp2(v, 32));
    comp2_merge(r, readlane_comp2(v, 48));
    return r;
}
__device__ __forceinline__ Comp2 block_comp2(Comp2 v, Comp2* sh) {
    v = wave_comp2(v);
    int w = threadIdx.x / PSR_WAVE;
    if (__lane_id() == 0) sh[w] = v;
    __syncthreads();
    Comp2 t = sh[0];
    for (int k = 1; k < kCgWaves; ++k) comp2_merge(t, sh[k]);
    __syncthreads();
    return t;
}

// Mixed form, one launch for all depths, one row per thread.  The two dot
// products, gamma = r.r and delta = w.r, are summed in FP64 (a product of two
// floats is exact in FP64), so gamma of a right-hand side b is ||b||^2 to the
// bit.  Per inner iteration k the record of row i in buffer k & 1 holds
// {r_k, w_k, s_{k-1}, x_k}; the row writes {r_{k+1}, w_{k+1}, s_k, x_{k+1}} to
// the other buffer.
template <bool OWN>
__device__ __forceinline__ void cg_mixed_row_solve(int psr_bid, const CgParams& P, const CgGroup& G, const RowMapArgs& maps,
                                                   const RowMap& m, RowGroup& g, RowShared& sh, int r0, int rows,
                                                   const float* __restrict__ b, float* x, float* rOut, float4* state,
                                                   int* __restrict__ iters, double* __restrict__ resid,
                                                   double* __restrict__ trueRel) {
    const int local = psr_bid - G.firstWg, t = int(threadIdx.x), M = uniform(P.M), i = r0 + t;
    const bool own = t < rows;
    const int* __restrict__ neigh = maps.neigh;
    float w[27];
    slot_weights<OWN>(maps.heads[psr_bid], w);
    const __amdgpu_buffer_rsrc_t st = vec_rsrc(state, sizeof(float4) * 2 * size_t(M));
    auto term = [](float a, float wq, float v) { return __fmaf_rn(wq, v, a); };
    auto ghost_values = [&](auto value) {  // value(row) into the ghosts' places
        float n[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            int j = m.ghostRow[e];
            asm volatile("" : "+v"(j));  // no address is kept from step to step
            n[e] = j >= 0 ? value(j) : 0.f;
        }
#pragma unroll
        for (int e = 0; e < 2; ++e)
            if (m.ghostRow[e] >= 0) sh.v[kRowThreads + e * kRowThreads + t] = n[e];
    };
    float xi = 0.f, ro = 0.f, wo = 0.f, so = 0.f, po = 0.f;
    // ||b||^2 in FP64 (the outer residual of x = 0 is b itself) is gamma of the
    // first outer step, whose sum is bit for bit that of b.b; a solve that
    // takes no step sums it alone.
    double bb = 0;
    const bool stepping = P.maxOuter > 0 && P.maxIter > 0;
    if (!stepping) {
        const double bi = own ? double(b[i]) : 0.0;
        double loc[1] = {bi * bi};
        if (!row_group_sum<1>(loc, sh, g)) return;
        bb = loc[0];
    }
    double rr = bb, rel = (bb > 0 || stepping) ? 1.0 : 0.0;
    const float* rhs = b;
    int total = 0, outer = 0;
    float gamma = 0.f;
    while (rel > P.relTol && outer < P.maxOuter && total < P.maxIter) {
        // r_0 = rhs, w_0 = A r_0, s_{-1} = 0, p_{-1} = 0
        int ii = i;
        asm volatile("" : "+v"(ii));  // nor this row's
        ro = own ? ld_shared(&rhs[ii]) : 0.f;
        sh.v[t] = ro;
        ghost_values([&](int j) { return ld_shared(&rhs[j]); });
        row_sync(g);
        {
            auto memory = [&](size_t e) { return ld_shared(&rhs[neigh[e]]); };
            wo = row_product<OWN>(m, maps, sh, w, ro, own, i, M, 0.f, term, memory);
            if (!own) wo = 0.f;
        }
        so = po = 0.f;
        if (m.boundary) st_vec4(st, i, make_float4(ro, wo, 0.f, xi));
        double d[2] = {double(ro) * double(ro), double(wo) * double(ro)};
        if (!row_group_sum<2>(d, sh, g)) return;
        if (outer == 0) {
            bb = rr = d[0];
            if (!(bb > 0)) {
                rel = 0.0;
                break;
            }
        }
        // inner target on the updated residual: half the tolerance left, no tighter than FP32 can follow
        const double tgt = fmax(0.5 * P.relTol * sqrt(bb), 1e-6 * sqrt(rr));
        const float tgt2 = uniform(float(tgt * tgt));
        gamma = uniform(float(d[0]));
        const float delta = float(d[1]);
        float alpha = uniform(gamma / delta), beta = 0.f;
        int k = 0, kBest = 0;
        float gBest = gamma, xBest = xi;
        while (gamma > tgt2 && total + k < P.maxIter && k - kBest < kCgStall) {
            const int cur = (k & 1) * M, nxt = M - cur;
            float4 n[2];
#pragma unroll
            for (int e = 0; e < 2; ++e)
                if (m.ghostRow[e] >= 0) n[e] = ld_vec4(st, cur + m.ghostRow[e]);
            const float si = s_next(wo, beta, so);
            const float rni = r_next(ro, alpha, si);
            po = __fmaf_rn(beta, po, ro);
            xi = __fmaf_rn(alpha, po, xi);
            sh.v[t] = rni;
#pragma unroll
            for (int e = 0; e < 2; ++e)
                if (m.ghostRow[e] >= 0)
                    sh.v[kRowThreads + e * kRowThreads + t] = r_next(n[e].x, alpha, s_next(n[e].y, beta, n[e].z));
            row_sync(g);
            auto memory = [&](size_t e) {
                const float4 r = ld_vec4(st, cur + neigh[e]);
                return r_next(r.x, alpha, s_next(r.y, beta, r.z));
            };
            wo = row_product<OWN>(m, maps, sh, w, rni, own, i, M, 0.f, term, memory);
            if (!own) wo = 0.f;
            ro = rni;
            so = si;
            if (m.boundary) st_vec4(st, nxt + i, make_float4(rni, wo, si, xi));
            d[0] = double(rni) * double(rni);
            d[1] = double(wo) * double(rni);
            if (!row_group_sum<2>(d, sh, g)) return;
            const float gNew = uniform(float(d[0])), dNew = float(d[1]);
            const float bNew = gNew / gamma;
            alpha = uniform(gNew / (dNew - bNew * gNew / alpha));
            beta = uniform(bNew);
            gamma = gNew;
            ++k;
            if (gamma < gBest) {  // the same in every workgroup of the group
                gBest = gamma;
                kBest = k;
                xBest = xi;
            }
        }
        total += k;
        ++outer;
        if (kBest < k) {
            // back to the iterate of the smallest residual; one more exchange
            // orders the restored x before the outer residual reads it
            gamma = gBest;
            xi = xBest;
            if (m.boundary) st_vec4(st, (k & 1) * M + i, make_float4(0.f, 0.f, 0.f, xi));
            double fence[1] = {0.0};
            if (!row_group_sum<1>(fence, sh, g)) return;
        }
        // outer residual in FP64, x from the rows and from the last sweep's records
        const int last = (k & 1) * M;
        if (g.oneWave) wave_sync_memory();
        else __syncthreads();  // sh.v of the last product has been read
        sh.v[t] = xi;
        ghost_values([&](int j) { return ld_vec4(st, last + j).w; });
        row_sync(g);
        double loc[1] = {0.0};
        if (own) {
            auto term64 = [](double a, float wq, float v) { return a - double(wq) * double(v); };
            auto memory = [&](size_t e) { return ld_vec4(st, last + neigh[e]).w; };
            asm volatile("" : "+v"(ii));
            const double acc = row_product<OWN>(m, maps, sh, w, xi, own, i, M, double(b[ii]), term64, memory);
            st_shared(&rOut[ii], float(acc));
            loc[0] = acc * acc;
        }
        if (!row_group_sum<1>(loc, sh, g)) return;
        rr = loc[0];
        rel = uniform(bb > 0 ? sqrt(rr / bb) : 0.0);
        rhs = rOut;
        // an inner solve that found no smaller residual leaves x as it was:
        // another outer step would repeat it
        if (kBest == 0) break;
    }
    if (own) x[i] = xi;
    if (local == 0 && t == 0) {
        iters[G.depth] = total;
        iters[PSR_MAX_DEPTH + 1 + G.depth] = outer;
        resid[G.depth] = sqrt(double(gamma));
        trueRel[G.depth] = rel;
    }
}
__device__ __forceinline__ void cg_mixed_row_body(int psr_bid, int psr_nbid, const CgParams& P, const RowMapArgs& maps,
                                                  const float* __restrict__ b, float* x, float* rOut, float4* state,
                                                  float4* slots, int* __restrict__ iters, double* __restrict__ resid,
                                                  double* __restrict__ trueRel, int* errFlag) {
    __shared__ RowShared sh;
    psr_bid = uniform(psr_bid);
    const CgGroup G = uniform_group(P, psr_bid);
    const int local = psr_bid - G.firstWg, r0 = G.rowBegin + local * G.rowsPerWg;
    const int rows = min(G.rowBegin + G.rows, r0 + G.rowsPerWg) - r0;
    RowGroup g = row_group(P, G, local, slots, errFlag);
    const RowMap m = row_map(sh, maps, psr_bid, r0, rows, P.M, g.multi, g.oneWave);
    if (g.oneWave && int(threadIdx.x) >= PSR_WAVE) return;
    if (m.form == 0)
        cg_mixed_row_solve<false>(psr_bid, P, G, maps, m, g, sh, r0, rows, b, x, rOut, state, iters, resid, trueRel);
    else
        cg_mixed_row_solve<true>(psr_bid, P, G, maps, m, g, sh, r0, rows, b, x, rOut, state, iters, resid, trueRel);
}
__global__ void __launch_bounds__(kRowThreads) __attribute__((amdgpu_waves_per_eu(kRowMixedWaves))) cg_mixed_row(
    CgParams P, RowMapArgs maps, const float* __restrict__ b, float* x, float* rOut, float4* state, float4* slots,
    int* __restrict__ iters, double* __restrict__ resid, double* __restrict__ trueRel, int* errFlag) {
    cg_mixed_row_body(blockIdx.x, gridDim.x, P, maps, b, x, rOut, state, slots, iters, resid, trueRel, errFlag);
}
PSR_BATCHABLE_WAVES(cg_mixed_row, kRowThreads, kRowMixedWaves)


// The mixed form's group of one workgroup with at most one row a thread,
// vectors in LDS: cg_mixed_all_depths' arithmetic without a memory round trip
// per sweep.
__device__ __forceinline__ void cg_small_mixed(const CgParams& P, const CgGroup& G, const int* __restrict__ neigh,
                                               const float* __restrict__ val, const float* __restrict__ b,
                                               float* __restrict__ x, int* __restrict__ iters,
                                               double* __restrict__ resid, double* __restrict__ trueRel,
                                               double* shd, Comp2* shc) {
    // the small groups' stencil is re-read every sweep (it stays in cache) rather than
    // held in registers: this path shares its kernel with the large-depth sweeps
    const float* vs = val;
    const int* ns = neigh;
    __shared__ float lx[kCgThreads], lro[kCgThreads], lr[2][kCgThreads], lw[2][kCgThreads], ls[2][kCgThreads];
    const int M = P.M, t = int(threadIdx.x), i = G.rowBegin + t, rb = G.rowBegin;
    const bool own = t < G.rows;
    // x = 0; ||b||^2 in FP64 (the outer residual of x = 0 is b itself)
    double loc = 0;
    if (own) {
        lx[t] = 0.f;
        const double bi = b[i];
        loc = bi * bi;
    }
    const double bb = block_sum_double(loc, shd);
    double rr = bb, rel = bb > 0 ? 1.0 : 0.0;
    bool fromB = true;  // the first outer step solves for b, the later ones for the residual in lro
    int total = 0, outer = 0;
    float gamma = 0.f, pv = 0.f;
    while (rel > P.relTol && outer < P.maxOuter && total < P.maxIter) {
        const double tgt = fmax(0.5 * P.relTol * sqrt(bb), 1e-6 * sqrt(rr));
        const float tgt2 = float(tgt * tgt);
        // r_0 = rhs, w_0 = A r_0, s_{-1} = 0, p_{-1} = 0
        Comp2 d0{0.f, 0.f, 0.f, 0.f};
        if (own) {
            float w = 0.f;
            opaque(vs);
            opaque(ns);
            w = row_product_n<27>(0x7ffffffu, i, M, vs, ns, w, [&](float a, float v, int j) {
                return __fmaf_rn(v, fromB ? b[j] : lro[j - rb], a);
            });
            const float ri = fromB ? b[i] : lro[t];
            lr[0][t] = ri;
            lw[0][t] = w;
            ls[1][t] = 0.f;
            pv = 0.f;
            dot2_acc(d0.gs, d0.gc, ri, ri);
            dot2_acc(d0.ds, d0.dc, w, ri);
        }
        Comp2 g = block_comp2(d0, shc);
        gamma = g.gs + g.gc;
        const float delta = g.ds + g.dc;
        float alpha = gamma / delta, beta = 0.f;
        int k = 0, kBest = 0;
        float gBest = gamma, xBest = own ? lx[t] : 0.f;
        while (gamma > tgt2 && total + k < P.maxIter && k - kBest < kCgStall) {
            const int c = k & 1, n = c ^ 1;  // r_k, w_k in c; s_{k-1} in n
            Comp2 dl{0.f, 0.f, 0.f, 0.f};
            if (own) {
                float w = 0.f;
                opaque(vs);
                opaque(ns);
                w = row_product_n<27>(0x7ffffffu, i, M, vs, ns, w, [&](float a, float v, int j) {
                    j -= rb;
                    return __fmaf_rn(v, r_next(lr[c][j], alpha, s_next(lw[c][j], beta, ls[n][j])), a);
                });
                const float ri = lr[c][t];
                const float si = s_next(lw[c][t], beta, ls[n][t]);
                const float rni = r_next(ri, alpha, si);
                pv = __fmaf_rn(beta, pv, ri);
                lx[t] = __fmaf_rn(alpha, pv, lx[t]);
                ls[c][t] = si;
                lr[n][t] = rni;
                lw[n][t] = w;
                dot2_acc(dl.gs, dl.gc, rni, rni);
                dot2_acc(dl.ds, dl.dc, w, rni);
            }
            g = block_comp2(dl, shc);
            const float gNew = g.gs + g.gc, dNew = g.ds + g.dc;
            const float bNew = gNew / gamma;
            alpha = gNew / (dNew - bNew * gNew / alpha);
            beta = bNew;
            gamma = gNew;
            ++k;
            if (gamma < gBest) {
                gBest = gamma;
                kBest = k;
                if (own) xBest = lx[t];
            }
        }
        total += k;
        ++outer;
        if (kBest < k) {  // back to the iterate of the smallest residual
            gamma = gBest;
            if (own) lx[t] = xBest;
            __syncthreads();
        }
        // outer residual in FP64
        loc = 0;
        if (own) {
            double acc = b[i];
            opaque(vs);
            opaque(ns);
            acc = row_product_n<27>(0x7ffffffu, i, M, vs, ns, acc, [&](double a, float v, int j) {
                return a - double(v) * double(lx[j - rb]);
            });
            lro[t] = float(acc);
            loc = acc * acc;
        }
        rr = block_sum_double(loc, shd);
        rel = bb > 0 ? sqrt(rr / bb) : 0.0;
        fromB = false;
        if (kBest == 0) break;  // no smaller residual: another outer step would repeat this one
    }
    if (own) x[i] = lx[t];
    if (threadIdx.x == 0) {
        iters[G.depth] = total;
        iters[PSR_MAX_DEPTH + 1 + G.depth] = outer;
        resid[G.depth] = sqrt(double(gamma));
        trueRel[G.depth] = rel;
    }
}

// The mixed form with several rows per thread (large depths): vectors in
// memory, the stencil read every sweep.  Instantiated twice: the CG kernel
// for definite depths (kMinres false) and the MINRES kernel for the depths
// whose operator is indefinite (kMinres true), each compiled without the
// other's path so that each keeps its own register budget.
template <bool kMinres>
__device__ __forceinline__ void cg_mixed_generic_body(int psr_bid, int psr_nbid, 
    const CgParams& P, const int* __restrict__ neigh, const float* __restrict__ val, const float* __restrict__ b,
    float* x, float* rOut, float* rbuf, float* wbuf, float* sbuf, float* __restrict__ pvec, double* partialD,
    Comp2* partialC, GroupCtl* ctlAll, int* __restrict__ iters, double* __restrict__ resid,
    double* __restrict__ trueRel, int* errFlag, const unsigned* __restrict__ slotMasks) {
    __shared__ double shd[kCgWaves];
    __shared__ Comp2 shc[kCgWaves];
    __shared__ int shFlag;
    __shared__ double shResD;
    __shared__ Comp2 shResC;
    int gi = 0;
    while (gi + 1 < P.ngroups && int(psr_bid) >= P.g[gi + 1].firstWg) ++gi;
    const CgGroup G = P.g[gi];
    const int local = psr_bid - G.firstWg;
    const int r0 = G.rowBegin + local * G.rowsPerWg;
    const int r1 = min(G.rowBegin + G.rows, r0 + G.rowsPerWg);
    const int M = P.M;
    double* partD = partialD + 2 * G.firstWg;
    Comp2* partC = partialC + 2 * G.firstWg;
    GroupCtl* ctl = ctlAll + gi;
    unsigned phase = 0;
    const bool multi = G.wgs > 1;
    if constexpr (!kMinres) {
        if (!multi && G.rows <= kCgThreads) {
            cg_small_mixed(P, G, neigh, val, b, x, iters, resid, trueRel, shd, shc);
            return;
        }
    }
    const unsigned slotMask = slotMasks[G.depth];

    auto sum_double = [&](double v, double& out) -> bool {
        double s = block_sum_double(v, shd);
        if (!multi) {
            out = s;
            return true;
        }
        return group_allreduce(s, out, partD, ctl, phase, G.wgs, local, P.spinLimit, errFlag, &shFlag, &shResD,
                               [&](const double* parts, int n) { return fold_double(parts, n, shd); });
    };
    auto sum_comp = [&](Comp2 v, Comp2& out) -> bool {
        Comp2 s = block_comp2(v, shc);
        if (!multi) {
            out = s;
            return true;
        }
        return group_allreduce(s, out, partC, ctl, phase, G.wgs, local, P.spinLimit, errFlag, &shFlag, &shResC,
                               [&](const Comp2* parts, int n) {
                                   Comp2 t{0.f, 0.f, 0.f, 0.f};
                                   for (int k = threadIdx.x; k < n; k += kCgThreads) comp2_merge(t, ld_agent(&parts[k]));
                                   return block_comp2(t, shc);
                               });
    };

    // x = 0; ||b||^2 in FP64 (the outer residual of x = 0 is b itself)
    double loc = 0;
    for (int i = r0 + threadIdx.x; i < r1; i += kCgThreads) {
        st_shared(&x[i], 0.f);
        double bi = b[i];
        loc += bi * bi;
    }
    double bb;
    if (!sum_double(loc, bb)) return;
    double rr = bb, rel = bb > 0 ? 1.0 : 0.0;
    const float* rhs = b;
    int total = 0, outer = 0;
    float gamma = 0.f;
    bool stalled = false;
    while (rel > P.relTol && outer < P.maxOuter && total < P.maxIter) {
        // inner target on the updated residual: half the tolerance left, no tighter than FP32 can follow
        const double tgt = fmax(0.5 * P.relTol * sqrt(bb), 1e-6 * sqrt(rr));
        const float tgt2 = float(tgt * tgt);
        if constexpr (kMinres) {
            // MINRES (Paige and Saunders) on A e = rhs, e_0 = 0, FP32 with
            // compensated sums.  Sweep k forms y_{k-1} = y'_{k-1} - c_{k-1} y_{k-2}
            // on the fly (c = alpha / beta), stores it, and computes
            // y'_k = A y_{k-1} / beta_k - (beta_k / beta_{k-1}) y_{k-2} with the
            // sums v_k . y'_k (= alpha_k) and ||y'_k||^2; v_k is a unit vector,
            // so beta_{k+1}^2 = ||y'_k||^2 - alpha_k^2 and one group reduction
            // per iteration suffices.  Iteration k's rotation is known only
            // after its reduction: its direction w_k = (v_k - eps w_{k-2} -
            // delta w_{k-1}) / gamma and the update e += phi w_k are applied in
            // the next sweep, and after the last one.
            float* Pb0 = rbuf;      // y'_k, k even
            float* Pb1 = rbuf + M;  // y'_k, k odd
            float* Qb0 = wbuf;      // y_k by k mod 3
            float* Qb1 = wbuf + M;
            float* Qb2 = sbuf;
            float* W1 = sbuf + M;   // w_{k-2}, own rows only
            float* W2 = pvec;       // w_{k-1}, own rows only
            auto Qsel = [&](int k) -> float* { const int m = k % 3; return m == 0 ? Qb0 : (m == 1 ? Qb1 : Qb2); };
            const float beta1 = float(sqrt(rr));
            const float tgtf = float(tgt);
            float beta = beta1, oldb = 1.f, cPrev = 0.f;
            float cs = -1.f, sn = 0.f, dbar = 0.f, epsln = 0.f, phibar = beta1;
            float lagEps = 0.f, lagDelta = 0.f, lagGamma = 1.f, lagPhi = 0.f;
            int it = 1, kdone = 0;
            while (beta1 > tgtf && total < P.maxIter) {
                const float* Pprev = (it & 1) ? Pb0 : Pb1;  // y'_{it-1}
                float* Pnew = (it & 1) ? Pb1 : Pb0;         // y'_it
                const float* Qold = Qsel(it + 1);           // y_{it-2}
                float* Qcur = Qsel(it + 2);                 // y_{it-1}
                const float invB = 1.f / beta;
                const float r1c = it >= 2 ? beta / oldb : 0.f;
                const float invOld = 1.f / oldb;
                Comp2 dl{0.f, 0.f, 0.f, 0.f};
                for (int i = r0 + threadIdx.x; i < r1; i += kCgThreads) {
                    float av = 0.f;
                    if (it == 1)
                        av = row_product(slotMask, i, M, val, neigh, av, [&](float a, float v, int j) {
                            return __fmaf_rn(v, ld_shared(&rhs[j]), a);
                        });
                    else
                        av = row_product(slotMask, i, M, val, neigh, av, [&](float a, float v, int j) {
                            return __fmaf_rn(v, __fmaf_rn(-cPrev, ld_shared(&Qold[j]), ld_shared(&Pprev[j])), a);
                        });
                    const float r1i = it >= 2 ? ld_shared(&Qold[i]) : 0.f;  // y_{it-2}
                    const float yi = it == 1 ? ld_shared(&rhs[i]) : __fmaf_rn(-cPrev, r1i, ld_shared(&Pprev[i]));
                    st_shared(&Qcur[i], yi);
                    const float ypi = __fmaf_rn(-r1c, r1i, av * invB);
                    st_shared(&Pnew[i], ypi);
                    dot2_acc(dl.gs, dl.gc, yi * invB, ypi);
                    dot2_acc(dl.ds, dl.dc, ypi, ypi);
                    float w1 = 0.f, w2 = 0.f;
                    if (it >= 2) {
                        w1 = W1[i];
                        w2 = W2[i];
                        const float wk = (r1i * invOld - lagEps * w1 - lagDelta * w2) / lagGamma;
                        st_shared(&x[i], __fmaf_rn(lagPhi, wk, ld_shared(&x[i])));
                        w1 = w2;
                        w2 = wk;
                    }
                    W1[i] = w1;
                    W2[i] = w2;
                }
                Comp2 g;
                if (!sum_comp(dl, g)) return;
                const float alfa = g.gs + g.gc, yy = g.ds + g.dc;
                const float betaN = sqrtf(fmaxf(yy - alfa * alfa, 0.f));
                const float oldeps = epsln;
                const float delta = cs * dbar + sn * alfa;
                const float gbar = sn * dbar - cs * alfa;
                epsln = sn * betaN;
                dbar = -cs * betaN;
                const float gam = fmaxf(sqrtf(gbar * gbar + betaN * betaN), 1e-30f);
                cs = gbar / gam;
                sn = betaN / gam;
                const float phi = cs * phibar;
                phibar = sn * phibar;
                lagEps = oldeps;
                lagDelta = delta;
                lagGamma = gam;
                lagPhi = phi;
                cPrev = alfa / beta;
                oldb = beta;
                beta = betaN;
                ++kdone;
                gamma = phibar * phibar;
                if (!(phibar > tgtf) || total + kdone >= P.maxIter || !(betaN > 0.f)) break;
                ++it;
            }
            if (kdone > 0) {
                // the last iteration's update: v = y_{it-1} / beta_it
                const float* Qcur = Qsel(it + 2);
                const float invOld = 1.f / oldb;
                for (int i = r0 + threadIdx.x; i < r1; i += kCgThreads) {
                    const float wk = (ld_shared(&Qcur[i]) * invOld - lagEps * W1[i] - lagDelta * W2[i]) / lagGamma;
                    st_shared(&x[i], __fmaf_rn(lagPhi, wk, ld_shared(&x[i])));
                }
            }
            total += kdone;
            ++outer;
            if (kdone == 0) break;
            // the last update wrote x after the last group reduction: one more
            // reduction orders it before the outer residual reads neighbours' x
            double fence;
            if (!sum_double(0.0, fence)) return;
        } else {
            // r_0 = rhs, w_0 = A r_0, s_{-1} = 0, p_{-1} = 0
            Comp2 d0{0.f, 0.f, 0.f, 0.f};
            for (int i = r0 + threadIdx.x; i < r1; i += kCgThreads) {
                float w = 0.f;
                w = row_product(slotMask, i, M, val, neigh, w, [&](float a, float v, int j) {
                    return __fmaf_rn(v, ld_shared(&rhs[j]), a);
                });
                float ri = ld_shared(&rhs[i]);
                st_shared(&rbuf[i], ri);
                st_shared(&wbuf[i], w);
                st_shared(&sbuf[M + i], 0.f);
                pvec[i] = 0.f;
                dot2_acc(d0.gs, d0.gc, ri, ri);
                dot2_acc(d0.ds, d0.dc, w, ri);
            }
            Comp2 g;
            if (!sum_comp(d0, g)) return;
            gamma = g.gs + g.gc;
            float delta = g.ds + g.dc;
            float alpha = gamma / delta, beta = 0.f;
            // the iterate of the smallest residual goes to rOut (free until
            // the outer residual) in the sweep after its reduction found it
            int k = 0, kBest = 0;
            float gBest = gamma;
            bool curBest = true;
            while (gamma > tgt2 && total + k < P.maxIter && k - kBest < kCgStall) {
                const float* rk = rbuf + (k & 1) * M;
                const float* wk = wbuf + (k & 1) * M;
                const float* sp = sbuf + ((k + 1) & 1) * M;  // s_{k-1}
                float* rn = rbuf + ((k + 1) & 1) * M;
                float* wn = wbuf + ((k + 1) & 1) * M;
                float* sk = sbuf + (k & 1) * M;
                Comp2 dl{0.f, 0.f, 0.f, 0.f};
                for (int i = r0 + threadIdx.x; i < r1; i += kCgThreads) {
                    float w = 0.f;
                    w = row_product(slotMask, i, M, val, neigh, w, [&](float a, float v, int j) {
                        const float rj = r_next(ld_shared(&rk[j]), alpha, s_next(ld_shared(&wk[j]), beta, ld_shared(&sp[j])));
                        return __fmaf_rn(v, rj, a);
                    });
                    float ri = ld_shared(&rk[i]);
                    float si = s_next(ld_shared(&wk[i]), beta, ld_shared(&sp[i]));
                    float rni = r_next(ri, alpha, si);
                    float pi = __fmaf_rn(beta, pvec[i], ri);
                    pvec[i] = pi;
                    const float xo = ld_shared(&x[i]);
                    if (curBest) st_shared(&rOut[i], xo);
                    st_shared(&x[i], __fmaf_rn(alpha, pi, xo));
                    st_shared(&sk[i], si);
                    st_shared(&rn[i], rni);
                    st_shared(&wn[i], w);
                    dot2_acc(dl.gs, dl.gc, rni, rni);
                    dot2_acc(dl.ds, dl.dc, w, rni);
                }
                if (!sum_comp(dl, g)) return;
                const float gNew = g.gs + g.gc, dNew = g.ds + g.dc;
                const float bNew = gNew / gamma;
                alpha = gNew / (dNew - bNew * gNew / alpha);
                beta = bNew;
                gamma = gNew;
                ++k;
                curBest = gamma < gBest;
                if (curBest) {
                    gBest = gamma;
                    kBest = k;
                }
            }
            total += k;
            ++outer;
            if (!curBest) {
                // back to the iterate of the smallest residual (kept in rOut);
                // one more reduction orders it before the outer residual
                gamma = gBest;
                for (int i = r0 + threadIdx.x; i < r1; i += kCgThreads) st_shared(&x[i], ld_shared(&rOut[i]));
                double fence;
                if (!sum_double(0.0, fence)) return;
            }
            stalled = kBest == 0;
        }
        // outer residual in FP64
        loc = 0;
        for (int i = r0 + threadIdx.x; i < r1; i += kCgThreads) {
            double acc = b[i];
            acc = row_product(slotMask, i, M, val, neigh, acc, [&](double a, float v, int j) {
                return a - double(v) * double(ld_shared(&x[j]));
            });
            st_shared(&rOut[i], float(acc));
            loc += acc * acc;
        }
        if (!sum_double(loc, rr)) return;
        rel = bb > 0 ? sqrt(rr / bb) : 0.0;
        rhs = rOut;
        if (stalled) break;  // no smaller residual: another outer step would repeat this one
    }
    if (local == 0 && threadIdx.x == 0) {
        iters[G.depth] = total;
        iters[PSR_MAX_DEPTH + 1 + G.depth] = outer;
        resid[G.depth] = sqrt(double(gamma));
        trueRel[G.depth] = rel;
    }
}
template <class... A>
__device__ __forceinline__ void cg_mixed_all_depths_body(int bid, int nbid, const A&... a) {
    cg_mixed_generic_body<false>(bid, nbid, a...);
}
template <class... A>
__device__ __forceinline__ void cg_mixed_minres_body(int bid, int nbid, const A&... a) {
    cg_mixed_generic_body<true>(bid, nbid, a...);
}
__global__ void __launch_bounds__(kCgThreads) __attribute__((amdgpu_waves_per_eu(kCgMixedGenericWaves))) cg_mixed_all_depths(
    CgParams P, const int* __restrict__ neigh, const float* __restrict__ val, const float* __restrict__ b,
    float* x, float* rOut, float* rbuf, float* wbuf, float* sbuf, float* __restrict__ pvec, double* partialD,
    Comp2* partialC, GroupCtl* ctlAll, int* __restrict__ iters, double* __restrict__ resid,
    double* __restrict__ trueRel, int* errFlag, const unsigned* __restrict__ slotMasks) {
    cg_mixed_all_depths_body(blockIdx.x, gridDim.x, P, neigh, val, b, x, rOut, rbuf, wbuf, sbuf, pvec, partialD, partialC, ctlAll, iters, resid, trueRel, errFlag, slotMasks);
}
PSR_BATCHABLE_WAVES(cg_mixed_all_depths, kCgThreads, kCgMixedGenericWaves)
__global__ void __launch_bounds__(kCgThreads) __attribute__((amdgpu_waves_per_eu(kCgMinresWaves))) cg_mixed_minres(
    CgParams P, const int* __restrict__ neigh, const float* __restrict__ val, const float* __restrict__ b,
    float* x, float* rOut, float* rbuf, float* wbuf, float* sbuf, float* __restrict__ pvec, double* partialD,
    Comp2* partialC, GroupCtl* ctlAll, int* __restrict__ iters, double* __restrict__ resid,
    double* __restrict__ trueRel, int* errFlag, const unsigned* __restrict__ slotMasks) {
    cg_mixed_minres_body(blockIdx.x, gridDim.x, P, neigh, val, b, x, rOut, rbuf, wbuf, sbuf, pvec, partialD, partialC, ctlAll, iters, resid, trueRel, errFlag, slotMasks);
}
PSR_BATCHABLE_WAVES(cg_mixed_minres, kCgThreads, kCgMinresWaves)



// --- MINRES with the vectors on chip -----------------------------------------
// The same solve as cg_mixed_minres, bit for bit (rows to threads, order of the
// sums and of every operation), for a depth whose operator stores the diagonal
// and the six faces: each of its workgroups keeps its rows' vectors where it
// works on them.  Per sweep cg_mixed_minres moves about 100 bytes a row through
// the caches and gathers 14 uncached values a row; here
//   * x, the two directions w and y' stay in registers, R rows a thread;
//   * y_{k-1} is formed once per row, in LDS, where all neighbours in the
//     workgroup read it (95% of them: a workgroup's rows are a patch of the
//     surface in Morton order), and once per neighbour outside it (a ghost: its
//     owner's record {y_{k-2}, y'_{k-1}}, one 8-byte load);
//   * the six columns of a row are 16-bit LDS places, the weights are one
//     constant per slot (checked row by row);
//   * only rows with a neighbour outside the workgroup write a record.
// A workgroup whose rows do not fit this (other weights, more ghosts than
// places) reads its neighbours' records instead, row by row, and stores all of
// its own.  10000 iterations at depth 9: 2.76M rows (displaced sphere) 872 ms
// with every vector in memory, 174 ms here (17 us a sweep: about 11 us of LDS
// reads and arithmetic, the rest the reduction); 723k rows 285 -> 75 ms, 141k
// rows 136 -> 63 ms (6 us a sweep, nearly all of it the reduction).
//
// Group reduction: every workgroup stores its block total (two stamped slots);
// four collector workgroups each fold one wave's share of the totals, in
// group_allreduce's order, and publish it in kResultCopies copies; every
// workgroup merges the four.
constexpr int kResultCopies = 16;
constexpr int kCollectors = kCgWaves;  // a collector per wave of the fold
constexpr int kFoldParts = 5;  // groups of at most kFoldParts * kCgThreads workgroups
constexpr size_t minres_result_slots() { return size_t(2) * kResultCopies * kCollectors * 2; }  // of a group
// Sum of the group's block totals `mine`, as group_allreduce folds them.  slots:
// [2][G][2] block totals, then [2][kResultCopies][kCollectors][2] wave totals,
// by phase parity, zero before the launch; a slot holds two words of payload and
// the phase.  The block's stores of the sweep have completed (its waves waited
// for them before the barrier that formed `mine`).
__device__ __forceinline__ bool collect_comp2(const Comp2& mine, Comp2& out, float4* slots, int G, int local,
                                              unsigned& phase, unsigned spinLimit, int* errFlag, Comp2* sh,
                                              Comp2* part) {
    __shared__ int shOk;
    ++phase;
    const float stamp = __uint_as_float(phase);
    const int lane = __lane_id(), wave = threadIdx.x / PSR_WAVE;
    const __amdgpu_buffer_rsrc_t in = vec_rsrc(slots + size_t(phase & 1u) * 2 * G, sizeof(float4) * 2 * size_t(G));
    float4* results = slots + size_t(4) * G + size_t(phase & 1u) * kResultCopies * kCollectors * 2;
    const __amdgpu_buffer_rsrc_t res = vec_rsrc(results, sizeof(float4) * kResultCopies * kCollectors * 2);
    if (threadIdx.x < 2)
        st_vec4(in, local * 2 + int(threadIdx.x),
                threadIdx.x == 0 ? make_float4(mine.gs, mine.gc, stamp, 0.f) : make_float4(mine.ds, mine.dc, stamp, 0.f));
    auto give_up = [&](unsigned spins) {
        if (spins < spinLimit && ((spins & 63u) != 63u || !__hip_atomic_load(errFlag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)))
            return false;
        __hip_atomic_store(errFlag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return true;
    };
    for (int w = local; w < kCollectors; w += G) {
        // thread (wave j, lane) reads the total of workgroup 64 w + lane + 256 j
        // (and j + 4 beyond 1024 workgroups)
        if (threadIdx.x == 0) shOk = 1;
        __syncthreads();
        for (int j = wave; j < kFoldParts; j += kCgWaves) {
            const int k = PSR_WAVE * w + lane + kCgThreads * j;
            Comp2 c{0.f, 0.f, 0.f, 0.f};
            if (k < G) {
                for (unsigned spins = 0;; ++spins) {
                    const float4 a = ld_vec4(in, 2 * k), b = ld_vec4(in, 2 * k + 1);
                    if (__float_as_uint(a.z) == phase && __float_as_uint(b.z) == phase) {
                        c = Comp2{a.x, a.y, b.x, b.y};
                        break;
                    }
                    if (give_up(spins)) {
                        shOk = 0;
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                }
            }
            part[j * PSR_WAVE + lane] = c;
        }
        __syncthreads();
        if (shOk == 0) return false;
        if (wave == 0) {
            Comp2 t{0.f, 0.f, 0.f, 0.f};
            for (int j = 0; PSR_WAVE * w + kCgThreads * j < G; ++j)
                if (PSR_WAVE * w + lane + kCgThreads * j < G) comp2_merge(t, part[j * PSR_WAVE + lane]);
            t = wave_comp2(t);
            if (lane < 2 * kResultCopies)
                st_vec4(res, ((lane >> 1) * kCollectors + w) * 2 + (lane & 1),
                        (lane & 1) == 0 ? make_float4(t.gs, t.gc, stamp, 0.f) : make_float4(t.ds, t.dc, stamp, 0.f));
        }
        __syncthreads();
    }
    if (wave == 0) {
        const int at = (local % kResultCopies) * kCollectors * 2 + lane;
        bool ok = true;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        for (unsigned spins = 0;; ++spins) {
            if (lane < 2 * kCollectors) v = ld_vec4(res, at);
            if (__ballot(lane < 2 * kCollectors && __float_as_uint(v.z) != phase) == 0) break;
            if (__ballot(give_up(spins)) != 0) {
                ok = false;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        if (lane < 2 * kCollectors) {
            float* d = (lane & 1) ? &sh[lane >> 1].ds : &sh[lane >> 1].gs;
            d[0] = v.x;
            d[1] = v.y;
        }
        if (lane == 0) shOk = ok ? 1 : 0;
    }
    __syncthreads();
    out = sh[0];
    for (int k = 1; k < kCollectors; ++k) comp2_merge(out, sh[k]);
    const bool ok = shOk != 0;
    __syncthreads();
    return ok;
}

constexpr unsigned kFaceSlots = 1u << 4 | 1u << 10 | 1u << 12 | 1u << 13 | 1u << 14 | 1u << 16 | 1u << 22;
// Ghost places of a workgroup: about 1000-1900 of 4096 rows' neighbours lie
// outside it on the displaced sphere, 600-1200 of 2048 rows'.
template <int R>
constexpr int minres_ghosts() { return R == 16 ? 3072 : (R == 8 ? 2048 : 1536); }

template <int R>
__device__ __forceinline__ void cg_minres_chip(int psr_bid, const CgParams& P, const int* __restrict__ neigh,
                                               const float* __restrict__ val, const float* __restrict__ b, float* x,
                                               float* rOut, float2* rec, float* __restrict__ avScratch,
                                               double* partialD, float4* slotsAll, GroupCtl* ctlAll,
                                               int* __restrict__ iters, double* __restrict__ resid,
                                               double* __restrict__ trueRel, int* errFlag,
                                               const unsigned* __restrict__ slotMasks, const int* __restrict__ q1Fired) {
    constexpr int kRows = R * kCgThreads, kGhosts = minres_ghosts<R>(), kZero = kRows + kGhosts;
    static_assert(kGhosts % kCgThreads == 0, "whole rounds of ghosts");
    static_assert(4 * kZero < 65536, "16-bit byte offsets");
    static_assert(sizeof(Comp2) * PSR_WAVE * kFoldParts <= sizeof(float) * kGhosts, "the fold works in the ghosts' place");
    __shared__ __align__(16) float ly[kRows + kGhosts + 1];  // y_{k-1} of the rows, of the ghosts, and a zero
    __shared__ int lg[kGhosts];                // the ghosts' rows
    __shared__ unsigned lw[7];
    __shared__ int shGhosts, shSlow;
    __shared__ double shd[kCgWaves];
    __shared__ Comp2 shc[kCgWaves];
    __shared__ int shFlag;
    __shared__ double shResD;
    int gi = 0;
    while (gi + 1 < P.ngroups && int(psr_bid) >= P.g[gi + 1].firstWg) ++gi;
    const CgGroup G = P.g[gi];
    const int local = psr_bid - G.firstWg, t = int(threadIdx.x);
    const int r0 = G.rowBegin + local * G.rowsPerWg;
    const int rows = max(0, min(G.rowBegin + G.rows, r0 + G.rowsPerWg) - r0);  // at most kRows (host)
    const int M = P.M;
    double* partD = partialD + 2 * G.firstWg;
    float4* slots = slotsAll + minres_result_slots() * gi + size_t(4) * G.firstWg;
    GroupCtl* ctl = ctlAll + gi;
    unsigned phase = 0, phaseC = 0;
    const bool multi = G.wgs > 1;
    const unsigned slotMask = slotMasks[G.depth];
    auto sum_double = [&](double v, double& out) -> bool {
        if (multi) __builtin_amdgcn_s_waitcnt(0);  // every wave's stores complete before the total
        double s = block_sum_double(v, shd);
        if (!multi) {
            out = s;
            return true;
        }
        return group_allreduce(s, out, partD, ctl, phase, G.wgs, local, P.spinLimit, errFlag, &shFlag, &shResD,
                               [&](const double* parts, int n) { return fold_double(parts, n, shd); });
    };

    auto y_at = [&](unsigned byteOffset) { return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(ly) + byteOffset); };
    // Row l's siblings lie at l ^ 4, l ^ 2 and l ^ 1 (x, y, z); the slots of its other three faces are the same for
    // all rows of a thread (256 rows apart).  Those faces' columns as byte offsets into ly: x and y in one word, the
    // z of two rows in another.
    const bool bx = (t & 4) != 0, by = (t & 2) != 0, bz = (t & 1) != 0;
    if (t < 7) lw[t] = 0u;
    if (t == 0) shGhosts = 0, shSlow = slotMask != kFaceSlots ? 1 : 0, ly[kZero] = 0.f;
    __syncthreads();
    unsigned placeXY[R], placeZ[(R + 1) / 2];
    unsigned boundary = 0u;  // bit k: row k has a neighbour outside the workgroup, and so a reader there
    {
        const int slotOf[7] = {bx ? 22 : 4, by ? 16 : 10, bz ? 14 : 12, bx ? 4 : 22, by ? 10 : 16, bz ? 12 : 14, 13};
        float w[7] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        unsigned bad = 0u;
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int l = k * kCgThreads + t, i = r0 + max(0, min(l, rows - 1));
            const bool own = l < rows;
            unsigned at[3];
#pragma unroll
            for (int q = 0; q < 7; ++q) {
                const size_t e = size_t(slotOf[q]) * M + i;
                const float v = val[e];
                const int j = neigh[e];
                bad |= own && v != 0.f && w[q] != 0.f && w[q] != v ? 1u : 0u;
                if (own && v != 0.f) w[q] = v;
                if (q >= 3) {  // a sibling or the row itself
                    const int flip = q == 3 ? 4 : (q == 4 ? 2 : (q == 5 ? 1 : 0));
                    bad |= own && (v == 0.f || j != r0 + (l ^ flip) || (l ^ flip) >= rows) ? 1u : 0u;
                    continue;
                }
                const bool outside = own && j >= 0 && unsigned(j - r0) >= unsigned(rows);
                if (outside) boundary |= 1u << k;
                const bool stored = own && v != 0.f;
                int p = stored ? j - r0 : kZero;
                if (stored && outside) {
                    const int h = atomicAdd(&shGhosts, 1);
                    p = kRows + min(h, kGhosts - 1);
                    if (h < kGhosts) lg[h] = j;
                }
                bad |= stored && j < 0 ? 1u : 0u;
                at[q] = unsigned(4 * p) & 0xffffu;
            }
            placeXY[k] = at[0] | at[1] << 16;
            placeZ[k / 2] = k % 2 == 0 ? at[2] : placeZ[k / 2] | at[2] << 16;
            // packed here and now: the rows' state fills the registers
            asm volatile("" : "+v"(placeXY[k]), "+v"(placeZ[k / 2]), "+v"(boundary), "+v"(bad) : : "memory");
#pragma unroll
            for (int q = 0; q < 7; ++q) asm volatile("" : "+v"(w[q]));
        }
        const int wordOf[7] = {bx ? 5 : 0, by ? 4 : 1, bz ? 3 : 2, bx ? 0 : 5, by ? 1 : 4, bz ? 2 : 3, 6};
#pragma unroll
        for (int q = 0; q < 7; ++q)
            if (w[q] != 0.f) atomicMax(&lw[wordOf[q]], __float_as_uint(w[q]));
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 7; ++q)
            if (w[q] != 0.f && __float_as_uint(w[q]) != lw[wordOf[q]]) bad = 1u;
        if (bad) shSlow = 1;
        __syncthreads();
    }
    const int ghosts = __builtin_amdgcn_readfirstlane(shGhosts);
    const bool slow = __builtin_amdgcn_readfirstlane(shSlow) != 0 || ghosts > kGhosts;
    // neighbour tables that the level-local child 0 rule changed need not be symmetric
    if (slow || *q1Fired != 0) {
        boundary = 0u;
        for (int k = 0; k < R; ++k) boundary |= k * kCgThreads + t < rows ? 1u << k : 0u;
    }
    float wq[7];
#pragma unroll
    for (int q = 0; q < 7; ++q) wq[q] = __uint_as_float(__builtin_amdgcn_readfirstlane(lw[q]));

    // x = 0; ||b||^2 in FP64 (the outer residual of x = 0 is b itself)
    float xr[R];
    double loc = 0;
#pragma unroll
    for (int k = 0; k < R; ++k) xr[k] = 0.f;
#pragma unroll 1
    for (int l = t; l < rows; l += kCgThreads) {
        const int i = r0 + l;
        {
            st_shared(&x[i], 0.f);
            const double bi = b[i];
            loc += bi * bi;
        }
    }
    double bb;
    if (!sum_double(loc, bb)) return;
    double rr = bb, rel = bb > 0 ? 1.0 : 0.0;
    const float* rhs = b;
    int total = 0, outer = 0;
    float gamma = 0.f;
    while (rel > P.relTol && outer < P.maxOuter && total < P.maxIter) {
        const double tgt = fmax(0.5 * P.relTol * sqrt(bb), 1e-6 * sqrt(rr));
        const float beta1 = float(sqrt(rr));
        const float tgtf = float(tgt);
        float beta = beta1, oldb = 1.f, cPrev = 0.f;
        float cs = -1.f, sn = 0.f, dbar = 0.f, epsln = 0.f, phibar = beta1;
        float lagEps = 0.f, lagDelta = 0.f, lagGamma = 1.f, lagPhi = 0.f;
        int it = 1, kdone = 0;
        // y_{-1} = 0 and y'_0 = rhs make the first sweep one like the others
        float yp[R], w1[R], w2[R];
#pragma unroll
        for (int k = 0; k < R; ++k) {
            int l = k * kCgThreads + t;
            asm volatile("" : "+v"(l));  // no address is kept from loop to loop
            const int i = r0 + l;
            yp[k] = l < rows ? ld_shared(&rhs[i]) : 0.f;
            w1[k] = w2[k] = 0.f;
            ly[l] = 0.f;
            if (l < rows) st_vec2(vec_rsrc(rec, sizeof(float2) * size_t(M)), i, make_float2(0.f, yp[k]));
        }
        double fence;
        if (!sum_double(0.0, fence)) return;  // the records are read by other workgroups
        while (beta1 > tgtf && total < P.maxIter) {
            // record buffer (it + 1) & 1 holds {y_{it-2}, y'_{it-1}}, it & 1 receives {y_{it-1}, y'_it}
            const __amdgpu_buffer_rsrc_t in = vec_rsrc(rec + size_t((it + 1) & 1) * M, sizeof(float2) * size_t(M));
            const __amdgpu_buffer_rsrc_t onto = vec_rsrc(rec + size_t(it & 1) * M, sizeof(float2) * size_t(M));
            const float invB = 1.f / beta;
            const float r1c = it >= 2 ? beta / oldb : 0.f;
            const float invOld = 1.f / oldb;
            // the rows' offsets and bounds are formed anew every sweep, not kept
            int tt = t, base = r0 + t;
            unsigned bnd = boundary;
            asm volatile("" : "+v"(tt), "+v"(base), "+v"(bnd));
            // the ghosts' records are on their way while the rows' y are formed
            constexpr int kEarly = 6;
            float2 g[kEarly];
            if (!slow) {
#pragma unroll
                for (int m = 0; m < kEarly; ++m) {
                    const int h = m * kCgThreads + tt;
                    g[m] = h < ghosts ? ld_vec2(in, lg[h]) : make_float2(0.f, 0.f);
                }
            }
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const int l = k * kCgThreads + t;
                const float r1 = ly[l];  // y_{it-2}
                // the previous iteration's direction and update (zero in the first sweep)
                const float num = __fmaf_rn(-lagDelta, w2[k], __fmaf_rn(r1, invOld, -__fmul_rn(lagEps, w1[k])));
                const float wk = num / lagGamma;
                xr[k] = __fmaf_rn(lagPhi, wk, xr[k]);
                w1[k] = w2[k];
                w2[k] = wk;
                ly[l] = __fmaf_rn(-cPrev, r1, yp[k]);
                yp[k] = r1;
                // the state stays in its registers from sweep to sweep
                asm volatile("" : "+v"(xr[k]), "+v"(w1[k]), "+v"(w2[k]), "+v"(yp[k]));
            }
            if (!slow) {
#pragma unroll
                for (int m = 0; m < kEarly; ++m) {
                    const int h = m * kCgThreads + tt;
                    if (h < ghosts) ly[kRows + h] = __fmaf_rn(-cPrev, g[m].x, g[m].y);
                }
                for (int h = kEarly * kCgThreads + tt; h < ghosts; h += kCgThreads) {
                    const float2 n = ld_vec2(in, lg[h]);
                    ly[kRows + h] = __fmaf_rn(-cPrev, n.x, n.y);
                }
            } else {
                for (int i = r0 + t; i < r0 + rows; i += kCgThreads) {
                    float av = 0.f;
#pragma unroll 1
                    for (int q = 0; q < 27; ++q) {
                        const float v = val[size_t(q) * M + i];
                        if (v == 0.f) continue;  // a term of weight zero adds nothing
                        const float2 n = ld_vec2(in, neigh[size_t(q) * M + i]);
                        av = __fmaf_rn(v, __fmaf_rn(-cPrev, n.x, n.y), av);
                    }
                    avScratch[i] = av;
                }
            }
            __syncthreads();
            Comp2 dl{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const int l = k * kCgThreads + t;
                const float yi = ly[l];
                // unpacked anew every sweep: 3 R addresses do not fit the registers
                unsigned pxy = placeXY[k], pz = placeZ[k / 2];
                asm volatile("" : "+v"(pxy), "+v"(pz));
                const float xe = y_at(pxy & 0xffffu), ye = y_at(pxy >> 16), ze = y_at(k % 2 == 0 ? pz & 0xffffu : pz >> 16);
                const float xs = ly[k * kCgThreads + (tt ^ 4)], ys = ly[k * kCgThreads + (tt ^ 2)],
                            zs = ly[k * kCgThreads + (tt ^ 1)];
                float av = __fmaf_rn(wq[0], bx ? xs : xe, 0.f);
                av = __fmaf_rn(wq[1], by ? ys : ye, av);
                av = __fmaf_rn(wq[2], bz ? zs : ze, av);
                av = __fmaf_rn(wq[6], yi, av);
                av = __fmaf_rn(wq[3], bz ? ze : zs, av);
                av = __fmaf_rn(wq[4], by ? ye : ys, av);
                av = __fmaf_rn(wq[5], bx ? xe : xs, av);
                if (slow) av = rows - tt > k * kCgThreads ? avScratch[base + k * kCgThreads] : 0.f;
                // rows past the workgroup's last are zero throughout and add nothing to the sums
                yp[k] = __fmaf_rn(-r1c, yp[k], __fmul_rn(av, invB));
                dot2_acc(dl.gs, dl.gc, __fmul_rn(yi, invB), yp[k]);
                dot2_acc(dl.ds, dl.dc, yp[k], yp[k]);
                if (bnd >> k & 1u) st_vec2(onto, base + k * kCgThreads, make_float2(yi, yp[k]));
                asm volatile("" : "+v"(yp[k]), "+v"(dl.gs), "+v"(dl.gc), "+v"(dl.ds), "+v"(dl.dc));
            }
            dl = wave_comp2(dl);
            __builtin_amdgcn_s_waitcnt(0);  // the records have left before the total does
            if (__lane_id() == 0) shc[t / PSR_WAVE] = dl;
            __syncthreads();
            Comp2 gsum = shc[0];
            for (int k = 1; k < kCgWaves; ++k) comp2_merge(gsum, shc[k]);
            __syncthreads();
            if (multi && !collect_comp2(gsum, gsum, slots, G.wgs, local, phaseC, P.spinLimit, errFlag, shc,
                                        reinterpret_cast<Comp2*>(ly + kRows)))
                return;
            const float alfa = gsum.gs + gsum.gc, yy = gsum.ds + gsum.dc;
            // one scalar per workgroup: kept in scalar registers between the sweeps
            auto uni = [](float v) { return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v))); };
            const float betaN = sqrtf(fmaxf(__fmaf_rn(-alfa, alfa, yy), 0.f));
            const float oldeps = epsln;
            const float delta = __fmaf_rn(cs, dbar, __fmul_rn(sn, alfa));
            const float gbar = __fmaf_rn(dbar, sn, -__fmul_rn(cs, alfa));
            epsln = uni(sn * betaN);
            dbar = uni(-cs * betaN);
            const float gam = fmaxf(sqrtf(__fmaf_rn(gbar, gbar, __fmul_rn(betaN, betaN))), 1e-30f);
            cs = uni(gbar / gam);
            sn = uni(betaN / gam);
            const float phi = cs * phibar;
            phibar = uni(sn * phibar);
            lagEps = uni(oldeps);
            lagDelta = uni(delta);
            lagGamma = uni(gam);
            lagPhi = uni(phi);
            cPrev = uni(alfa / beta);
            oldb = beta;
            beta = uni(betaN);
            ++kdone;
            gamma = phibar * phibar;
            if (!(phibar > tgtf) || total + kdone >= P.maxIter || !(betaN > 0.f)) break;
            ++it;
        }
        if (kdone > 0) {
            // the last iteration's update: v = y_{it-1} / beta_it
            const float invOld = 1.f / oldb;
#pragma unroll
            for (int k = 0; k < R; ++k) {
                int l = k * kCgThreads + t;
                asm volatile("" : "+v"(l));
                const float num = __fmaf_rn(-lagDelta, w2[k], __fmaf_rn(ly[l], invOld, -__fmul_rn(lagEps, w1[k])));
                xr[k] = __fmaf_rn(lagPhi, num / lagGamma, xr[k]);
                if (l < rows) st_shared(&x[r0 + l], xr[k]);
            }
        }
        total += kdone;
        ++outer;
        if (kdone == 0) break;
        // orders x before the outer residual reads neighbours' x
        if (!sum_double(0.0, fence)) return;
        // outer residual in FP64
        loc = 0;
        for (int i = r0 + t; i < r0 + rows; i += kCgThreads) {
            double acc = b[i];
#pragma unroll 1
            for (int q = 0; q < 27; ++q) {
                const float v = val[size_t(q) * M + i];
                if (v != 0.f) acc -= double(v) * double(ld_shared(&x[neigh[size_t(q) * M + i]]));  // the product is exact
            }
            st_shared(&rOut[i], float(acc));
            loc += acc * acc;
        }
        if (!sum_double(loc, rr)) return;
        rel = bb > 0 ? sqrt(rr / bb) : 0.0;
        rhs = rOut;
    }
    if (local == 0 && t == 0) {
        iters[G.depth] = total;
        iters[PSR_MAX_DEPTH + 1 + G.depth] = outer;
        resid[G.depth] = sqrt(double(gamma));
        trueRel[G.depth] = rel;
    }
}
// R rows a thread at most, and the waves per SIMD its registers allow (with
// the launch's residency): 16 rows and 3 waves hold 3.1M rows, 8 rows and 5
// waves all depths of workgroups of 2048 rows or fewer.
#define PSR_MINRES_CHIP(NAME, R, WAVES)                                                                                 \
    template <class... A>                                                                                               \
    __device__ __forceinline__ void NAME##_body(int bid, int, const A&... a) {                                          \
        cg_minres_chip<R>(bid, a...);                                                                                   \
    }                                                                                                                   \
    __global__ void __launch_bounds__(kCgThreads) __attribute__((amdgpu_waves_per_eu(WAVES))) NAME(                     \
        CgParams P, const int* __restrict__ neigh, const float* __restrict__ val, const float* __restrict__ b,          \
        float* x, float* rOut, float2* rec, float* __restrict__ avScratch, double* partialD, float4* slots,             \
        GroupCtl* ctlAll, int* __restrict__ iters, double* __restrict__ resid, double* __restrict__ trueRel,            \
        int* errFlag, const unsigned* __restrict__ slotMasks, const int* __restrict__ q1Fired) {                        \
        cg_minres_chip<R>(blockIdx.x, P, neigh, val, b, x, rOut, rec, avScratch, partialD, slots, ctlAll, iters, resid, \
                          trueRel, errFlag, slotMasks, q1Fired);                                                        \
    }                                                                                                                   \
    PSR_BATCHABLE_WAVES(NAME, kCgThreads, WAVES)
PSR_MINRES_CHIP(cg_minres_chip16, 16, 3)
PSR_MINRES_CHIP(cg_minres_chip8, 8, 5)
PSR_MINRES_CHIP(cg_minres_chip4, 4, 5)

// --- implicit function at points (LaplacianSolver.cu:85-118, 269-305) ------
// Neighbour columns: d_x of neighbour i of every node, and, when the
// level-local child 0 rule changed a parent, its basis parameters as well, so
// the 27 terms of a node need no dependent index loads.  (The kernels of a
// regular octree take the centres from the node grid; the few that need an
// ancestor's neighbour centres read them through the neighbour table.)
// Also clears the nZero words at zero (the mesh stage's node tables and face
// marks) and, when the octree is regular, the nDense dense d_x grid cells,
// which saves the mesh stage launches of its own.
// Bound by memory: 8 bytes an entry and 4 a cell, and d_x of the neighbours from
// the cache.  With 16-byte loads and stores in place of an entry a thread: 32
// clouds 366 -> 171 us (0.8 GB), 200k torus at depth 7 7.8 -> 7.3 us, 300k points
// at depth 8 26 us as before (134 MB, at the rate of a copy).
constexpr int kColumnItems = 4;
__device__ __forceinline__ void neighbour_columns_body(int psr_bid, int psr_nbid, int M, const int* __restrict__ neigh,
                                                              const float4* __restrict__ basis,
                                                              const float* __restrict__ dx,
                                                              float4* __restrict__ nbrCol, float* __restrict__ dCol,
                                                              unsigned* __restrict__ zero, size_t nZero,
                                                              float* __restrict__ dense, size_t nDense,
                                                              const int* __restrict__ q1Fired,
                                                              unsigned* __restrict__ ctl, size_t nCtl,
                                                              unsigned* __restrict__ slots, size_t nSlots) {
    const size_t t = size_t(psr_bid) * kThreads + threadIdx.x, stride = size_t(psr_nbid) * kThreads;
    for (size_t i = t; i < nZero; i += stride) zero[i] = 0u;
    // the CG's group controls and slots, used: zero again for the next solve
    for (size_t i = t; i < nCtl; i += stride) ctl[i] = 0u;
    for (size_t i = t; i < nSlots; i += stride) slots[i] = 0u;
    const bool cols = *q1Fired != 0;
    if (nDense && !cols) {
        float4* dense4 = reinterpret_cast<float4*>(dense);
        for (size_t i = t; i < nDense / 4; i += stride) dense4[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (t < nDense % 4) dense[nDense - 1 - t] = 0.f;
    }
    const size_t n = size_t(27) * M;
    if (cols) {
        // 16 bytes an entry: a workgroup's entries side by side, an entry a thread at a time
#pragma unroll
        for (int k = 0; k < kColumnItems; ++k) {
            const size_t e = (size_t(psr_bid) * kColumnItems + k) * kThreads + threadIdx.x;
            if (e >= n) break;
            const int nb = neigh[e];
            float4 col = make_float4(0.f, 0.f, 0.f, 0.f);
            if (nb >= 0) {
                const float4 b = basis[nb];
                col = make_float4(b.x, b.y, b.z, dx[nb]);
            }
            nbrCol[e] = col;
            dCol[e] = col.w;
        }
        return;
    }
    // four entries a thread (the columns are one array, 16-byte aligned)
    const size_t e = kColumnItems * t;
    if (e >= n) return;
    static_assert(kColumnItems == 4, "a 16-byte load and store");
    int nb[kColumnItems];
    if (e + kColumnItems <= n) {
        const int4 v = *reinterpret_cast<const int4*>(neigh + e);
        nb[0] = v.x, nb[1] = v.y, nb[2] = v.z, nb[3] = v.w;
    } else {
        for (int k = 0; k < kColumnItems; ++k) nb[k] = e + k < n ? neigh[e + k] : -1;
    }
    float d[kColumnItems];
#pragma unroll
    for (int k = 0; k < kColumnItems; ++k) d[k] = nb[k] < 0 ? 0.f : dx[nb[k]];
    if (e + kColumnItems <= n) *reinterpret_cast<float4*>(dCol + e) = make_float4(d[0], d[1], d[2], d[3]);
    else
        for (int k = 0; e + k < n; ++k) dCol[e + k] = d[k];
}
__global__ void __launch_bounds__(kThreads) neighbour_columns(int M, const int* __restrict__ neigh,
                                                              const float4* __restrict__ basis,
                                                              const float* __restrict__ dx,
                                                              float4* __restrict__ nbrCol, float* __restrict__ dCol,
                                                              unsigned* __restrict__ zero, size_t nZero,
                                                              float* __restrict__ dense, size_t nDense,
                                                              const int* __restrict__ q1Fired,
                                                              unsigned* __restrict__ ctl, size_t nCtl,
                                                              unsigned* __restrict__ slots, size_t nSlots) {
    neighbour_columns_body(blockIdx.x, gridDim.x, M, neigh, basis, dx, nbrCol, dCol, zero, nZero, dense, nDense, q1Fired, ctl, nCtl, slots, nSlots);
}
PSR_BATCHABLE(neighbour_columns, kThreads)



// stored (non-dropped) operator entries per depth
__device__ __forceinline__ void zero_u32_body(int psr_bid, int psr_nbid, unsigned* a, int n) {
    int i = psr_bid * blockDim.x + threadIdx.x;
    if (i < n) a[i] = 0u;
}
__global__ void __launch_bounds__(256) zero_u32(unsigned* a, int n) {
    zero_u32_body(blockIdx.x, gridDim.x, a, n);
}
PSR_BATCHABLE(zero_u32, 256)


}  // namespace

std::mutex& cg_order_lock() {
    static std::mutex m;
    return m;
}

// Resident-workgroup accounting of the CG launches in flight on the device
// (one GPU per process; guarded by cg_order_lock): a launch holds its share of
// the device's resident workgroups, in units of kCgUnits for the whole device,
// until its completion event (its context's CG end event) has fired.
struct CgInflight {
    hipEvent_t done;
    long long units;
};
constexpr long long kCgUnits = 1ll << 20;
std::vector<CgInflight>& cg_inflight() {
    static std::vector<CgInflight> v;
    return v;
}

int cg_batch_budget(Ctx& c) {
    const void* fn = c.cfg.precision == PSR_PRECISION_MIXED
                         ? multi_queue_kernel_of<cg_mixed_all_depths_k>(cg_mixed_all_depths)
                         : multi_queue_kernel_of<cg_all_depths_k>(cg_all_depths);
    int per = 0, cus = 0;
    PSR_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, fn, kCgThreads, 0));
    PSR_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c.device));
    return std::max(1, per * cus);
}

void cg_admit_device(hipEvent_t self) {
    std::unique_lock<std::mutex> order(cg_order_lock());
    for (;;) {
        auto& v = cg_inflight();
        v.erase(std::remove_if(v.begin(), v.end(),
                               [&](const CgInflight& f) { return f.done == self || hipEventQuery(f.done) == hipSuccess; }),
                v.end());
        if (v.empty()) return;
        order.unlock();
        std::this_thread::sleep_for(std::chrono::microseconds(20));
        order.lock();
    }
}

void cg_hold_device(hipEvent_t done) {
    std::lock_guard<std::mutex> order(cg_order_lock());
    cg_inflight().push_back(CgInflight{done, kCgUnits});
}

void cg_forget_event(hipEvent_t e) {
    std::lock_guard<std::mutex> order(cg_order_lock());
    auto& v = cg_inflight();
    v.erase(std::remove_if(v.begin(), v.end(), [&](const CgInflight& f) { return f.done == e; }), v.end());
}

void solve_depths(Ctx& c) {
    Octree& o = c.oct;
    const Levels& L = o.L;
    const int D = L.D, M = o.M;
    hipStream_t s = c.stream;
    float* val = c.buf<float>("lap_val", size_t(27) * M);
    DevResults* res = c.results();
    int* nnz = res->cgNnz;
    c.fld.dx = c.buf<float>("dx", M);
    if (size_t(M) * 2 * sizeof(float4) > size_t(INT32_MAX)) throw std::runtime_error("CG state exceeds 2 GiB");
    CgParams P{};
    P.M = M;
    P.tolSq = c.cfg.cg_tol * c.cfg.cg_tol;
    P.maxIter = c.cfg.cg_max_iter;
    P.spinLimit = 1u << 26;  // row form: polls of about a microsecond each, set below
    const bool mixed = c.cfg.precision == PSR_PRECISION_MIXED;
    const void* rowKernel = mixed ? reinterpret_cast<const void*>(cg_mixed_row) : reinterpret_cast<const void*>(cg_fp32_row);
    const void* genKernel =
        mixed ? reinterpret_cast<const void*>(cg_mixed_all_depths) : reinterpret_cast<const void*>(cg_all_depths);
    // workgroup budgets: every workgroup of a CG launch must be resident at once
    // (the groups meet in barriers).  The launch is an ordinary one: the budget,
    // with the accounting of concurrent launches below, is the residency
    // guarantee, and the barriers' spin bound turns a broken one into an error.
    // A batch merges the clouds' launches into the kernels' batched forms,
    // which the compiler may give other register counts: a budget is the
    // smaller occupancy of the two forms, so that a plan made for one cloud
    // also fits the merged launch.
    auto occupancy = [](const void* single, const void* batched, int threads) {
        int a = 0, b = 0;
        PSR_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&a, single, threads, 0));
        PSR_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, batched, threads, 0));
        return std::min(a, b);
    };
    if (c.cgMaxWgs <= 0) {
        const void* rowQueue = mixed ? multi_queue_kernel_of<cg_mixed_row_k>(cg_mixed_row)
                                     : multi_queue_kernel_of<cg_fp32_row_k>(cg_fp32_row);
        const void* genQueue = mixed ? multi_queue_kernel_of<cg_mixed_all_depths_k>(cg_mixed_all_depths)
                                     : multi_queue_kernel_of<cg_all_depths_k>(cg_all_depths);
        const int perRow = occupancy(rowKernel, rowQueue, kRowThreads), perGen = occupancy(genKernel, genQueue, kCgThreads);
        PSR_HIP_CHECK(hipDeviceGetAttribute(&c.cus, hipDeviceAttributeMultiprocessorCount, c.device));
        c.cgMaxWgsRow = std::max(0, perRow * c.cus);
        c.cgMaxWgs = std::max(1, perGen * c.cus);
    }
    // the mixed form solves indefinite depths with MINRES, in a launch of its
    // own (the MINRES kernel) after the CG launch of the other depths
    bool isMinres[PSR_MAX_DEPTH + 1];
    bool anyIndef = false;
    for (int d = 0; d <= D; ++d) anyIndef |= (isMinres[d] = mixed && c.indefinite[d]);
    if (anyIndef && c.cgMaxWgsMinres <= 0) {
        c.cgMaxWgsMinres = std::max(1, c.cus * occupancy(reinterpret_cast<const void*>(cg_mixed_minres),
                                                         multi_queue_kernel_of<cg_mixed_minres_k>(cg_mixed_minres), kCgThreads));
        c.cgMaxWgsChip[0] = c.cus * occupancy(reinterpret_cast<const void*>(cg_minres_chip4),
                                              multi_queue_kernel_of<cg_minres_chip4_k>(cg_minres_chip4), kCgThreads);
        c.cgMaxWgsChip[1] = c.cus * occupancy(reinterpret_cast<const void*>(cg_minres_chip8),
                                              multi_queue_kernel_of<cg_minres_chip8_k>(cg_minres_chip8), kCgThreads);
        c.cgMaxWgsChip[2] = c.cus * occupancy(reinterpret_cast<const void*>(cg_minres_chip16),
                                              multi_queue_kernel_of<cg_minres_chip16_k>(cg_minres_chip16), kCgThreads);
    }
    auto need_of = [&](int rpw, bool minresSet) {
        long long w = 0;
        for (int d = 0; d <= D; ++d)
            if (isMinres[d] == minresSet) w += std::max<long long>(1, (L.count[d] + rpw - 1) / rpw);
        return w;
    };
    auto need = [&](int rpw) { return need_of(rpw, false) + need_of(rpw, true); };
    // One row per thread, kRowThreads rows a workgroup, when all workgroups are
    // resident (about 390k rows) and every group's blocks fit the fold;
    // otherwise several rows per thread, the row blocks widened until they fit.
    int rowsPerWg = c.cgRowsPerWg > 0 ? c.cgRowsPerWg : kRowThreads;
    auto blocks_of = [&](int rows, int rpw) { return int(div_up(unsigned(rows), unsigned(rpw))) * (rpw > kRowBlock ? 2 : 1); };
    // (the override of the rows per workgroup reaches the several-rows form beyond 256)
    bool rowForm = (c.cgRowsPerWg == 0 || c.cgRowsPerWg <= kRowBlock) && need(rowsPerWg) <= c.cgMaxWgsRow;
    for (int d = 0; d <= D; ++d)
        if (blocks_of(L.count[d], rowsPerWg) > kRowMaxBlocks) rowForm = false;
    // MINRES runs in the several-rows-per-thread form only
    if (anyIndef) rowForm = false;
    if (!rowForm && c.cgRowsPerWg == 0) rowsPerWg = kCgThreads;
    int rowsPerWgMinres = rowsPerWg;
    if (!rowForm) {
        while (need_of(rowsPerWg, false) > c.cgMaxWgs) rowsPerWg *= 2;
        while (need_of(rowsPerWgMinres, true) > c.cgMaxWgsMinres) rowsPerWgMinres *= 2;
    }
    // A batch sets the rows a workgroup takes instead (cgRowTarget, from the
    // batch's total rows and the resident budget): a depth of n rows gets
    // ceil(n / target) workgroups of equal shares; one row per thread when
    // every share fits the workgroup's threads.  The target is the whole batch's,
    // in several waves of the budget: a cloud whose own workgroups would not all
    // be resident doubles it until they are.
    int capRows[PSR_MAX_DEPTH + 1];
    for (long long target = c.cgRowTarget; target > 0; target *= 2) {
        rowForm = !anyIndef;
        long long w[2] = {0, 0};  // workgroups of the CG and of the MINRES launch
        for (int d = 0; d <= D; ++d) {
            const int n = std::max(1, int(div_up(L.count[d], unsigned(target))));
            capRows[d] = std::max(1, int(div_up(L.count[d], unsigned(n))));
            if (capRows[d] > kRowThreads || blocks_of(L.count[d], capRows[d]) > kRowMaxBlocks) rowForm = false;
            w[isMinres[d] ? 1 : 0] += std::max(1, int(div_up(L.count[d], unsigned(capRows[d]))));
        }
        if (w[0] <= (rowForm ? c.cgMaxWgsRow : c.cgMaxWgs) && w[1] <= std::max(1, c.cgMaxWgsMinres)) break;
    }
    // largest depths first so their groups start on separate CUs early; the
    // MINRES depths form a second launch (PM) with its own workgroup numbering
    CgParams PM = P;
    int wg = 0, wgM = 0;
    for (int d = D; d >= 0; --d) {
        CgParams& Q = isMinres[d] ? PM : P;
        int& w = isMinres[d] ? wgM : wg;
        CgGroup& g = Q.g[Q.ngroups++];
        g.depth = d;
        g.rowBegin = L.base[d];
        g.rows = L.count[d];
        g.firstWg = w;
        g.rowsPerWg = c.cgRowTarget > 0 ? capRows[d] : (isMinres[d] ? rowsPerWgMinres : rowsPerWg);
        g.wgs = std::max(1, int(div_up(g.rows, g.rowsPerWg)));
        g.indef = isMinres[d] ? 1 : 0;
        w += g.wgs;
    }
    // The MINRES launch keeps its vectors on chip when its row blocks fit the
    // rows a thread holds and all its workgroups are resident in that form: up
    // to 3.1M rows here.  The row blocks, and so the sums, are the same either
    // way.
    int chip = -1;
    if (PM.ngroups > 0) {
        int widest = 0;
        for (int k = 0; k < PM.ngroups; ++k) widest = std::max(widest, PM.g[k].rowsPerWg);
        const int want = widest <= 4 * kCgThreads ? 0 : (widest <= 8 * kCgThreads ? 1 : 2);
        if (!c.minresInMemory && widest <= 16 * kCgThreads && wgM <= c.cgMaxWgsChip[want] && wgM <= kFoldParts * kCgThreads)
            chip = want;
    }
    const int capMinres = chip >= 0 ? c.cgMaxWgsChip[chip] : std::max(1, c.cgMaxWgsMinres);
    if (wg > (rowForm ? c.cgMaxWgsRow : c.cgMaxWgs) || wgM > capMinres)
        throw std::runtime_error("CG launch exceeds the resident workgroup budget");
    c.stats.cg_workgroups = uint32_t(wg + wgM);
    double* partial = rowForm ? nullptr : c.buf<double>("cg_partial", size_t(2) * (wg + wgM));
    GroupCtl* ctl = c.buf<GroupCtl>("cg_ctl", PSR_MAX_DEPTH + 1);
    const int ctlWords = int(sizeof(GroupCtl) / 4) * (PSR_MAX_DEPTH + 1);
    int* iters = res->cgIters;  // [inner iterations | outer steps] per depth
    double* resid = res->cgResid;
    double* trueRel = res->cgTrueRel;
    int* err = &res->cgErr;
    // slots of the row form's groups, or of the on-chip MINRES's
    const size_t slotCount = rowForm ? size_t(2) * kRowBlocks * kSlotStride * wg
                                     : (chip >= 0 ? size_t(4) * wgM + PM.ngroups * minres_result_slots() : 0);
    float4* slots = slotCount ? c.buf<float4>("cg_slots", slotCount) : nullptr;
    // The group controls and slots start at zero: the neighbour-column kernel
    // clears them after every solve, so they need a launch of their own only
    // when the last call on this context did not complete or the slots moved.
    // The CG writes every depth's results itself; its error flag is cleared
    // with the operator counts (by the vector-field kernel).
    const size_t slotWords = 4 * slotCount;
    if (!c.cgClean || slots != c.cgSlots || slotWords != c.cgSlotWords)
        zero_spans({{ctl, size_t(ctlWords)}, {slots, slotWords}}, s);
    c.cgClean = false;
    c.cgCtl = ctl;
    c.cgCtlWords = size_t(ctlWords);
    c.cgSlots = slots;
    c.cgSlotWords = slotWords;
    RowMapArgs maps{o.neigh, val, c.tables.weights, o.q1Fired, nullptr, nullptr, nullptr};
    char* rowState = nullptr;  // of the row form: the rows' records
    float* rowOut = nullptr;   // and the mixed form's outer residual
    if (rowForm) {
        BlockParts parts;
        const size_t oPlaces = parts.add(sizeof(unsigned) * 13 * M), oGhosts = parts.add(sizeof(int) * kGhostMax * wg),
                     oHeads = parts.add(sizeof(RowHead) * wg),
                     oState = parts.add((mixed ? sizeof(float4) : sizeof(float2)) * 2 * M), oOut = parts.add(sizeof(float) * M);
        char* block = c.buf<char>("cg_rows", parts.bytes);
        maps.places = reinterpret_cast<unsigned*>(block + oPlaces);
        maps.ghosts = reinterpret_cast<int*>(block + oGhosts);
        maps.heads = reinterpret_cast<RowHead*>(block + oHeads);
        rowState = block + oState;
        rowOut = reinterpret_cast<float*>(block + oOut);
    }
    const CoarsePlan& coarse = c.fld.foldArgs.plan;
    const int mapBlocks = rowForm ? wg : 0;
    PSR_LAUNCH(solve_prepare, mapBlocks + int(div_up(coarse.base[coarse.depths], kRowThreads)), 0, s, P, maps, mapBlocks,
               c.fld.foldArgs);
    // CG kernels of different contexts (streams) never compete for residency
    // while spinning in their group barriers: a launch is queued only once the
    // launches still in flight leave room for all its workgroups beside them
    // (the host waits otherwise), so concurrent contexts -- the batch workers --
    // run their solves side by side whenever they fit.
    // the two launches of a split solve run one after the other on the stream:
    // the account holds the larger
    const long long cap = rowForm ? c.cgMaxWgsRow : c.cgMaxWgs;
    const long long units = std::max((wg * kCgUnits + cap - 1) / cap, (wgM * kCgUnits + capMinres - 1) / capMinres);
    // While a batch records, the batch merges every cloud's solve into launches
    // that fit the resident budget and accounts for them itself.
    const bool recording = current_recorder() != nullptr;
    if (!recording) {
        std::unique_lock<std::mutex> order(cg_order_lock());
        for (;;) {
            auto& v = cg_inflight();
            // this context's earlier launch is ahead of this one in its stream
            v.erase(std::remove_if(v.begin(), v.end(),
                                   [&](const CgInflight& f) {
                                       return f.done == c.ev[9] || hipEventQuery(f.done) == hipSuccess;
                                   }),
                    v.end());
            long long used = 0;
            for (const CgInflight& f : v) used += f.units;
            if (used + units <= kCgUnits) break;
            order.unlock();
            std::this_thread::sleep_for(std::chrono::microseconds(20));
            order.lock();
        }
        PSR_HIP_CHECK(hipEventRecord(c.ev[8], s));
    }
    if (rowForm) P.spinLimit = 1u << 22;
    if (chip >= 0) PM.spinLimit = 1u << 24;  // polls of about a microsecond; a batch's group may wait for the solves before it
    if (c.cgSpinLimit >= 0) P.spinLimit = PM.spinLimit = unsigned(c.cgSpinLimit);
    static const char siteMixedRow = 0, siteMixedGen = 0, siteMinres = 0, siteRow = 0, siteGen = 0;
    static const char siteChip[3] = {0, 0, 0};
    if (mixed) {
        P.relTol = PM.relTol = c.cfg.refine_rel_tol;
        P.maxOuter = PM.maxOuter = std::max(1, c.cfg.refine_max_outer);
        if (rowForm) {
            launch_kernel<cg_mixed_row_k>(&siteMixedRow, cg_mixed_row, wg, 0, s, true, P, maps, c.fld.div, c.fld.dx,
                                          rowOut, reinterpret_cast<float4*>(rowState), slots, iters, resid, trueRel, err);
        } else {
            float* rOut = c.buf<float>("cg_rout", M);
            Comp2* partialC = c.buf<Comp2>("cg_partial_c", size_t(2) * (wg + wgM));
            // also the on-chip MINRES's two buffers of records
            float* rbuf = c.buf<float>("cg_rbuf", size_t(chip >= 0 ? 4 : 2) * M);
            float* wbuf = c.buf<float>("cg_wbuf", size_t(2) * M);
            float* sbuf = c.buf<float>("cg_sbuf", size_t(2) * M);
            float* pvec = c.buf<float>("cg_pa", M);
            if (P.ngroups > 0)
                launch_kernel<cg_mixed_all_depths_k>(&siteMixedGen, cg_mixed_all_depths, wg, 0, s, true, P, o.neigh,
                                                     val, c.fld.div, c.fld.dx, rOut, rbuf, wbuf, sbuf, pvec, partial,
                                                     partialC, ctl, iters, resid, trueRel, err, res->cgSlotMask);
            // the MINRES launch uses the group controls and partials after the CG launch's
            auto launch_chip = [&](auto k, auto kernel, const char* site) {
                launch_kernel<decltype(k)>(site, kernel, wgM, 0, s, true, PM, o.neigh, val, c.fld.div, c.fld.dx, rOut,
                                           reinterpret_cast<float2*>(rbuf), sbuf, partial + size_t(2) * wg, slots,
                                           ctl + P.ngroups, iters, resid, trueRel, err, res->cgSlotMask, o.q1Fired);
            };
            if (chip == 0) launch_chip(cg_minres_chip4_k{}, cg_minres_chip4, &siteChip[0]);
            else if (chip == 1) launch_chip(cg_minres_chip8_k{}, cg_minres_chip8, &siteChip[1]);
            else if (chip == 2) launch_chip(cg_minres_chip16_k{}, cg_minres_chip16, &siteChip[2]);
            else if (PM.ngroups > 0)
                launch_kernel<cg_mixed_minres_k>(&siteMinres, cg_mixed_minres, wgM, 0, s, true, PM, o.neigh, val,
                                                 c.fld.div, c.fld.dx, rOut, rbuf, wbuf, sbuf, pvec,
                                                 partial + size_t(2) * wg, partialC + size_t(2) * wg,
                                                 ctl + P.ngroups, iters, resid, trueRel, err, res->cgSlotMask);
        }
    } else if (rowForm) {
        launch_kernel<cg_fp32_row_k>(&siteRow, cg_fp32_row, wg, 0, s, true, P, maps, c.fld.div, c.fld.dx,
                                     reinterpret_cast<float2*>(rowState), slots, iters, resid, err);
    } else {
        float* r = c.buf<float>("cg_r", M);
        float* pA = c.buf<float>("cg_pa", M);
        float* pB = c.buf<float>("cg_pb", M);
        float* Ap = c.buf<float>("cg_ap", M);
        launch_kernel<cg_all_depths_k>(&siteGen, cg_all_depths, wg, 0, s, true, P, o.neigh, val, c.fld.div, c.fld.dx, r,
                                       pA, pB, Ap, partial, ctl, iters, resid, err, res->cgSlotMask);
    }
    c.stats.cg_row_form = rowForm ? 1 : 0;
    for (int d = 0; d <= D; ++d) c.cgForm[d] = isMinres[d] ? (chip >= 0 ? 4 << chip : -1) : (rowForm ? 1 : 0);
    if (!recording) {
        PSR_HIP_CHECK(hipEventRecord(c.ev[9], s));
        std::lock_guard<std::mutex> order(cg_order_lock());
        cg_inflight().push_back(CgInflight{c.ev[9], units});
    }
    PSR_HIP_CHECK(hipGetLastError());
}

void points_implicit(Ctx& c) {
    Octree& o = c.oct;
    const Levels& L = o.L;
    hipStream_t s = c.stream;
    int N = o.N, nb = int(div_up(N, kPointsChiThreads));
    c.fld.chiPts = c.buf<float>("chi_points", N);
    double* part = c.buf<double>("iso_part", nb);
    c.fld.isoSum = c.buf<double>("iso_sum", 1);
    c.fld.nbrCol = c.buf<float4>("nbr_col", size_t(27) * o.M);
    c.fld.dCol = c.buf<float>("nbr_dcol", size_t(27) * o.M);
    // the mesh stage's node tables and face marks, cleared with the columns:
    // nodeVert [8][M], nodeFace [6][M], nodeEdge [12][n_D], face marks (6M, the face bound)
    const size_t M = size_t(o.M), nD = size_t(L.count[L.D]), nZero = 8 * M + 6 * M + 12 * nD + 6 * M;
    int* zeroed = c.buf<int>("mesh_zeroed", nZero);
    c.geo.nodeVert = zeroed;
    c.geo.nodeFace = zeroed + 8 * M;
    c.geo.nodeEdge = zeroed + 14 * M;
    c.geo.faceMarks = zeroed + 14 * M + 12 * nD;
    // dense d_x grids for the subdivision of a regular octree (filled by the
    // mesh stage's first kernel)
    const size_t nDense = L.D <= kDenseEarlyDepth ? dense_grid_cells(L.D) : 0;
    c.geo.dxGrid = nDense ? c.buf<float>("sub_dx_grid", nDense) : nullptr;
    PSR_LAUNCH(neighbour_columns, div_up(size_t(27) * o.M, kColumnItems * kThreads), 0, s,
        o.M, o.neigh, o.basis, c.fld.dx, c.fld.nbrCol, c.fld.dCol, reinterpret_cast<unsigned*>(zeroed), nZero, c.geo.dxGrid,
        nDense, o.q1Fired, reinterpret_cast<unsigned*>(c.cgCtl), c.cgCtlWords,
        reinterpret_cast<unsigned*>(c.cgSlots), c.cgSlotWords);
    // the implicit function at the points runs beside the mesh stage's first
    // kernel (build_geometry), then the iso value
    c.fld.chiArgs = PointsChiArgs{N,        L.base[L.D], o.M,          L.D,      o.spos,        o.point2node,
                                  o.parent, c.fld.nbrCol, c.fld.dCol, o.basis, o.q1Fired, c.fld.chiPts, part};
    c.fld.chiBlocks = nb;
    PSR_HIP_CHECK(hipGetLastError());
}

}  // namespace psr
