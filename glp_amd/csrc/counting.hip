// Approximate and bounded-memory counting methods, and SLPA post-processing.
//
//   count-min  (method/countmin.cuh:10-263, used as a filter by
//               l_big_update_syn3, header/kernel.cuh:1420-1566): per vertex a
//               d x W sketch in LDS; every edge adds its frequency to one cell
//               per row; a label's estimate is the minimum of its cells after
//               all edges are in; the winner is the packed maximum of
//               (estimate, label).  Integer sums commute, so the result does
//               not depend on the order edges are added.  cm_aliased=1 keeps
//               the rows exactly as countmin.cuh writes them (d=3 adds row 3's
//               hash into row 2, :185-191; d=4 adds h3 into row 2 twice,
//               :197-221); cm_aliased=0 uses d independent rows.
//   frequent   (method/frequent.cuh SharedFA, a Misra-Gries table of C
//               slots): each vertex's edges are taken in CSR order; a present
//               label gains its frequency, an absent one takes a free slot,
//               and with no free slot every counter drops by
//               min(frequency, smallest counter), emptied slots are freed
//               and the label enters with what is left (the unit-step
//               Misra-Gries rule applied frequency times).
//   buffer     (method/buffer.cuh Buffer): as frequent, except that with no
//               free slot every counter drops by min(counter, frequency),
//               emptied slots are freed and the incoming label is dropped
//               (buffer.cuh:161-172).
// For frequent and buffer the table is processed sequentially per vertex,
// the order-dependent semantics the reference's concurrent tables only
// approximate.  The winner is the largest (count, label) left in the table;
// a vertex whose table ends empty keeps its label.
//
// Degree tiers.  Count-min: 16 lanes per vertex up to kCountminSmallDeg
// edges, with no sketch (each edge's estimate is summed over the vertex's
// edges whose cells coincide with its own, which is what the sketch cell
// would hold); one wavefront per vertex up to kCountminWaveMaxDeg edges and
// one 1024-thread workgroup per vertex up to kCountminHubDeg, with the sketch
// in LDS; above that, chunks of kCountminChunk edges on workgroups of their
// own (one pass adds each chunk's LDS sketch into the vertex's sketch in HBM,
// a second estimates every edge's label against the whole sketch and keeps
// the packed maximum with a 64-bit atomic max, a third commits).  Frequent and buffer: one lane per
// vertex up to kTableLaneMaxDeg edges (the lane walks its table slot by
// slot), one wavefront per vertex above, with table slot i held by lane i
// and the edges applied in CSR order, the order the semantics fix, several at
// once where that gives the same table, so both forms agree.  The vertices
// above the thresholds are listed once per session.

#include "device.h"
#include "device_prims.h"
#include "session.h"

#include <algorithm>
#include <memory>

namespace glp {
using namespace dev;

// Row hashes of method/countmin.cuh:97-142 (the constants must match for
// count-min results to match).
__device__ __forceinline__ uint32_t cm_hash(int r, uint32_t k) {
    switch (r) {
        case 0:
            k ^= k >> 16; k *= 0x12ebcb3bu; k ^= k >> 13; k *= 0xc123ae53u; k ^= k >> 16;
            return k;
        case 1:
            k ^= k >> 16; k *= 0x21eb21bbu; k ^= k >> 13; k *= 0x2cb2ea35u; k ^= k >> 16;
            return k;
        case 2:
            k ^= k >> 16; k *= 0x8febce61u; k ^= k >> 13; k *= 0xa2b2be25u; k ^= k >> 16;
            return k;
        case 3:
            k ^= k >> 12; k *= 0x13ebdb3au; k ^= k >> 12; k *= 0xc123ae53u; k ^= k >> 14;
            return k;
        default:
            k ^= k >> 13; k *= 0x312b521bu; k ^= k >> 5; k *= 0x1cb3ea22u; k ^= k >> 17;
            return k;
    }
}

// x mod W with m = floor(2^32 / W) (cm_mod_magic; W = 1: 2^32 - 1): the
// estimate floor(x m / 2^32) is the quotient or one less, so what is left
// after it is below 2 W.
__device__ __forceinline__ uint32_t cm_mod(uint32_t x, uint32_t m, uint32_t W) {
    const uint32_t r = x - __umulhi(x, m) * W;
    return min(r, r - W);  // r - W wraps above r when r < W
}
__host__ __device__ inline uint32_t cm_mod_magic(uint32_t W) { return W > 1u ? (uint32_t)((1ull << 32) / W) : ~0u; }

// The cells (row * W + column) a key touches, one entry per increment, R
// rows.  ALIASED (R = 3 or 4): row 3's hash lands in row 2, and for R = 4 h3
// goes into row 2 again.  The hashes and remainders (multiplications at a
// quarter rate) bound the count-min kernels, so the number of rows is a
// template parameter, the remainder takes two multiplications, and a
// thread's cells are kept from the sketch pass to the estimate pass.
template <int R, bool ALIASED>
__device__ __forceinline__ void cm_cells(uint32_t key, uint32_t W, uint32_t m, uint32_t* cell) {
    static_assert(!ALIASED || R == 3 || R == 4, "aliasing touches three or four rows");
#pragma unroll
    for (int r = 0; r < (ALIASED ? 3 : R); ++r) cell[r] = (uint32_t)r * W + cm_mod(cm_hash(r, key), m, W);
    if constexpr (ALIASED) cell[2] -= W;
    if constexpr (ALIASED && R == 4) cell[3] = cell[2];
}

// A key's cells, two to a word (rows * width <= 5 * 4096).
template <int R>
struct CmCells {
    uint32_t w[(R + 1) / 2];
    __device__ __forceinline__ void set(const uint32_t* c) {
#pragma unroll
        for (int i = 0; i < (R + 1) / 2; ++i) w[i] = c[2 * i] | (2 * i + 1 < R ? c[2 * i + 1] << 16 : 0u);
    }
    __device__ __forceinline__ uint32_t get(int r) const { return r & 1 ? w[r >> 1] >> 16 : w[r >> 1] & 0xffffu; }
};

constexpr int32_t kCountminSmallDeg = 16;
constexpr int kCmSmallClasses = 5;  // lane groups of 1, 2, 4, 8, 16 for degrees 1, 2, 3-4, 5-8, 9-16
static_assert(1 << (kCmSmallClasses - 1) == kCountminSmallDeg, "the last class reaches kCountminSmallDeg");
constexpr int32_t kCountminWaveMaxDeg = 1024;
constexpr int32_t kCountminMidDeg = 4096;  // up to here 256 threads per vertex, then 1024
constexpr int32_t kCountminHubDeg = 8192;
constexpr int32_t kCountminChunk = 8192;  // 1024 threads x 8 edges
constexpr int32_t kTableLaneMaxDeg = 32;

// The vertices of `verts` (degrees 1..G), G lanes each (lane i holds edge
// i; G = 1, 2, 4, 8 or 16, so 64 / G vertices share a wavefront).  The
// sketch cell an entry c of edge i lands in ends up holding the sum, over
// the vertex's edges j and their entries, of f_j where the entry is c; the
// estimate is the minimum of that over edge i's entries.
template <bool W, int G, int R, bool ALIASED>
__global__ __launch_bounds__(256) void k_countmin_small(StepArgs a, const int32_t* __restrict__ verts, int32_t nv,
                                                       uint32_t width, uint32_t m) {
    constexpr int kShift = G == 1 ? 0 : G == 2 ? 1 : G == 4 ? 2 : G == 8 ? 3 : 4;
    static_assert((1 << kShift) == G && G <= kCountminSmallDeg, "group of 1, 2, 4, 8 or 16 lanes");
    const int lane = lane_id(), ql = lane & (G - 1), g0 = lane & ~(G - 1);
    const int64_t vv = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> kShift;
    const bool in = vv < nv;
    const int32_t v = in ? verts[vv] : 0;
    int32_t b = 0, e = 0;
    if (in) {
        b = a.off[v];
        e = a.off[v + 1];
    }
    const bool live = in && ql < e - b;
    uint32_t key = 0u, f = 0u;  // a lane without an edge adds nothing (f = 0)
    if (live) {
        key = (uint32_t)a.L[a.nbr[b + ql]] + 1u;
        f = W ? a.w[b + ql] : 1u;
    }
    uint32_t c[R];
    cm_cells<R, ALIASED>(key, width, m, c);
    // Proper rows occupy disjoint bands [r W, (r+1) W), so entry t of one
    // edge can only meet entry t of another; aliased rows put entries 1..3
    // in one band, so those are compared crosswise.
    // edges of the wave's groups: the loop runs to the largest degree among them
    const int32_t dmax = __builtin_amdgcn_readfirstlane(
        (int32_t)wave_max_u64(live ? (uint64_t)(e - b) : 0ull));
    uint32_t sum[R] = {};
    for (int jj = 0; jj < dmax; ++jj) {
        const uint32_t fj = shfl_u32(f, g0 + jj);
        uint32_t cj[R];
#pragma unroll
        for (int t = 0; t < R; ++t) cj[t] = shfl_u32(c[t], g0 + jj);
#pragma unroll
        for (int t = 0; t < R; ++t) {
            if constexpr (!ALIASED) {
                sum[t] += cj[t] == c[t] ? fj : 0u;
            } else {
#pragma unroll
                for (int t2 = 0; t2 < R; ++t2) sum[t] += cj[t2] == c[t] ? fj : 0u;
            }
        }
    }
    uint32_t est = 0xffffffffu;
#pragma unroll
    for (int t = 0; t < R; ++t) est = min(est, sum[t]);
    uint64_t best = live ? pack_score((int32_t)min(est, 0x7fffffffu), key) : 0ull;
#pragma unroll
    for (int d = G / 2; d >= 1; d >>= 1) best = max_u64(best, shfl_u64(best, lane ^ d));
    bool changed = false;
    if (in && ql == 0) {
        const int32_t old = a.keep[v];
        const int32_t nl = best ? packed_label(best) : old;
        a.Lw[v] = nl;
        changed = nl != old;
    }
    const unsigned long long bal = __ballot(changed);
    if (lane == 0 && bal)
        atomicAdd(&a.changes[blockIdx.x & (kChangeSlots - 1)], (unsigned long long)__popcll(bal));
}

// Vertices without edges keep their label.
__global__ __launch_bounds__(256) void k_countmin_keep(StepArgs a, const int32_t* __restrict__ verts, int32_t nv) {
    const int32_t i = (int32_t)(blockIdx.x * 256 + threadIdx.x);
    if (i < nv) {
        const int32_t v = verts[i];
        a.Lw[v] = a.keep[v];
    }
}

// Up to kCmBatch edges of a thread (j, j + NT, ...) loaded at once: the
// indices past the last edge are clamped to it (every vertex here has edges)
// and their keys never applied, so the loads need no branches and all are in
// flight together.
constexpr int kCmBatch = 4;

template <bool W, int NT>
__device__ __forceinline__ void cm_load_batch(const StepArgs& a, int32_t j, int32_t last, uint32_t* key,
                                              uint32_t* f) {
    int32_t id[kCmBatch];
#pragma unroll
    for (int u = 0; u < kCmBatch; ++u) id[u] = a.nbr[min(j + u * NT, last)];
#pragma unroll
    for (int u = 0; u < kCmBatch; ++u) key[u] = (uint32_t)a.L[id[u]] + 1u;
#pragma unroll
    for (int u = 0; u < kCmBatch; ++u) f[u] = W ? a.w[min(j + u * NT, last)] : 1u;
}

// Vertex verts[blockIdx.x], the sketch in LDS (NT = 64: degrees up to
// kCountminWaveMaxDeg; NT = 256: up to kCountminMidDeg; NT = 1024: up to
// kCountminHubDeg).  A thread's keys (at most KB of them) and their cells stay
// in registers from the sketch pass to the estimate pass, so each neighbour
// label is read and hashed once.
template <bool W, int NT, int R, bool ALIASED>
__global__ __launch_bounds__(NT) void k_countmin(StepArgs a, const int32_t* __restrict__ verts, uint32_t width,
                                                 uint32_t m) {
    constexpr int KB =
        (NT == 64 ? kCountminWaveMaxDeg : NT == 256 ? kCountminMidDeg : kCountminHubDeg) / NT;
    static_assert(KB % kCmBatch == 0, "whole batches");
    extern __shared__ uint32_t cells[];
    __shared__ unsigned long long s_best[NT / 64];
    const int lane = lane_id();
    const int32_t v = verts[blockIdx.x];
    const int32_t b = a.off[v], e = a.off[v + 1];
    const int32_t last = e - 1;
    const int32_t ncell = R * (int32_t)width;
    for (int32_t i = threadIdx.x; i < ncell; i += NT) cells[i] = 0u;
    __syncthreads();
    uint32_t key[KB];
    CmCells<R> at[KB];
#pragma unroll
    for (int q = 0; q < KB; q += kCmBatch) {
        if (b + q * NT > last) break;  // uniform: no edges left for any thread
        const int32_t j = b + (int32_t)threadIdx.x + q * NT;
        uint32_t f[kCmBatch];
        cm_load_batch<W, NT>(a, j, last, key + q, f);
#pragma unroll
        for (int u = 0; u < kCmBatch; ++u) {
            if (j + u * NT > last) break;
            uint32_t c[R];
            cm_cells<R, ALIASED>(key[q + u], width, m, c);
            at[q + u].set(c);
#pragma unroll
            for (int i = 0; i < R; ++i) atomicAdd(&cells[c[i]], f[u]);
        }
    }
    __syncthreads();
    uint64_t best = 0ull;
#pragma unroll
    for (int q = 0; q < KB; q += kCmBatch) {
        if (b + q * NT > last) break;
        const int32_t j = b + (int32_t)threadIdx.x + q * NT;
#pragma unroll
        for (int u = 0; u < kCmBatch; ++u) {
            if (j + u * NT > last) break;
            uint32_t est = 0xffffffffu;
#pragma unroll
            for (int i = 0; i < R; ++i) est = min(est, cells[at[q + u].get(i)]);
            best = max_u64(best, pack_score((int32_t)min(est, 0x7fffffffu), key[q + u]));
        }
    }
    best = wave_max_u64(best);
    if (NT > 64) {
        if (lane == 0) s_best[threadIdx.x >> 6] = best;
        __syncthreads();
        best = lane < NT / 64 ? s_best[lane] : 0ull;
        best = wave_max_u64(best);
    }
    if (threadIdx.x == 0) {
        const int32_t old = a.keep[v];
        const int32_t nl = best ? packed_label(best) : old;
        a.Lw[v] = nl;
        if (nl != old) atomicAdd(&a.changes[blockIdx.x & (kChangeSlots - 1)], 1ull);
    }
}

// NV vertices of `verts` (degrees up to 64 EPL) per wavefront, one after
// another in one sketch: the loads of all of them are issued before any is
// counted, and a vertex's edges clear the cells they touched.  One vertex per
// wavefront spent its time in three dependent loads and in clearing the
// sketch (R-MAT scale 21, 3 x 200, degrees 17-1024: 210 us a step, now 192).
constexpr int kCmVerts = 4;
template <bool W, int EPL, int R, bool ALIASED>
__global__ __launch_bounds__(64) void k_countmin_few(StepArgs a, const int32_t* __restrict__ verts, int32_t nv,
                                                     uint32_t width, uint32_t m) {
    extern __shared__ uint32_t cells[];
    const int lane = lane_id();
    const int32_t i0 = (int32_t)blockIdx.x * kCmVerts;
    int32_t v[kCmVerts], b[kCmVerts], e[kCmVerts], old[kCmVerts];
#pragma unroll
    for (int k = 0; k < kCmVerts; ++k) v[k] = verts[min(i0 + k, nv - 1)];
#pragma unroll
    for (int k = 0; k < kCmVerts; ++k) {
        b[k] = a.off[v[k]];
        e[k] = a.off[v[k] + 1];
        old[k] = a.keep[v[k]];
    }
    const int32_t ncell = R * (int32_t)width;
    for (int32_t i = lane; i < ncell; i += 64) cells[i] = 0u;
    // (clamped to the last edge; every vertex here has edges)
    uint32_t key[kCmVerts][EPL], f[kCmVerts][EPL];
#pragma unroll
    for (int k = 0; k < kCmVerts; ++k)
#pragma unroll
        for (int i = 0; i < EPL; ++i) {
            const int32_t j = min(b[k] + lane + 64 * i, e[k] - 1);
            key[k][i] = (uint32_t)a.nbr[j];
            f[k][i] = W ? a.w[j] : 1u;
        }
#pragma unroll
    for (int k = 0; k < kCmVerts; ++k)
#pragma unroll
        for (int i = 0; i < EPL; ++i) key[k][i] = (uint32_t)a.L[key[k][i]] + 1u;
    uint32_t nch = 0u;
#pragma unroll
    for (int k = 0; k < kCmVerts; ++k) {
        if (i0 + k >= nv) break;  // wave-uniform
        CmCells<R> at[EPL];
        wave_lds_sync();  // the cells are clear
#pragma unroll
        for (int i = 0; i < EPL; ++i) {
            if (64 * i >= e[k] - b[k]) break;  // wave-uniform
            uint32_t c[R];
            cm_cells<R, ALIASED>(key[k][i], width, m, c);
            at[i].set(c);
            if (b[k] + lane + 64 * i < e[k]) {
#pragma unroll
                for (int r = 0; r < R; ++r) atomicAdd(&cells[c[r]], f[k][i]);
            }
        }
        wave_lds_sync();
        uint64_t best = 0ull;
#pragma unroll
        for (int i = 0; i < EPL; ++i) {
            if (64 * i >= e[k] - b[k]) break;
            uint32_t est = 0xffffffffu;
#pragma unroll
            for (int r = 0; r < R; ++r) est = min(est, cells[at[i].get(r)]);
            // (a lane past the last edge repeats that edge's estimate)
            best = max_u64(best, pack_score((int32_t)min(est, 0x7fffffffu), key[k][i]));
        }
        wave_lds_sync();
#pragma unroll
        for (int i = 0; i < EPL; ++i) {
            if (64 * i >= e[k] - b[k]) break;
#pragma unroll
            for (int r = 0; r < R; ++r) cells[at[i].get(r)] = 0u;
        }
        best = wave_max_u64(best);
        const int32_t nl = packed_label(best);
        if (lane == 0) a.Lw[v[k]] = nl;
        nch += nl != old[k] ? 1u : 0u;
    }
    if (lane == 0 && nch) atomicAdd(&a.changes[blockIdx.x & (kChangeSlots - 1)], (unsigned long long)nch);
}

// Count-min hubs (degree above kCountminHubDeg): workgroup i takes chunk
// chunks[i] = (hub slot h, first edge of the chunk within the hub's edges),
// kCountminChunk edges.  `sketch` holds rows * width cells per hub and
// `best` one packed maximum per hub; both are zero between steps
// (k_countmin_hub_final clears them).  Sums of cells wrap modulo 2^32 as the
// single-workgroup form's LDS sums do, so the estimates are the same.  The
// sketch pass leaves each edge's key in `keys` (kCountminChunk slots per
// chunk, in edge order), which the estimate pass reads back in order instead
// of gathering the labels again.
template <bool W, int R, bool ALIASED>
__global__ __launch_bounds__(1024) void k_countmin_hub_sketch(StepArgs a, const int32_t* __restrict__ hubs,
                                                              const int2* __restrict__ chunks,
                                                              uint32_t* __restrict__ sketch,
                                                              uint32_t* __restrict__ keys, uint32_t width, uint32_t m) {
    extern __shared__ uint32_t cells[];
    const int2 ch = chunks[blockIdx.x];
    const int32_t v = hubs[ch.x];
    const int32_t b = a.off[v] + ch.y, e = min(a.off[v + 1], b + kCountminChunk);
    const int32_t last = e - 1;
    const int32_t ncell = R * (int32_t)width;
    for (int32_t i = threadIdx.x; i < ncell; i += 1024) cells[i] = 0u;
    __syncthreads();
    uint32_t* ck = keys + (size_t)blockIdx.x * kCountminChunk;  // ck[j - b]: edge j's key
    for (int32_t j = b + (int32_t)threadIdx.x; j < e; j += 1024 * kCmBatch) {
        uint32_t key[kCmBatch], f[kCmBatch];
        cm_load_batch<W, 1024>(a, j, last, key, f);
#pragma unroll
        for (int u = 0; u < kCmBatch; ++u) {
            if (j + u * 1024 > last) break;
            ck[j - b + u * 1024] = key[u];
            uint32_t c[R];
            cm_cells<R, ALIASED>(key[u], width, m, c);
#pragma unroll
            for (int i = 0; i < R; ++i) atomicAdd(&cells[c[i]], f[u]);
        }
    }
    __syncthreads();
    uint32_t* hs = sketch + (size_t)ch.x * ncell;
    for (int32_t i = threadIdx.x; i < ncell; i += 1024) {
        const uint32_t c = cells[i];
        if (c) atomicAdd(&hs[i], c);
    }
}

template <int R, bool ALIASED>
__global__ __launch_bounds__(1024) void k_countmin_hub_est(StepArgs a, const int32_t* __restrict__ hubs,
                                                           const int2* __restrict__ chunks,
                                                           const uint32_t* __restrict__ sketch,
                                                           const uint32_t* __restrict__ keys,
                                                           unsigned long long* __restrict__ best_out, uint32_t width, uint32_t m) {
    extern __shared__ uint32_t cells[];
    __shared__ unsigned long long s_best[16];
    const int lane = lane_id();
    const int2 ch = chunks[blockIdx.x];
    const int32_t v = hubs[ch.x];
    const int32_t b = a.off[v] + ch.y, e = min(a.off[v + 1], b + kCountminChunk);
    const int32_t last = e - 1;
    const int32_t ncell = R * (int32_t)width;
    const uint32_t* hs = sketch + (size_t)ch.x * ncell;
    for (int32_t i = threadIdx.x; i < ncell; i += 1024) cells[i] = hs[i];
    __syncthreads();
    const uint32_t* ck = keys + (size_t)blockIdx.x * kCountminChunk;
    uint64_t best = 0ull;
    for (int32_t j = b + (int32_t)threadIdx.x; j < e; j += 1024 * kCmBatch) {
        uint32_t key[kCmBatch];
#pragma unroll
        for (int u = 0; u < kCmBatch; ++u) key[u] = ck[min(j + u * 1024, last) - b];
#pragma unroll
        for (int u = 0; u < kCmBatch; ++u) {
            if (j + u * 1024 > last) break;
            uint32_t c[R];
            cm_cells<R, ALIASED>(key[u], width, m, c);
            uint32_t est = 0xffffffffu;
#pragma unroll
            for (int i = 0; i < R; ++i) est = min(est, cells[c[i]]);
            best = max_u64(best, pack_score((int32_t)min(est, 0x7fffffffu), key[u]));
        }
    }
    best = wave_max_u64(best);
    if (lane == 0) s_best[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x < 64) {
        best = wave_max_u64(lane < 16 ? s_best[lane] : 0ull);
        if (lane == 0 && best) atomicMax(&best_out[ch.x], (unsigned long long)best);
    }
}

// One workgroup per count-min hub: commits its winner, then clears its
// sketch and maximum for the next step.
__global__ __launch_bounds__(256) void k_countmin_hub_final(StepArgs a, const int32_t* __restrict__ hubs,
                                                            uint32_t* __restrict__ sketch,
                                                            unsigned long long* __restrict__ best, int32_t ncell) {
    const int32_t h = (int32_t)blockIdx.x;
    uint32_t* hs = sketch + (size_t)h * ncell;
    for (int32_t i = threadIdx.x; i < ncell; i += 256) hs[i] = 0u;
    if (threadIdx.x == 0) {
        const int32_t v = hubs[h];
        const unsigned long long bb = best[h];
        const int32_t old = a.keep[v];
        const int32_t nl = bb ? packed_label(bb) : old;
        a.Lw[v] = nl;
        if (nl != old) atomicAdd(&a.changes[(uint32_t)h & (kChangeSlots - 1)], 1ull);
        best[h] = 0ull;
    }
}

// A wide table: slot i is lane i's (K, A).  A slot's count is A - off, so a
// drop of every slot is one scalar addition to `off`; `fr` holds the free
// slots (key 0).  Lanes >= cap hold the key 0xffffffff, which no edge carries
// (keys are labels + 1 <= 2^31), and the largest A: they never match, are
// never free and never the smallest.  A and off stay below 2^31 (the host
// checks the largest frequency sum).
struct WideTable {
    uint32_t K, A;
    uint32_t off;  // wave-uniform
    uint64_t fr;   // wave-uniform
};

// Applies a chunk's edges (lane l: key, frequency f; `all` the lanes with an
// edge) at once where that gives what applying them in order gives: no edge
// misses, or the table is full and its smallest count exceeds what all the
// misses together take off, so no slot can empty between them.  False (and
// nothing applied) otherwise.  `sum` is the wave's LDS.
template <bool W>
__device__ __forceinline__ bool table_bulk(uint32_t key, uint32_t f, uint64_t all, int32_t cap, WideTable& t,
                                           uint32_t* sum) {
    const int lane = lane_id();
    int32_t at = -1;  // the slot holding this edge's key
#pragma unroll 4
    for (int32_t s = 0; s < cap; ++s)
        at = key == (uint32_t)__builtin_amdgcn_readlane((int)t.K, s) ? s : at;
    const bool in = (all >> lane) & 1u;
    const uint64_t miss = __ballot(in && at < 0);
    uint32_t drop = 0u;
    if (miss) {
        if (t.fr) return false;
        drop = W ? wave_sum_u32(in && at < 0 ? f : 0u) : (uint32_t)__popcll(miss);
        drop = (uint32_t)__builtin_amdgcn_readfirstlane((int)drop);
        if (__ballot(t.A <= t.off + drop)) return false;
    }
    sum[lane] = 0u;
    wave_lds_sync();
    if (in && at >= 0) atomicAdd(&sum[at], W ? f : 1u);
    wave_lds_sync();
    t.A += sum[lane];
    t.off += drop;
    wave_lds_sync();
    return true;
}

// Lane src's 64-bit value, held as two words.
__device__ __forceinline__ uint64_t readlane_u64(uint32_t lo, uint32_t hi, int src) {
    return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)hi, src) << 32) |
           (uint32_t)__builtin_amdgcn_readlane((int)lo, src);
}

constexpr int kTableBlk = 4;               // most chunks of 64 edges loaded together
constexpr uint32_t kNoEdge = 0xfffffffeu;  // key of a lane past the last edge

// For each of a block's chunks (lane l: edge l's key) the edge lanes whose
// key may occur more than once in the chunk: every one that does, and the few
// that share a hash bit.  The block's chunks go through LDS together, so its
// latency is paid once.
constexpr uint32_t kDupWords = 128;
struct TableLds {
    uint32_t bits[kTableBlk][2][kDupWords];  // per chunk 4,096 bits: a key hashed here; another one did
};
template <int B>
__device__ __forceinline__ void table_repeats(const uint32_t* key, uint64_t* dup, TableLds& t) {
    const int lane = lane_id();
    uint32_t* flat = &t.bits[0][0][0];
#pragma unroll
    for (uint32_t i = 0; i < B * 2 * kDupWords; i += 64) flat[i + (uint32_t)lane] = 0u;
    wave_lds_sync();
    uint32_t w[B], bit[B], old[B];
#pragma unroll
    for (int u = 0; u < B; ++u) {
        const uint32_t h = (key[u] * 0x9e3779b1u) >> 20;
        static_assert(kDupWords * 32 == 1u << (32 - 20), "one bit per hash value");
        w[u] = h >> 5;
        // lanes past the last edge set no bit
        bit[u] = key[u] != kNoEdge ? 1u << (h & 31u) : 0u;
        old[u] = atomicOr(&t.bits[u][0][w[u]], bit[u]);
    }
#pragma unroll
    for (int u = 0; u < B; ++u) atomicOr(&t.bits[u][1][w[u]], old[u] & bit[u]);
    wave_lds_sync();
#pragma unroll
    for (int u = 0; u < B; ++u) old[u] = t.bits[u][1][w[u]];
#pragma unroll
    for (int u = 0; u < B; ++u) dup[u] = __ballot((old[u] & bit[u]) != 0u);
    wave_lds_sync();
}

// Applies an unweighted chunk (lane l: edge l's key; `all` the lanes with an
// edge, the others' key kNoEdge; `dup` the lanes whose key may repeat) as if
// its edges came one after another: a key in the table gains one, else it
// takes a free slot with one, else (full) every slot drops by one, emptied
// slots are freed and the key is dropped.  (Which free slot a key takes does
// not matter: the winner is a maximum over the table.  Every count is >= 1
// and every frequency 1, so frequent and buffer agree.)
// Between two changes of the key set hits only add up, so the chunk is
// applied event by event instead of edge by edge.  An entry is a table slot
// (lane i: K, A) or, entered in this chunk, its first edge's lane (key, An);
// mo and mn are the lane's masks of the chunk's later edges with its key, so
// an entry's count at edge p is A + (mask bits below p) - off.  `miss` holds
// the edges not yet applied whose key has no entry:
//  * with free slots the first misses enter, all at once while their keys
//    occur once in the chunk (`run`), else one at a time, its later edges
//    becoming hits;
//  * full, the next miss drops every entry (off + 1) and frees the emptied
//    ones, whose later edges miss again; if it empties none, no miss before
//    the cmin-th can (cmin the smallest count), so those are skipped;
//  * a run that fills the f free slots loses those entries again to its next
//    miss, f + 1 misses a turn, as long as no older entry empties: such turns
//    are skipped together.
// While labels are diverse a chunk takes about three events; one edge at a
// time it took 64 ballots, each followed by a dependent update.  The chain
// of events of the largest hub sets the step: latency bound, one wavefront.
__device__ __forceinline__ void table_chunk(uint32_t key, uint64_t all, uint64_t dup, int32_t cap, WideTable& t,
                                            uint32_t* lds) {
    const int lane = lane_id();
    uint32_t mo_lo = 0u, mo_hi = 0u, mn_lo = 0u, mn_hi = 0u, An = 0u;
    const uint64_t slots = cap == 64 ? ~0ull : (1ull << cap) - 1ull;
    uint64_t live_o = slots & ~t.fr, live_n = 0ull;
    const int top = live_o ? 64 - (int)__builtin_clzll(live_o) : 0;  // past the highest slot in use
    int at = -1;  // the slot holding this edge's key
    for (int s = 0; s < top; s += 4) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            // a free slot's key is 0, lanes without a slot hold 0xffffffff: no edge carries either
            at = key == (uint32_t)__builtin_amdgcn_readlane((int)t.K, s + u) ? s + u : at;
        }
    }
    const uint64_t hit = __ballot(at >= 0);
    if (hit) {
        lds[lane] = 0u;
        lds[64 + lane] = 0u;
        wave_lds_sync();
        if (at >= 0) atomicOr(&lds[at + (lane & 32 ? 64 : 0)], 1u << (lane & 31));
        wave_lds_sync();
        mo_lo = lds[lane];
        mo_hi = lds[64 + lane];
        wave_lds_sync();
    }
    uint64_t miss = all & ~hit;
    uint32_t off = t.off, nfree = (uint32_t)__popcll(t.fr);
    while (miss) {  // every pass applies at least the first miss
        if (nfree) {
            const uint64_t low = miss & (0ull - miss);
            if (dup & low) {
                const int p = (int)__builtin_ctzll(miss);
                const uint32_t kk = (uint32_t)__builtin_amdgcn_readlane((int)key, p);
                const uint64_t m = __ballot(key == kk) & (0ull - low);  // from p on
                const uint64_t later = m & ~low;
                const bool mine = lane == p;
                An = mine ? off + 1u : An;
                mn_lo = mine ? (uint32_t)later : mn_lo;
                mn_hi = mine ? (uint32_t)(later >> 32) : mn_hi;
                live_n |= low;
                miss &= ~m;
                --nfree;
            } else {
                // the misses before the first whose key may repeat
                const uint64_t d = miss & dup;
                uint64_t run = miss & ((d & (0ull - d)) - 1ull);  // d = 0: all of them
                uint32_t n = (uint32_t)__popcll(run);
                if (n > nfree) {
                    const uint32_t r = (uint32_t)lanes_below(run);
                    uint32_t skip = 0u;
                    if (live_n == 0ull) {
                        uint32_t turns = 0u, left = n;
                        for (; left > nfree; left -= nfree + 1u) ++turns;
                        if ((__ballot(t.A <= off + turns) & live_o) == 0ull) {
                            skip = n - left;
                            n = left;
                            off += turns;
                        }
                    }
                    const uint64_t gone = run & __ballot(r < skip);
                    run = run & ~gone & __ballot(r < skip + nfree);
                    miss &= ~gone;
                    n = min(n, nfree);
                }
                const bool mine = __builtin_amdgcn_inverse_ballot_w64(run);
                An = mine ? off + 1u : An;
                mn_lo = mine ? 0u : mn_lo;
                mn_hi = mine ? 0u : mn_hi;
                live_n |= run;
                miss &= ~run;
                nfree -= n;
            }
            if (nfree || miss == 0ull) continue;
        }
        const uint64_t low = miss & (0ull - miss), below = low - 1ull;
        const uint32_t b_lo = (uint32_t)below, b_hi = (uint32_t)(below >> 32);
        const uint32_t co = t.A + (uint32_t)(__popc(mo_lo & b_lo) + __popc(mo_hi & b_hi));
        const uint32_t cn = An + (uint32_t)(__popc(mn_lo & b_lo) + __popc(mn_hi & b_hi));
        const uint64_t dead_o = __ballot(co == off + 1u) & live_o;
        const uint64_t dead_n = __ballot(cn == off + 1u) & live_n;
        if ((dead_o | dead_n) == 0ull) {
            const uint32_t lo_o = __builtin_amdgcn_inverse_ballot_w64(live_o) ? co : 0xffffffffu;
            const uint32_t lo_n = __builtin_amdgcn_inverse_ballot_w64(live_n) ? cn : 0xffffffffu;
            const uint32_t cmin = wave_min_u32(min(lo_o, lo_n)) - off;  // >= 2
            const uint32_t skip = min(cmin - 1u, (uint32_t)__popcll(miss));
            for (uint32_t k = 0u; k < skip; ++k) miss &= miss - 1ull;
            off += skip;
            continue;
        }
        ++off;
        miss &= ~low;
        const uint64_t after = ~(below | low);  // the edges past this miss
        const uint32_t a_lo = (uint32_t)after, a_hi = (uint32_t)(after >> 32);
        const bool d_o = __builtin_amdgcn_inverse_ballot_w64(dead_o), d_n = __builtin_amdgcn_inverse_ballot_w64(dead_n);
        const uint32_t back_lo = ((d_o ? mo_lo : 0u) | (d_n ? mn_lo : 0u)) & a_lo;
        const uint32_t back_hi = ((d_o ? mo_hi : 0u) | (d_n ? mn_hi : 0u)) & a_hi;
        for (uint64_t q = __ballot((back_lo | back_hi) != 0u); q; q &= q - 1ull)
            miss |= readlane_u64(back_lo, back_hi, (int)__builtin_ctzll(q));
        live_o &= ~dead_o;
        live_n &= ~dead_n;
        nfree = (uint32_t)(__popcll(dead_o) + __popcll(dead_n));
    }
    t.off = off;
    t.A += (uint32_t)(__popc(mo_lo) + __popc(mo_hi));  // 0 for lanes without a slot
    t.fr = slots & ~live_o;
    if (__builtin_amdgcn_inverse_ballot_w64(t.fr)) t.K = 0u;
    if (live_n) {  // this chunk's entries move to free slots
        const uint32_t cnt = (uint32_t)__popcll(live_n);
        uint32_t* ks = lds;
        uint32_t* as = lds + 64;
        if (__builtin_amdgcn_inverse_ballot_w64(live_n)) {
            const uint32_t r = (uint32_t)lanes_below(live_n);
            ks[r] = key;
            as[r] = An + (uint32_t)(__popc(mn_lo) + __popc(mn_hi));
        }
        wave_lds_sync();
        const uint32_t r = (uint32_t)lanes_below(t.fr);
        const bool takes = __builtin_amdgcn_inverse_ballot_w64(t.fr) && r < cnt;
        if (takes) {
            t.K = ks[r];
            t.A = as[r];
        }
        t.fr &= ~__ballot(takes);
        wave_lds_sync();
    }
}

// Applies one weighted edge: a key in the table gains the frequency, else it
// takes the lowest free slot, else (full) every counter drops and emptied
// slots are freed.  Buffer drops by min(counter, frequency) and the key is
// dropped; frequent drops by d = min(frequency, smallest counter) and what is
// left of the frequency enters the first freed slot.
template <bool BUF>
__device__ __forceinline__ void table_edge(uint32_t kk, uint32_t ff, WideTable& t) {
    const uint64_t hm = __ballot(t.K == kk);
    if (hm) {
        t.A += __builtin_amdgcn_inverse_ballot_w64(hm) ? ff : 0u;
        return;
    }
    if (t.fr) {
        const uint64_t low = t.fr & (0ull - t.fr);
        const bool mine = __builtin_amdgcn_inverse_ballot_w64(low);
        t.K = mine ? kk : t.K;
        t.A = mine ? t.off + ff : t.A;
        t.fr ^= low;
        return;
    }
    const uint32_t to = t.off + ff;
    const uint64_t gone = __ballot(t.A <= to);
    if (gone == 0ull) {
        t.off = to;
        return;
    }
    if constexpr (BUF) {
        t.off = to;
        t.fr = gone;
        t.K = __builtin_amdgcn_inverse_ballot_w64(gone) ? 0u : t.K;
    } else {
        const uint32_t least = wave_min_u32(t.A);  // off + the smallest counter
        const uint32_t left = ff - (least - t.off);
        t.off = least;
        t.fr = __ballot(t.A == least);
        t.K = __builtin_amdgcn_inverse_ballot_w64(t.fr) ? 0u : t.K;
        if (left) {
            const uint64_t low = t.fr & (0ull - t.fr);
            const bool mine = __builtin_amdgcn_inverse_ballot_w64(low);
            t.K = mine ? kk : t.K;
            t.A = mine ? t.off + left : t.A;
            t.fr ^= low;
        }
    }
}

// Applies the edges [b, e) (e > b) of a vertex to its table.  Edges come in
// chunks of 64, one per lane, applied at once where table_bulk can, else by
// table_chunk (weighted: edge by edge); the bulk form is tried after it
// worked and on every fourth chunk, so that diverse labels, where it does
// not, pay little for it.  B chunks' loads are issued together, a block
// ahead (the neighbour ids two blocks ahead): a chunk applied at once takes
// less time than its loads.  Lanes past the last edge load the last edge
// again (in bounds, never applied), so the loads need no branches and stay in
// flight across the block.
template <bool W, bool BUF, int B>
__device__ __forceinline__ void table_run(const StepArgs& a, int32_t b, int32_t e, int32_t cap, WideTable& t,
                                          TableLds& lds) {
    const int lane = lane_id();
    uint32_t* words = &lds.bits[0][0][0];  // scratch of one chunk
    const int32_t last = e - 1;
    // this lane's edge of chunk u of the block at j (an int64 j: the blocks
    // loaded ahead may lie past 2^31)
    auto edge = [&](int64_t j, int u) { return (int32_t)min(j + 64 * u + lane, (int64_t)last); };
    bool calm = false;  // the last chunk was applied at once
    uint32_t chunk = 0u;
    int32_t id[B];
    uint32_t lab[B], f[B];
#pragma unroll
    for (int u = 0; u < B; ++u) id[u] = a.nbr[edge(b, u)];
#pragma unroll
    for (int u = 0; u < B; ++u) {
        lab[u] = (uint32_t)a.L[id[u]];
        f[u] = W ? a.w[edge(b, u)] : 1u;
    }
#pragma unroll
    for (int u = 0; u < B; ++u) id[u] = a.nbr[edge((int64_t)b + 64 * B, u)];
    for (int64_t j0 = b; j0 < e; j0 += 64 * B) {
        const int64_t j1 = j0 + 64 * B, j2 = j1 + 64 * B;
        uint32_t nlab[B], nf[B];
#pragma unroll
        for (int u = 0; u < B; ++u) {
            nlab[u] = (uint32_t)a.L[id[u]];
            nf[u] = W ? a.w[edge(j1, u)] : 1u;
        }
#pragma unroll
        for (int u = 0; u < B; ++u) id[u] = a.nbr[edge(j2, u)];
        uint32_t key[B];
        uint64_t dup[B] = {};
        bool have = false;  // dup is known
#pragma unroll
        for (int u = 0; u < B; ++u) key[u] = j0 + 64 * u + lane < e ? lab[u] + 1u : kNoEdge;
        // one chunk's code for all of them: the block's registers rotate
#pragma unroll 1
        for (int u = 0; u < B; ++u) {
            const int32_t cnt = (int32_t)min((int64_t)64, (int64_t)e - j0 - 64 * u);
            if (cnt <= 0) break;
            const uint64_t all = cnt == 64 ? ~0ull : (1ull << cnt) - 1ull;
            calm = (calm || chunk++ % 4u == 3u) && table_bulk<W>(key[0], f[0], all, cap, t, words);
            if (!calm) {
                if constexpr (W) {
                    auto apply = [&](int k) {
                        table_edge<BUF>((uint32_t)__builtin_amdgcn_readlane((int)key[0], k),
                                        (uint32_t)__builtin_amdgcn_readlane((int)f[0], k), t);
                    };
                    if (cnt == 64) {
#pragma unroll 64
                        for (int k = 0; k < 64; ++k) apply(k);
                    } else {
                        for (int k = 0; k < cnt; ++k) apply(k);
                    }
                } else {
                    if (!have) table_repeats<B>(key, dup, lds);
                    have = true;
                    table_chunk(key[0], all, dup[0], cap, t, words);
                }
            }
#pragma unroll
            for (int k = 0; k + 1 < B; ++k) {
                key[k] = key[k + 1];
                f[k] = f[k + 1];
                dup[k] = dup[k + 1];
            }
        }
#pragma unroll
        for (int u = 0; u < B; ++u) {
            lab[u] = nlab[u];
            f[u] = nf[u];
        }
    }
}

// One wavefront per vertex of `verts` (degrees above kTableLaneMaxDeg), its
// table a WideTable; the vertex and its edge range are wave-uniform (scalar
// loop control).  Up to kTableShort edges the loads of four chunks at a time
// would mostly be clamped ones (planted graph of 100,000 vertices of degree
// 48, 4 steps: 0.95 ms, with one chunk at a time 0.59).  The chain of edges
// of the largest hub sets the step, not bandwidth: R-MAT scale 21, 16 slots,
// 3 steps from L0, 20.4 ms with every edge applied on its own (64 ns an
// edge), 8.0 ms with table_chunk (22 ns); weighted at scale 20 (frequent)
// 23.9 -> 17.7 ms with the offset in place of a drop per slot and the chunk
// unrolled.
constexpr int32_t kTableShort = 256;
template <bool W, bool BUF>
__global__ __launch_bounds__(256) void k_table_wave(StepArgs a, const int32_t* __restrict__ verts, int32_t nv,
                                                    int32_t cap) {
    __shared__ TableLds s_lds[4];
    const int lane = lane_id();
    const int32_t i = (int32_t)(blockIdx.x * 4 + (threadIdx.x >> 6));
    if (i >= nv) return;  // wave-uniform
    const int32_t v = __builtin_amdgcn_readfirstlane(verts[i]);
    const int32_t b = __builtin_amdgcn_readfirstlane(a.off[v]);
    const int32_t e = __builtin_amdgcn_readfirstlane(a.off[v + 1]);
    const bool slot = lane < cap;
    WideTable t{slot ? 0u : 0xffffffffu, slot ? 0u : 0xffffffffu, 0u, __ballot(slot)};
    TableLds& lds = s_lds[threadIdx.x >> 6];
    if (e - b <= kTableShort) table_run<W, BUF, 1>(a, b, e, cap, t, lds);
    else table_run<W, BUF, kTableBlk>(a, b, e, cap, t, lds);
    const uint64_t best = wave_max_u64(slot && t.K ? pack_score((int32_t)(t.A - t.off), t.K) : 0ull);
    if (lane == 0) {
        const int32_t old = a.keep[v];
        const int32_t nl = best ? packed_label(best) : old;
        a.Lw[v] = nl;
        if (nl != old) atomicAdd(&a.changes[(uint32_t)i & (kChangeSlots - 1)], 1ull);
    }
}

// One lane per vertex of degree <= kTableLaneMaxDeg; the lane's table lives
// in LDS (cap key and cap count slots per lane), slot-major (slot i of lane l
// at word i * 64 + l), so the lanes' accesses to one slot fall in different
// banks.  The next edge's label loads while an edge is applied.
template <bool W, bool BUF>
__global__ __launch_bounds__(64) void k_table(StepArgs a, int32_t cap) {
    extern __shared__ uint32_t tbl[];
    const int lane = lane_id();
    const int32_t v = (int32_t)(blockIdx.x * 64 + lane);
    uint32_t* const K = tbl + lane;             // K[i * 64]: slot i's key
    uint32_t* const C = tbl + cap * 64 + lane;  // C[i * 64]: slot i's count
    bool changed = false;
    if (v < a.n && a.off[v + 1] - a.off[v] <= kTableLaneMaxDeg) {
        for (int i = 0; i < cap; ++i) { K[i * 64] = 0u; C[i * 64] = 0u; }
        const int32_t b = a.off[v], e = a.off[v + 1];
        uint32_t nkey = b < e ? (uint32_t)a.L[a.nbr[b]] + 1u : 0u;
        for (int32_t j = b; j < e; ++j) {
            const uint32_t key = nkey;
            if (j + 1 < e) nkey = (uint32_t)a.L[a.nbr[j + 1]] + 1u;
            const uint32_t f = W ? a.w[j] : 1u;
            int hit = -1, fr = -1;
            uint32_t cmin = 0xffffffffu;
            for (int i = 0; i < cap; ++i) {
                const uint32_t k = K[i * 64];
                if (k == key) hit = i;
                if (k == 0u) { if (fr < 0) fr = i; }
                else cmin = min(cmin, C[i * 64]);
            }
            if (hit >= 0) { C[hit * 64] += f; continue; }
            if (fr >= 0) { K[fr * 64] = key; C[fr * 64] = f; continue; }
            // table full
            const uint32_t d = min(f, cmin);
            int freed = -1;
            for (int i = 0; i < cap; ++i) {
                const uint32_t c = C[i * 64];
                const uint32_t nc = BUF ? (c > f ? c - f : 0u) : c - d;
                C[i * 64] = nc;
                if (nc == 0u) { K[i * 64] = 0u; if (freed < 0) freed = i; }
            }
            if (!BUF && f > d) { K[freed * 64] = key; C[freed * 64] = f - d; }
        }
        uint64_t best = 0ull;
        for (int i = 0; i < cap; ++i)
            if (K[i * 64]) best = max_u64(best, pack_score((int32_t)min(C[i * 64], 0x7fffffffu), K[i * 64]));
        const int32_t old = a.keep[v];
        const int32_t nl = best ? packed_label(best) : old;
        a.Lw[v] = nl;
        changed = nl != old;
    }
    unsigned long long bal = __ballot(changed);
    if (lane == 0 && bal)
        atomicAdd(&a.changes[blockIdx.x & (kChangeSlots - 1)], (unsigned long long)__popcll(bal));
}

template <int R, bool ALIASED>
static void set_countmin_limits() {
    auto set = [](const void* f) {
        (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 5 * 4096 * 4);
    };
    set((const void*)k_countmin<false, 64, R, ALIASED>);
    set((const void*)k_countmin<true, 64, R, ALIASED>);
    set((const void*)k_countmin_few<false, 1, R, ALIASED>);
    set((const void*)k_countmin_few<true, 1, R, ALIASED>);
    set((const void*)k_countmin_few<false, 4, R, ALIASED>);
    set((const void*)k_countmin_few<true, 4, R, ALIASED>);
    set((const void*)k_countmin<false, 256, R, ALIASED>);
    set((const void*)k_countmin<true, 256, R, ALIASED>);
    set((const void*)k_countmin<false, 1024, R, ALIASED>);
    set((const void*)k_countmin<true, 1024, R, ALIASED>);
    set((const void*)k_countmin_hub_sketch<false, R, ALIASED>);
    set((const void*)k_countmin_hub_sketch<true, R, ALIASED>);
    set((const void*)k_countmin_hub_est<R, ALIASED>);
}
// k_countmin takes rows * width * 4 bytes of dynamic LDS, up to 5 * 4096 * 4
// = 80 KB (the limits check_params enforces), above the 64 KB a launch gets
// without the attribute; k_table takes at most 64 * 2 * 64 * 4 = 32 KB.
void init_counting_kernels() {
    set_countmin_limits<1, false>();
    set_countmin_limits<2, false>();
    set_countmin_limits<3, false>();
    set_countmin_limits<4, false>();
    set_countmin_limits<5, false>();
    set_countmin_limits<3, true>();
    set_countmin_limits<4, true>();
}

// The counting methods' vertex lists (built once per session), in one
// array: count-min, the vertices of degree in (kCountminSmallDeg,
// kCountminWaveMaxDeg] (nmid of them), then those up to kCountminHubDeg
// (nwide: the ncm256 up to kCountminMidDeg first), then the hubs above (ncmhub, with their chunk list, sketches and
// maxima), then degrees 1..kCountminSmallDeg (nsmall) and 0 (niso);
// frequent and buffer, the vertices above kTableLaneMaxDeg (nwide).  The
// lists of one workgroup or wavefront per vertex, and the hubs, run largest
// degree first, so the longest counts start at once whatever the vertex ids.
int counting_wide_list(glp_session* s) {
    const HostCSR& g = s->g->csr;
    const bool cm = s->p.method == GLP_COUNTMIN;
    const int32_t lim = cm ? kCountminWaveMaxDeg : kTableLaneMaxDeg;
    std::vector<int32_t> wide, big, big1024, hubs, iso;
    std::vector<int32_t> small[kCountminSmallDeg + 1];  // by degree, so a wavefront's groups have alike degrees
    std::vector<int2> chunks;
    for (int32_t v = 0; v < g.n; ++v) {
        const int32_t d = g.offsets[v + 1] - g.offsets[v];
        if (cm && d > kCountminHubDeg) hubs.push_back(v);
        else if (cm && d > kCountminMidDeg) big1024.push_back(v);
        else if (d > lim) big.push_back(v);
        else if (cm && d > kCountminSmallDeg) wide.push_back(v);
        else if (cm && d > 0) small[d].push_back(v);
        else if (cm) iso.push_back(v);
    }
    auto deg = [&g](int32_t v) { return g.offsets[v + 1] - g.offsets[v]; };
    for (auto* list : {&wide, &big, &big1024, &hubs})
        std::stable_sort(list->begin(), list->end(), [&](int32_t x, int32_t y) { return deg(x) > deg(y); });
    for (int32_t h = 0; h < (int32_t)hubs.size(); ++h)
        for (int32_t c0 = 0; c0 < deg(hubs[h]); c0 += kCountminChunk) chunks.push_back(make_int2(h, c0));
    s->nmid = (int32_t)wide.size();
    for (int32_t v : wide) ++s->nmid_g[deg(v) > 256 ? 0 : deg(v) > 64 ? 1 : 2];
    s->ncm256 = (int32_t)big.size();
    big.insert(big.end(), big1024.begin(), big1024.end());
    s->nwide = (int32_t)big.size();
    s->ncmhub = (int32_t)hubs.size();
    s->ncmchunk = (int32_t)chunks.size();
    s->niso = (int32_t)iso.size();
    wide.insert(wide.end(), big.begin(), big.end());
    wide.insert(wide.end(), hubs.begin(), hubs.end());
    for (const auto& sd : small) wide.insert(wide.end(), sd.begin(), sd.end());
    s->nsmall = (int32_t)(wide.size() - s->nmid - s->nwide - s->ncmhub);
    // the small list's lane-group classes: degree 1, 2, 3-4, 5-8, 9-16
    for (int gi = 0, d = 1; gi < kCmSmallClasses; ++gi) {
        s->nsmall_g[gi] = 0;
        for (; d <= (1 << gi); ++d) s->nsmall_g[gi] += (int32_t)small[d].size();
    }
    wide.insert(wide.end(), iso.begin(), iso.end());
    if (wide.empty()) return GLP_OK;
    GLP_HIP(hipMalloc(&s->wide, wide.size() * 4));
    GLP_HIP(hipMemcpyAsync(s->wide, wide.data(), wide.size() * 4, hipMemcpyHostToDevice, s->stream));
    s->bytes += wide.size() * 4;
    if (!hubs.empty()) {
        const size_t sk = (size_t)hubs.size() * s->p.cm_rows * s->p.cm_width * 4;
        GLP_HIP(hipMalloc(&s->cm_chunks, chunks.size() * sizeof(int2)));
        GLP_HIP(hipMalloc(&s->cm_sketch, sk));
        GLP_HIP(hipMalloc(&s->cm_best, hubs.size() * 8));
        GLP_HIP(hipMalloc(&s->cm_keys, chunks.size() * (size_t)kCountminChunk * 4));
        GLP_HIP(hipMemcpyAsync(s->cm_chunks, chunks.data(), chunks.size() * sizeof(int2), hipMemcpyHostToDevice,
                               s->stream));
        GLP_HIP(hipMemsetAsync(s->cm_sketch, 0, sk, s->stream));
        GLP_HIP(hipMemsetAsync(s->cm_best, 0, hubs.size() * 8, s->stream));
        s->bytes += chunks.size() * (sizeof(int2) + (size_t)kCountminChunk * 4) + sk + hubs.size() * 8;
    }
    GLP_HIP(hipStreamSynchronize(s->stream));  // the host vectors are released on return
    return GLP_OK;
}

// The count-min launches of a step.
template <bool W, int R, bool ALIASED>
static void countmin_rows(glp_session* s, const StepArgs& a) {
    const uint32_t wd = (uint32_t)s->p.cm_width, m = cm_mod_magic(wd);
    const size_t lds = (size_t)R * wd * 4;
    const hipStream_t st = s->stream;
    const int32_t* small = s->wide + s->nmid + s->nwide + s->ncmhub;
    // lane groups of 1, 2, 4, 8 and 16
    const int32_t* n = s->nsmall_g;
    auto blocks = [](int64_t items) { return dim3((unsigned)((items + 255) / 256)); };
    const int32_t* at = small;
    if (n[0]) hipLaunchKernelGGL((k_countmin_small<W, 1, R, ALIASED>), blocks(n[0]), dim3(256), 0, st, a, at, n[0], wd, m);
    at += n[0];
    if (n[1])
        hipLaunchKernelGGL((k_countmin_small<W, 2, R, ALIASED>), blocks(2ll * n[1]), dim3(256), 0, st, a, at, n[1], wd, m);
    at += n[1];
    if (n[2])
        hipLaunchKernelGGL((k_countmin_small<W, 4, R, ALIASED>), blocks(4ll * n[2]), dim3(256), 0, st, a, at, n[2], wd, m);
    at += n[2];
    if (n[3])
        hipLaunchKernelGGL((k_countmin_small<W, 8, R, ALIASED>), blocks(8ll * n[3]), dim3(256), 0, st, a, at, n[3], wd, m);
    at += n[3];
    if (n[4])
        hipLaunchKernelGGL((k_countmin_small<W, 16, R, ALIASED>), blocks(16ll * n[4]), dim3(256), 0, st, a, at, n[4], wd, m);
    if (s->niso > 0) hipLaunchKernelGGL(k_countmin_keep, blocks(s->niso), dim3(256), 0, st, a, small + s->nsmall, s->niso);
    // the list runs largest degree first
    const int32_t n1024 = s->nmid_g[0], n256 = s->nmid_g[1], n64 = s->nmid_g[2];
    auto few = [](int32_t items) { return dim3((unsigned)((items + kCmVerts - 1) / kCmVerts)); };
    if (n1024) hipLaunchKernelGGL((k_countmin<W, 64, R, ALIASED>), dim3(n1024), dim3(64), lds, st, a, s->wide, wd, m);
    if (n256)
        hipLaunchKernelGGL((k_countmin_few<W, 4, R, ALIASED>), few(n256), dim3(64), lds, st, a, s->wide + n1024, n256,
                           wd, m);
    if (n64)
        hipLaunchKernelGGL((k_countmin_few<W, 1, R, ALIASED>), few(n64), dim3(64), lds, st, a, s->wide + n1024 + n256,
                           n64, wd, m);
    if (s->ncm256 > 0)
        hipLaunchKernelGGL((k_countmin<W, 256, R, ALIASED>), dim3(s->ncm256), dim3(256), lds, st, a, s->wide + s->nmid,
                           wd, m);
    if (s->nwide > s->ncm256)
        hipLaunchKernelGGL((k_countmin<W, 1024, R, ALIASED>), dim3((unsigned)(s->nwide - s->ncm256)), dim3(1024), lds, st,
                           a, s->wide + s->nmid + s->ncm256, wd, m);
    if (s->ncmhub > 0) {
        const int32_t* hubs = s->wide + s->nmid + s->nwide;
        const dim3 grid((unsigned)s->ncmchunk);
        hipLaunchKernelGGL((k_countmin_hub_sketch<W, R, ALIASED>), grid, dim3(1024), lds, st, a, hubs, s->cm_chunks,
                           s->cm_sketch, s->cm_keys, wd, m);
        hipLaunchKernelGGL((k_countmin_hub_est<R, ALIASED>), grid, dim3(1024), lds, st, a, hubs, s->cm_chunks,
                           s->cm_sketch, s->cm_keys, s->cm_best, wd, m);
        hipLaunchKernelGGL(k_countmin_hub_final, dim3(s->ncmhub), dim3(256), 0, st, a, hubs, s->cm_sketch, s->cm_best,
                           (int32_t)(R * wd));
    }
}
template <bool W>
static void countmin_step(glp_session* s, const StepArgs& a) {
    // aliasing touches rows 2 and 3 of three or four
    const bool al = s->p.cm_aliased != 0;
    switch (s->p.cm_rows) {
        case 1: return countmin_rows<W, 1, false>(s, a);
        case 2: return countmin_rows<W, 2, false>(s, a);
        case 3: return al ? countmin_rows<W, 3, true>(s, a) : countmin_rows<W, 3, false>(s, a);
        case 4: return al ? countmin_rows<W, 4, true>(s, a) : countmin_rows<W, 4, false>(s, a);
        default: return countmin_rows<W, 5, false>(s, a);
    }
}

int enqueue_counting_step(glp_session* s) {
    const DeviceGraph& dg = *s->g->dev;
    StepArgs a{};
    a.off = dg.off;
    a.nbr = dg.nbr;
    a.w = dg.w;
    a.n = s->n;
    a.t = s->t + 1;
    a.changes = step_counters(s);
    a.L = s->L[s->cur];
    a.keep = s->L[s->cur];
    a.Lw = s->L[s->cur ^ 1];
    const bool w = s->p.weighted != 0;
    if (s->n > 0) {
        if (s->p.method == GLP_COUNTMIN) {
            if (w) countmin_step<true>(s, a);
            else countmin_step<false>(s, a);
        } else {
            const size_t lds = (size_t)64 * 2 * s->p.table_cap * 4;
            const unsigned grid = (unsigned)((s->n + 63) / 64);
            const bool buf = s->p.method == GLP_BUFFER;
            const int32_t cap = s->p.table_cap;
            const unsigned wgrid = (unsigned)((s->nwide + 3) / 4);
            if (buf) {
                if (w) hipLaunchKernelGGL((k_table<true, true>), dim3(grid), dim3(64), lds, s->stream, a, cap);
                else hipLaunchKernelGGL((k_table<false, true>), dim3(grid), dim3(64), lds, s->stream, a, cap);
                if (s->nwide > 0) {
                    if (w) hipLaunchKernelGGL((k_table_wave<true, true>), dim3(wgrid), dim3(256), 0, s->stream, a,
                                              s->wide, s->nwide, cap);
                    else hipLaunchKernelGGL((k_table_wave<false, true>), dim3(wgrid), dim3(256), 0, s->stream, a,
                                            s->wide, s->nwide, cap);
                }
            } else {
                if (w) hipLaunchKernelGGL((k_table<true, false>), dim3(grid), dim3(64), lds, s->stream, a, cap);
                else hipLaunchKernelGGL((k_table<false, false>), dim3(grid), dim3(64), lds, s->stream, a, cap);
                if (s->nwide > 0) {
                    if (w) hipLaunchKernelGGL((k_table_wave<true, false>), dim3(wgrid), dim3(256), 0, s->stream,
                                              a, s->wide, s->nwide, cap);
                    else hipLaunchKernelGGL((k_table_wave<false, false>), dim3(wgrid), dim3(256), 0, s->stream,
                                            a, s->wide, s->nwide, cap);
                }
            }
        }
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return set_error(GLP_E_HIP, "counting launch: %s", hipGetErrorString(e));
    }
    int rc = end_step(s, a.nbr, a.Lw, false);
    if (rc != GLP_OK) return rc;
    s->cur ^= 1;
    s->t += 1;
    return GLP_OK;
}

// SLPA post-processing (builder-defined; the reference's SLPA keeps one
// memory slot and has no threshold): for vertex v the labels whose count in
// M_v[0..t] is >= r*(t+1), ascending, and the dominant label (highest count,
// then highest label).
__global__ __launch_bounds__(64) void k_slpa_post(const int32_t* __restrict__ mem, int32_t n,
                                                  int32_t rows, int32_t r_num, int32_t r_den,
                                                  int32_t kmax, int32_t* dominant, int32_t* nsets,
                                                  int32_t* sets) {
    const int32_t v = (int32_t)(blockIdx.x * blockDim.x + threadIdx.x);
    if (v >= n) return;
    int32_t vals[256];
    for (int32_t i = 0; i < rows; ++i) vals[i] = mem[(size_t)i * n + v];
    for (int32_t i = 1; i < rows; ++i) {  // insertion sort, ascending
        const int32_t x = vals[i];
        int32_t j = i - 1;
        while (j >= 0 && vals[j] > x) { vals[j + 1] = vals[j]; --j; }
        vals[j + 1] = x;
    }
    uint64_t best = 0ull;
    int32_t kept = 0;
    for (int32_t i = 0; i < rows;) {
        int32_t j = i;
        while (j < rows && vals[j] == vals[i]) ++j;
        const int32_t c = j - i;
        best = max(best, ((uint64_t)(uint32_t)c << 32) | ((uint32_t)vals[i] + 1u));
        if ((int64_t)c * r_den >= (int64_t)r_num * rows) {
            if (kept < kmax) sets[(size_t)v * kmax + kept] = vals[i];
            ++kept;
        }
        i = j;
    }
    for (int32_t k = kept; k < kmax; ++k) sets[(size_t)v * kmax + k] = -1;
    if (dominant) dominant[v] = packed_label(best);
    if (nsets) nsets[v] = kept;
}

int slpa_post(glp_session* s, int32_t kmax, int32_t* dominant, int32_t* nsets, int32_t* sets) {
    const int32_t n = s->n;
    if (n == 0) return GLP_OK;
    const int32_t rows = s->t + 1;
    int32_t *d_dom = nullptr, *d_ns = nullptr, *d_sets = nullptr;
    struct Guard {
        int32_t** p[3];
        ~Guard() { for (auto q : p) (void)hipFree(*q); }
    } guard{{&d_dom, &d_ns, &d_sets}};
    GLP_HIP(hipMalloc(&d_dom, (size_t)n * 4));
    GLP_HIP(hipMalloc(&d_ns, (size_t)n * 4));
    if (kmax > 0) GLP_HIP(hipMalloc(&d_sets, (size_t)n * kmax * 4));
    hipLaunchKernelGGL(k_slpa_post, dim3((n + 63) / 64), dim3(64), 0, s->stream, s->mem, n, rows,
                       s->p.slpa_r_num, s->p.slpa_r_den, kmax, d_dom, d_ns, d_sets);
    GLP_HIP(hipGetLastError());
    int rc = GLP_OK;
    if (dominant) rc = copy_to_host(*s->staging, dominant, d_dom, (size_t)n * 4, s->stream);
    if (!rc && nsets) rc = copy_to_host(*s->staging, nsets, d_ns, (size_t)n * 4, s->stream);
    if (!rc && kmax > 0 && sets) rc = copy_to_host(*s->staging, sets, d_sets, (size_t)n * kmax * 4, s->stream);
    GLP_HIP(hipStreamSynchronize(s->stream));  // before the arrays go
    return rc;
}

}  // namespace glp
