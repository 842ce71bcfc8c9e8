// Auxiliary kernels of a step (pick, gather, frontier, volumes, dominant
// label, step end) and the dispatch of its counting to the tier kernels
// (tiers.h, instantiated per hook set in tiers_*.hip).

#include "tiers.h"

#include <algorithm>

namespace glp {

// ------------------------------------------------------------ auxiliaries ----
template <class H>
__global__ __launch_bounds__(256) void k_pick(StepArgs a, int32_t* __restrict__ shown) {
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v < a.n) shown[v] = H::pick_label(a, (int32_t)v);
}

// adj[j] = L[nbr[j]] (header/kernel.cuh:225-256 gather_labels), four
// neighbours per lane with 16-byte streaming loads and stores.
typedef int32_t v4i32 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void gather_all(const int32_t* __restrict__ nbr,
                                           const int32_t* __restrict__ L,
                                           int32_t* __restrict__ adj, int64_t m) {
    const int64_t nvec = m >> 2;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const v4i32* nb4 = reinterpret_cast<const v4i32*>(nbr);
    v4i32* ad4 = reinterpret_cast<v4i32*>(adj);
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nvec; i += stride) {
        const v4i32 u = __builtin_nontemporal_load(&nb4[i]);
        v4i32 r;
        r.x = L[u.x];
        r.y = L[u.y];
        r.z = L[u.z];
        r.w = L[u.w];
        __builtin_nontemporal_store(r, &ad4[i]);
    }
    const int64_t t = (nvec << 2) + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (blockIdx.x == 0 && t < m) adj[t] = L[nbr[t]];
}

__global__ __launch_bounds__(256) void k_gather(const int32_t* __restrict__ nbr,
                                                const int32_t* __restrict__ L,
                                                int32_t* __restrict__ adj, int64_t m) {
    gather_all(nbr, L, adj, m);
}

// ---------------------------------------------------- frontier gather ----
// The frontier form of the separate gather (header/kernel.cuh:21-78's
// if_update gathers) pushes labels from sources instead of pulling them per
// edge.  An inverse index lists, for each vertex u, the CSR positions j with
// nbr[j] = u (the reference gets the same lists by sorting (nbr[j], j) pairs
// with thrust::sort_by_key, prop/layeredLprop.cuh:228-237, and reads them in
// gather_labels_inverse, header/kernel.cuh:64-78; a counting pass builds
// them here in O(m)).  adj holds the labels of two steps back, so writing
// L[u] to the positions of every u that changed in the previous step makes
// it equal L[nbr]: the work is the changed sources' in-edges, not m.
//
// With the two-step lookahead (the reference's onestep = false,
// tutorial/Lprop.cuh:383-461) adj alternates between two buffers, each
// refreshed every other step, and a vertex's bit records a change against
// its label of two steps back: a vertex that flips between two labels then
// pushes nothing.
//
// Frontier control words used here (the rest of fctl is the tiers'):
//   fctl[3] = steps adj has been gathered in, at most 2 (set by k_end_step,
//             0 after a reset), fctl[4] = push entries listed for this step,
//   fctl[5] = in-edges of the sources that changed in the previous step,
//   fctl[6] = 1 when that step changed at most fctl[7] labels (a changed
//             vertex has an in-edge, so more changes than that rule the push
//             out before its sources are counted),
//   fctl[7] = m / kPushRatio, the most in-edges a push takes (set at reset).
// A push writes each in-edge's label to a random position; measured on
// RMAT-25 that costs about five times a streamed edge of the full gather, so
// the push is taken only below m / 8 in-edges.
constexpr int32_t kPushChunk = 256;   // in-edges per push entry at most
constexpr int64_t kPushRatio = 8;

__global__ __launch_bounds__(256) void k_inv_count(const int32_t* __restrict__ nbr, int64_t m,
                                                   int32_t* __restrict__ cnt) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < m; j += stride)
        atomicAdd(&cnt[nbr[j]], 1);
}
// cursor[u] starts at inv_off[u]; each edge claims the next slot of its
// source's list (the order inside a list does not matter).
__global__ __launch_bounds__(256) void k_inv_fill(const int32_t* __restrict__ nbr, int64_t m,
                                                  int32_t* __restrict__ cursor,
                                                  int32_t* __restrict__ inv_pos) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < m; j += stride)
        inv_pos[atomicAdd(&cursor[nbr[j]], 1)] = (int32_t)j;
}

// Exclusive scan of int32 counts in place (sums < 2^31): block sums, a scan
// of the sums in one workgroup, then each block rescans its run.
constexpr int kScanPer = 16;                       // elements per thread
constexpr int kScanBlock = 256 * kScanPer;         // elements per workgroup
__global__ __launch_bounds__(256) void k_scan_sums(const int32_t* __restrict__ x, int64_t count,
                                                   int32_t* __restrict__ sums) {
    const int64_t b0 = (int64_t)blockIdx.x * kScanBlock + (int64_t)threadIdx.x * kScanPer;
    int32_t s = 0;
    for (int i = 0; i < kScanPer; ++i)
        if (b0 + i < count) s += x[b0 + i];
    int32_t total;
    (void)block_excl_sum(s, &total);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}
__global__ __launch_bounds__(256) void k_scan_top(int32_t* __restrict__ sums, int64_t nsums) {
    int32_t carry = 0;
    for (int64_t b = 0; b < nsums; b += 256) {
        const int64_t i = b + threadIdx.x;
        const int32_t x = i < nsums ? sums[i] : 0;
        int32_t total;
        const int32_t ex = block_excl_sum(x, &total);
        if (i < nsums) sums[i] = carry + ex;
        carry += total;
    }
}
__global__ __launch_bounds__(256) void k_scan_apply(int32_t* __restrict__ x, int64_t count,
                                                    const int32_t* __restrict__ sums) {
    const int64_t b0 = (int64_t)blockIdx.x * kScanBlock + (int64_t)threadIdx.x * kScanPer;
    int32_t v[kScanPer];
    int32_t s = 0;
    for (int i = 0; i < kScanPer; ++i) {
        v[i] = b0 + i < count ? x[b0 + i] : 0;
        s += v[i];
    }
    int32_t total;
    int32_t run = sums[blockIdx.x] + block_excl_sum(s, &total);
    for (int i = 0; i < kScanPer; ++i) {
        if (b0 + i < count) x[b0 + i] = run;
        run += v[i];
    }
}

// One push entry: label to write, first in-edge position, in-edge count.
struct PushEntry {
    int32_t label, begin, count, pad;
};

// Push entries of the sources whose bit is set in chg (the previous step's
// changes), one per kPushChunk in-edges, in vertex order: each thread takes
// one bitmap word; k_push_count sums every workgroup's entries and in-edges,
// k_push_scan turns the sums into offsets and totals (fctl[4], fctl[5]), and
// k_push_write lists the entries when the gather is going to push them.
// No atomics: the totals of a step with many changes come at the cost of one
// read of the bitmap.
__device__ __forceinline__ void push_word_counts(const uint32_t* __restrict__ chg, int64_t w,
                                                 int64_t nwords, const int32_t* __restrict__ inv_off,
                                                 int32_t* cnt, int32_t* edges) {
    const uint32_t bits = w < nwords ? chg[w] : 0u;
    int32_t c = 0, e = 0;
    if (__builtin_popcount(bits) >= 8) {
        // many changed: read the word's 33 offsets at once (inv_off + 32w is
        // 128-byte aligned, and inv_off has n + 1 >= 32w + 33 entries when
        // bit 31 can be set; the last word reads up to its highest bit + 1)
        const int32_t* o = inv_off + w * 32;
        const int hi = 32 - __builtin_clz(bits);  // highest set bit + 1
        int32_t prev = o[0];
#pragma unroll
        for (int i = 0; i < 32; ++i) {
            if (i < hi) {
                const int32_t next = o[i + 1];
                if ((bits >> i) & 1u) {
                    const int32_t d = next - prev;
                    c += (d + kPushChunk - 1) / kPushChunk;
                    e += d;
                }
                prev = next;
            }
        }
    } else {
        for (uint32_t b = bits; b; b &= b - 1u) {
            const int32_t u = (int32_t)(w * 32 + __builtin_ctz(b));
            const int32_t d = inv_off[u + 1] - inv_off[u];
            c += (d + kPushChunk - 1) / kPushChunk;
            e += d;
        }
    }
    *cnt = c;
    *edges = e;
}
// need: steps adj must have been gathered in (1; 2 with the lookahead,
// whose two buffers are each first filled by a full gather).  The rule-out
// by the previous step's change count holds for one-step changes only.
__device__ __forceinline__ bool push_possible(const int32_t* fctl, int32_t need) {
    return fctl[3] >= need && (need == 2 || fctl[6] != 0);
}
__global__ __launch_bounds__(256) void k_push_count(const uint32_t* __restrict__ chg, int64_t nwords,
                                                    const int32_t* __restrict__ inv_off,
                                                    int2* __restrict__ psum,
                                                    const int32_t* __restrict__ fctl, int32_t need) {
    if (!push_possible(fctl, need)) return;  // the gather rewrites every edge this step
    int32_t c, e, tc, te;
    push_word_counts(chg, (int64_t)blockIdx.x * blockDim.x + threadIdx.x, nwords, inv_off, &c, &e);
    (void)block_excl_sum(c, &tc);
    (void)block_excl_sum(e, &te);
    if (threadIdx.x == 0) psum[blockIdx.x] = make_int2(tc, te);
}
__global__ __launch_bounds__(256) void k_push_scan(int2* __restrict__ psum, int64_t nblocks,
                                                   int32_t* __restrict__ fctl, int32_t need) {
    if (!push_possible(fctl, need)) return;
    int32_t carry = 0, edges = 0;
    for (int64_t b = 0; b < nblocks; b += 256) {
        const int64_t i = b + threadIdx.x;
        const int2 x = i < nblocks ? psum[i] : make_int2(0, 0);
        int32_t tc, te;
        const int32_t ex = block_excl_sum(x.x, &tc);
        (void)block_excl_sum(x.y, &te);
        if (i < nblocks) psum[i].x = carry + ex;
        carry += tc;
        edges += te;
    }
    if (threadIdx.x == 0) {
        fctl[4] = carry;
        fctl[5] = edges;
    }
}
__device__ __forceinline__ bool push_taken(const int32_t* fctl, int32_t need) {
    return push_possible(fctl, need) && fctl[5] <= fctl[7];
}
__global__ __launch_bounds__(256) void k_push_write(const uint32_t* __restrict__ chg, int64_t nwords,
                                                    const int32_t* __restrict__ inv_off,
                                                    const int32_t* __restrict__ L,
                                                    const int2* __restrict__ psum,
                                                    PushEntry* __restrict__ ent,
                                                    const int32_t* __restrict__ fctl, int32_t need) {
    if (!push_taken(fctl, need)) return;
    const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int32_t c, e, tc;
    push_word_counts(chg, w, nwords, inv_off, &c, &e);
    int32_t k = psum[blockIdx.x].x + block_excl_sum(c, &tc);
    if (c == 0) return;
    for (uint32_t b = chg[w]; b; b &= b - 1u) {
        const int32_t u = (int32_t)(w * 32 + __builtin_ctz(b));
        const int32_t end = inv_off[u + 1];
        const int32_t lab = L[u];
        for (int32_t p = inv_off[u]; p < end; p += kPushChunk)
            ent[k++] = PushEntry{lab, p, min(kPushChunk, end - p), 0};
    }
}

// The gather of a frontier step: the first step, and any step whose changed
// sources have more than m / kPushRatio in-edges, rewrite every edge
// (gather_all); otherwise each wave takes 64 push entries at a time and
// spreads their in-edges evenly over its lanes.
__global__ __launch_bounds__(256) void k_gather_frontier(const int32_t* __restrict__ nbr,
                                                         const int32_t* __restrict__ L,
                                                         int32_t* __restrict__ adj, int64_t m,
                                                         const int32_t* __restrict__ inv_pos,
                                                         const PushEntry* __restrict__ ent,
                                                         const int32_t* __restrict__ fctl, int32_t need) {
    if (!push_taken(fctl, need)) {
        gather_all(nbr, L, adj, m);
        return;
    }
    const int64_t nent = fctl[4];
    const int lane = lane_id();
    const int64_t nwaves = (int64_t)gridDim.x * (blockDim.x >> 6);
    const int64_t wave = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    for (int64_t b0 = wave * 64; b0 < nent; b0 += nwaves * 64) {
        PushEntry e{0, 0, 0, 0};
        if (b0 + lane < nent) e = ent[b0 + lane];
        const int32_t incl = wave_incl_sum(e.count);
        const int32_t total = shfl_i32(incl, 63);
        for (int32_t f0 = 0; f0 < total; f0 += 64) {
            const int32_t f = f0 + lane;
            // owner: the smallest lane whose inclusive sum exceeds f
            int lo = 0, hi = 63;
#pragma unroll
            for (int k = 0; k < 6; ++k) {
                const int mid = (lo + hi) >> 1;
                if (shfl_i32(incl, mid) <= f) lo = mid + 1;
                else hi = mid;
            }
            const int32_t o_incl = shfl_i32(incl, lo);
            const int32_t o_cnt = shfl_i32(e.count, lo);
            const int32_t o_beg = shfl_i32(e.begin, lo);
            const int32_t o_lab = shfl_i32(e.label, lo);
            if (f < total) adj[inv_pos[o_beg + f - (o_incl - o_cnt)]] = o_lab;
        }
    }
}

__global__ void k_fill_i32(int32_t* p, int32_t value, int64_t count) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride)
        p[i] = value;
}
// Layered LP's volume V(l) = #{v : L[v] = l} of the labels a step wrote
// (header/kernel.cuh:2626's gcounter_temp, counted in a pass of its own).
// While labels consolidate, a few labels each hold millions of vertices
// spread over the id range, and one global atomic per vertex on their
// counters serialises in L2.  A workgroup counts a chunk of kVolChunk
// vertices in an LDS table of (label+1, count) slots (each wave first merges
// its row's first label) and flushes one atomic per distinct label; a label
// that finds no slot within kVolProbe probes goes to global memory directly.
// Edge-less vertices keep their label for ever, and in a power-law graph they
// are half of all vertices, each with a label of its own: the pass that
// clears V gives them their 1, and only the others are counted here.  A
// chunk of 16,384 keeps the global atomics few (8,192: more of them than the
// extra workgroups bring); 16 waves share it, which hides the latency of the
// table's probes.  R-MAT scale 22: 137 us with every vertex counted by
// 256-thread workgroups, 118 without the edge-less ones, 108 with 1,024
// threads; tens of jobs of up to 65,536 vertices in one launch: 105, 82, 40.
constexpr int kVolThreads = 1024;
constexpr int kVolChunk = 16384;
constexpr uint32_t kVolSlots = 2048;
constexpr int kVolProbe = 8;
constexpr int kVolRows = 4;  // loads in flight per lane
__device__ __forceinline__ bool counted_alone(const int32_t* __restrict__ off, int64_t v, int32_t label) {
    return label == (int32_t)v && off[v] == off[v + 1];
}
__device__ __forceinline__ void volume_body(const int32_t* __restrict__ off, const int32_t* __restrict__ L,
                                            int32_t* __restrict__ V, int32_t n, uint32_t blk) {
    __shared__ unsigned long long T[kVolSlots];
    const int lane = lane_id();
    for (uint32_t i = threadIdx.x; i < kVolSlots; i += kVolThreads) T[i] = 0ull;
    __syncthreads();
    const int64_t c0 = (int64_t)blk * kVolChunk;
    const int64_t c1 = min((int64_t)n, c0 + kVolChunk);
    auto count = [&](int32_t l) {  // one row of a wave; -1: nothing to count
        uint32_t c = 1u;
        const unsigned long long act = __ballot(l >= 0);
        if (act == 0ull) return;
        const int first = (int)__builtin_ctzll(act);
        const int32_t lead = __builtin_amdgcn_readlane(l, first);
        const unsigned long long sm = __ballot(l == lead);
        if (l == lead) {
            if (lane == first) c = (uint32_t)__popcll(sm);
            else l = -1;  // merged into the first lane
        }
        if (l < 0) return;
        const uint32_t key = (uint32_t)l + 1u;
        uint32_t h = fmix32(key) & (kVolSlots - 1u);
        bool done = false;
        for (int k = 0; k < kVolProbe && !done; ++k) {
            unsigned long long cur = lds_load(&T[h]);
            if (cur == 0ull) {
                cur = atomicCAS(&T[h], 0ull, ((unsigned long long)key << 32) | c);
                if (cur == 0ull) done = true;
            }
            if (!done && (uint32_t)(cur >> 32) == key) {
                atomicAdd(&T[h], (unsigned long long)c);
                done = true;
            }
            h = (h + 1u) & (kVolSlots - 1u);
        }
        if (!done) atomicAdd(&V[l], (int32_t)c);
    };
    for (int64_t r = c0 + (threadIdx.x & ~63); r < c1; r += kVolThreads * kVolRows) {  // wave-uniform rows
        int32_t l[kVolRows];
#pragma unroll
        for (int i = 0; i < kVolRows; ++i) {
            const int64_t at = r + i * kVolThreads + lane, v = min(at, c1 - 1);
            const int32_t x = L[v], d = off[v + 1] - off[v];  // always loaded: no branch between the rows' loads
            l[i] = (at >= c1) | ((d == 0) & (x == (int32_t)v)) ? -1 : x;
        }
#pragma unroll
        for (int i = 0; i < kVolRows; ++i) count(l[i]);
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < kVolSlots; i += kVolThreads) {
        const unsigned long long x = T[i];
        if (x) atomicAdd(&V[(uint32_t)(x >> 32) - 1u], (int32_t)(uint32_t)x);
    }
}
__global__ __launch_bounds__(kVolThreads) void k_volume(const int32_t* __restrict__ off,
                                                        const int32_t* __restrict__ L, int32_t* __restrict__ V,
                                                        int32_t n) {
    volume_body(off, L, V, n, blockIdx.x);
}

// Folded forms for the serving path: one launch zeroes (before the tiers)
// or fills (after them) the write-side volumes of every layered job of a
// step; cum[j] is job j's first workgroup, as for k_multi.
constexpr int kZeroPerBlock = 256 * 16;
__global__ __launch_bounds__(256) void k_multi_zero(const VolumeJob* __restrict__ jobs,
                                                    const int32_t* __restrict__ cum, int32_t nj) {
    const int32_t j = job_of(cum, nj, blockIdx.x);
    const VolumeJob& jb = jobs[j];
    const int64_t b0 = (int64_t)(blockIdx.x - (uint32_t)cum[j]) * kZeroPerBlock;
    const int64_t b1 = min((int64_t)jb.n, b0 + kZeroPerBlock);
    for (int64_t i = b0 + threadIdx.x; i < b1; i += 256) jb.V[i] = counted_alone(jb.off, i, jb.L[i]) ? 1 : 0;
}
__global__ __launch_bounds__(kVolThreads) void k_multi_volume(const VolumeJob* __restrict__ jobs,
                                                              const int32_t* __restrict__ cum, int32_t nj) {
    const int32_t j = job_of(cum, nj, blockIdx.x);
    volume_body(jobs[j].off, jobs[j].L, jobs[j].V, jobs[j].n, blockIdx.x - (uint32_t)cum[j]);
}
// The slot-score jobs' records LV[u] = {L[u], V[L[u]]}, kZeroPerBlock rows
// per workgroup.
__global__ __launch_bounds__(256) void k_multi_records(const VolumeJob* __restrict__ jobs,
                                                       const int32_t* __restrict__ cum, int32_t nj) {
    const int32_t j = job_of(cum, nj, blockIdx.x);
    const VolumeJob& jb = jobs[j];
    const int64_t b0 = (int64_t)(blockIdx.x - (uint32_t)cum[j]) * kZeroPerBlock;
    const int64_t b1 = min((int64_t)jb.n, b0 + kZeroPerBlock);
    for (int64_t i = b0 + threadIdx.x; i < b1; i += 256) {
        const int32_t l = jb.L[i];
        jb.LV[i] = make_int2(l, jb.V[l]);
    }
}

void volume_job_blocks(int32_t n, int32_t* zero_blocks, int32_t* volume_blocks) {
    *zero_blocks = (int32_t)(((int64_t)n + kZeroPerBlock - 1) / kZeroPerBlock);
    *volume_blocks = (int32_t)(((int64_t)n + kVolChunk - 1) / kVolChunk);
}

int launch_multi_volume(VolumeMode mode, const VolumeJob* jobs, const int32_t* cum, int32_t nj, int32_t grid,
                        hipStream_t s) {
    if (nj == 0 || grid == 0) return GLP_OK;
    if (mode == kVolumeZero) hipLaunchKernelGGL(k_multi_zero, dim3(grid), dim3(256), 0, s, jobs, cum, nj);
    else if (mode == kVolumeRecords) hipLaunchKernelGGL(k_multi_records, dim3(grid), dim3(256), 0, s, jobs, cum, nj);
    else hipLaunchKernelGGL(k_multi_volume, dim3(grid), dim3(kVolThreads), 0, s, jobs, cum, nj);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? GLP_OK : set_error(GLP_E_HIP, "folded volume launch: %s", hipGetErrorString(e));
}

// The write-side volumes before the step's labels are counted (L: any label
// buffer, edge-less vertices hold their label in both).
__global__ void k_volume_init(const int32_t* __restrict__ off, const int32_t* __restrict__ L, int32_t* __restrict__ V,
                              int32_t n) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        V[i] = counted_alone(off, i, L[i]) ? 1 : 0;
}
// The same, and the slot-score records LV from the read-side volumes Vr.
__global__ void k_label_volumes(const int32_t* __restrict__ off, const int32_t* __restrict__ L,
                                const int32_t* __restrict__ Vr, int2* __restrict__ LV, int32_t* __restrict__ Vw,
                                int32_t n) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const int32_t l = L[i];
        LV[i] = make_int2(l, Vr[l]);
        Vw[i] = counted_alone(off, i, l) ? 1 : 0;
    }
}
__global__ void k_iota(int32_t* p, int64_t count) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride)
        p[i] = (int32_t)i;
}
// The end of `rows` plain steps (no frontier, no dominant label): wave i sums
// rows i, i + 16, ... of change counters into the ring.  One launch for the
// steps of a call (at most kAccRows) instead of one each: on a graph of a
// thousand vertices it was half of a step's 10 us.
__global__ __launch_bounds__(1024) void k_end_steps(unsigned long long* acc, int32_t rows, unsigned long long* ring,
                                                    int32_t* ctr, int32_t ring_size) {
    const int lane = lane_id();
    const int32_t t = *ctr;
    for (int32_t r = threadIdx.x >> 6; r < rows; r += 16) {
        unsigned long long* row = acc + (size_t)r * kChangeSlots;
        unsigned long long x = 0ull;
#pragma unroll
        for (int i = 0; i < kChangeSlots; i += 64) {
            x += row[i + lane];
            row[i + lane] = 0ull;
        }
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) x += shfl_u64(x, lane ^ d);
        if (lane == 0) ring[(t + r) % ring_size] = x;
    }
    __syncthreads();
    if (threadIdx.x == 0) *ctr = t + rows;
}

// A session's reset (ResetArgs; seeded labels as header/kernel.cuh:453-466):
// launch bound on small graphs, one launch
// instead of seven.
__global__ __launch_bounds__(256) void k_reset(ResetArgs r) {
    const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t v = t0; v < r.n; v += stride) {
        const int32_t l = r.unseeded || (r.seeds && !r.seeds[v]) ? -1 : (int32_t)v;
        r.L[0][v] = l;
        r.L[1][v] = l;
        if (r.V[0]) {
            r.V[0][v] = 1;  // V_0(l) = #{u : L_0[u] = l} = 1
            r.V[1][v] = 0;
        }
        if (r.mem) r.mem[v] = (int32_t)v;  // M_v[0] = v
    }
#pragma unroll
    for (int k = 0; k < 7; ++k)
        if (r.zero[k])
            for (int64_t i = t0; i < r.zero_words[k]; i += stride) r.zero[k][i] = 0;
    if (t0 == 0 && r.fctl)
        for (int i = 0; i < 8; ++i) r.fctl[i] = r.fctl_words[i];
    if (t0 == 0 && r.domctl)
        for (int i = 0; i < 4; ++i) r.domctl[i] = i == 0 ? 1 : 0;
}

// Sums and clears the step's change counters into the ring and advances
// the step counter.  One workgroup of kChangeSlots threads.
// With a frontier control block fctl = {all_active, mark, threshold, ...}:
// the next step recomputes everything unless this step marked, and marks
// when this step changed at most `threshold` labels; the frontier gather's
// words 3-5 are set up for the next step.
// With dom.ctl set, the next step's dominant label (see k_dominant_edges):
// kChangeSlots edges spread evenly over the CSR show their neighbours' new
// labels, and a label on at least kDomShare of them is it (its share of the
// edges to within 2%; which label is taken changes no result).
// dom.ctl = {1 when there is none, 0, the label}.
struct DominantSample {
    const int32_t* nbr;
    const int32_t* L;  // the labels this step wrote
    int64_t m;         // > 0
    int32_t* ctl;
};
constexpr uint32_t kDomShare = kChangeSlots / 2;
__global__ __launch_bounds__(kChangeSlots) void k_end_step(unsigned long long* acc,
                                                           unsigned long long* ring, int32_t* ctr,
                                                           int32_t ring_size, int32_t* fctl,
                                                           DominantSample dom) {
    if (dom.ctl) {  // uniform
        __shared__ unsigned long long T[2 * kChangeSlots], s_red[kChangeSlots / 64];
        T[threadIdx.x] = 0ull;
        T[threadIdx.x + kChangeSlots] = 0ull;
        const int32_t u = dom.nbr[(int64_t)threadIdx.x * dom.m / kChangeSlots];
        const uint32_t key = (uint32_t)dom.L[u] + 1u;
        __syncthreads();
        const uint32_t at = kc_insert(T, 2 * kChangeSlots - 1, key, 1u) & ~kClaimed;
        __syncthreads();
        const uint64_t top =
            block_max_u64<kChangeSlots>(((uint64_t)(uint32_t)T[at] << 32) | threadIdx.x, s_red);
        if (threadIdx.x == 0) {
            s_red[0] = top;
            if ((uint32_t)(top >> 32) < kDomShare) dom.ctl[0] = 1;
        }
        __syncthreads();
        if ((uint32_t)s_red[0] == threadIdx.x && (uint32_t)(s_red[0] >> 32) >= kDomShare) {
            dom.ctl[0] = 0;
            dom.ctl[2] = (int32_t)key - 1;
        }
    }
    __shared__ unsigned long long part[kChangeSlots / 64];
    unsigned long long x = acc[threadIdx.x];
    acc[threadIdx.x] = 0ull;
    const int lane = lane_id();
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) x += shfl_u64(x, lane ^ d);
    if (lane == 0) part[threadIdx.x >> 6] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long sum = 0ull;
        for (int i = 0; i < kChangeSlots / 64; ++i) sum += part[i];
        const int32_t t = *ctr;
        ring[t % ring_size] = sum;
        *ctr = t + 1;
        if (fctl) {
            const int32_t marked = fctl[1];
            fctl[0] = marked ? 0 : 1;
            fctl[1] = sum <= (unsigned long long)fctl[2] ? 1 : 0;
            fctl[3] = min(fctl[3] + 1, 2);  // steps a frontier gather has filled adj in
            fctl[4] = 0;
            fctl[5] = 0;
            fctl[6] = sum <= (unsigned long long)fctl[7] ? 1 : 0;
        }
    }
}

// The dominant label of a step.  Once an R-MAT graph's labels converge, one
// label D shows on most edges, yet every edge still fetched its neighbour's
// 4-byte label, a random 128-byte line; those lines bound the tiers.  Three
// passes over bits settle the vertices that have D on more than half of their
// edges, whatever the other labels; the tiers recompute the rest (act = 1):
//  k_dominant_bits    bit v: vertex v shows D (n/8 bytes)
//  k_dominant_edges   bit j: edge j's neighbour shows D (m/8 bytes), a stream
//                     over the CSR whose lookups mostly stay in LDS
//  k_dominant_decide  a vertex's count is the population count of its edges'
//                     bits
// Without a dominant label (ctl[0] = 1) all three return at once.
// (and bit b of `blocks`: all of vertices [64 b, 64 b + 64) do)
__global__ __launch_bounds__(256) void k_dominant_bits(const int32_t* __restrict__ L, int32_t n,
                                                       const int32_t* __restrict__ ctl,
                                                       unsigned long long* __restrict__ bits,
                                                       uint32_t* __restrict__ blocks) {
    if (ctl[0]) return;
    const int32_t label = __builtin_amdgcn_readfirstlane(ctl[2]);
    constexpr int kRows = 8;  // loads in flight per lane
    const int lane = lane_id();
    const int64_t words = ((int64_t)n + 63) / 64;
    // a wave takes 32 words of bits, one of blocks
    const int64_t w0 = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * 32;
    if (w0 >= words) return;
    uint32_t full = 0u;
#pragma unroll
    for (int r = 0; r < 32; r += kRows) {
        int32_t l[kRows];
#pragma unroll
        for (int i = 0; i < kRows; ++i) l[i] = L[min((w0 + r + i) * 64 + lane, (int64_t)n - 1)];
#pragma unroll
        for (int i = 0; i < kRows; ++i) {
            const unsigned long long b = __ballot(l[i] == label);
            if (lane == 0 && w0 + r + i < words) bits[w0 + r + i] = b;  // (bits past n are never read)
            full |= b == ~0ull ? 1u << (r + i) : 0u;
        }
    }
    if (lane == 0) blocks[w0 >> 5] = full;
}

// One 1,024-thread workgroup per CU holds in LDS the bits of the first
// fine * 32 vertices (on degree-sorted graphs the ones most edges name) and
// one bit per block of 64 for all of them, and streams its share of the
// edges, four per lane and load.  Only a vertex outside both, in a block that
// does not show D throughout, has its bit looked up in L2: such a lookup
// costs a line fill in L1 as its label did.  Converged step of R-MAT scale
// 25 (1.05G edges): every lookup in L2 5.4 ms a step; the first 1.05M
// vertices in LDS 1.58 ms for this pass, and with the blocks 0.94 (4.6 TB/s,
// what a copy reaches).
constexpr int kDomThreads = 1024;
constexpr int kDomLdsWords = 152 * 256;  // of 160 KB per CU
constexpr int kDomU = 2;  // loads in flight per lane (and as many of the next round)
// ALL: fine covers every vertex; else `nblocks` words of blocks follow (0:
// the graph has too many, every vertex past fine is looked up).
template <bool ALL>
__global__ __launch_bounds__(kDomThreads) void k_dominant_edges(const int32_t* __restrict__ nbr, int64_t m,
                                                                const uint32_t* __restrict__ bits,
                                                                const uint32_t* __restrict__ blocks, int32_t fine,
                                                                int32_t nblocks, const int32_t* __restrict__ ctl,
                                                                uint32_t* __restrict__ ebits) {
    if (ctl[0]) return;
    extern __shared__ __align__(16) uint32_t s_dyn[];
    for (int32_t i = threadIdx.x; i < fine; i += kDomThreads) s_dyn[i] = bits[i];
    if constexpr (!ALL) {
        // without blocks one word of zeros stands for them
        for (int32_t i = threadIdx.x; i < nblocks; i += kDomThreads) s_dyn[fine + i] = blocks[i];
        if (nblocks == 0 && threadIdx.x == 0) s_dyn[fine] = 0u;
    }
    __syncthreads();
    const int lane = lane_id();
    const uint32_t in_lds = (uint32_t)fine, last_block = (uint32_t)max(nblocks, 1) - 1u;
    const v4i32* nb4 = reinterpret_cast<const v4i32*>(nbr);
    const int64_t nvec = (m + 3) / 4;  // groups of four edges; the last may be short
    const int64_t stride = (int64_t)gridDim.x * kDomThreads;
    auto load = [&](int64_t i0, v4i32* u) {
#pragma unroll
        for (int k = 0; k < kDomU; ++k) {
            const int64_t i = i0 + k * stride + lane;
            if (i * 4 + 4 <= m) {
                u[k] = __builtin_nontemporal_load(&nb4[i]);
            } else {  // past the end, or the short group: its edges, then any vertex
                const int64_t j = min(i * 4, m - 1);
                u[k].x = nbr[j];
                u[k].y = nbr[min(j + 1, m - 1)];
                u[k].z = nbr[min(j + 2, m - 1)];
                u[k].w = nbr[min(j + 3, m - 1)];
            }
        }
    };
    // whole waves stay in the loop together (the words below join lanes)
    int64_t i0 = (int64_t)blockIdx.x * kDomThreads + (threadIdx.x & ~63);
    v4i32 u[kDomU];
    if (i0 < nvec) load(i0, u);
    while (i0 < nvec) {
        const int64_t i1 = i0 + stride * kDomU;
        v4i32 next[kDomU];
        if (i1 < nvec) load(i1, next);
        // all LDS lookups, then all L2 lookups (lanes that need none read
        // word 0 together), each issued before any is used
        uint32_t x[4 * kDomU];
#pragma unroll
        for (int k = 0; k < 4 * kDomU; ++k) {
            const uint32_t v = (uint32_t)u[k >> 2][k & 3], w = v >> 5;
            if constexpr (ALL) x[k] = s_dyn[w];
            else x[k] = s_dyn[w < in_lds ? w : in_lds + min(v >> 11, last_block)];
        }
#pragma unroll
        for (int k = 0; k < 4 * kDomU; ++k) {
            const uint32_t v = (uint32_t)u[k >> 2][k & 3];
            x[k] = (x[k] >> (ALL || (v >> 5) < in_lds ? v & 31u : (v >> 6) & 31u)) & 1u;
        }
        if constexpr (!ALL) {
            uint32_t y[4 * kDomU];
            uint32_t any = 0u;
#pragma unroll
            for (int k = 0; k < 4 * kDomU; ++k) {
                const uint32_t w = (uint32_t)u[k >> 2][k & 3] >> 5;
                y[k] = w >= in_lds && !x[k] ? w : 0u;  // (word 0 is in LDS)
                any |= y[k];
            }
            if (__ballot(any != 0u)) {  // wave-uniform
                uint32_t z[4 * kDomU];
#pragma unroll
                for (int k = 0; k < 4 * kDomU; ++k) z[k] = bits[y[k]];
#pragma unroll
                for (int k = 0; k < 4 * kDomU; ++k)
                    if (y[k]) x[k] = (z[k] >> (u[k >> 2][k & 3] & 31)) & 1u;
            }
        }
#pragma unroll
        for (int k = 0; k < kDomU; ++k) {
            // this lane's four bits in place, then joined over groups of
            // eight lanes (quad neighbours, quad pairs, half-row mirror)
            uint32_t z = (x[4 * k] | x[4 * k + 1] << 1 | x[4 * k + 2] << 2 | x[4 * k + 3] << 3) << (4 * (lane & 7));
            z |= (uint32_t)__builtin_amdgcn_update_dpp((int)z, (int)z, 0xB1, 0xf, 0xf, false);
            z |= (uint32_t)__builtin_amdgcn_update_dpp((int)z, (int)z, 0x4E, 0xf, 0xf, false);
            z |= (uint32_t)__builtin_amdgcn_update_dpp((int)z, (int)z, 0x141, 0xf, 0xf, false);
            const int64_t i = i0 + k * stride + lane;
            if ((lane & 7) == 0 && i < nvec) ebits[i >> 3] = z;  // (bits past m are never counted)
        }
#pragma unroll
        for (int k = 0; k < kDomU; ++k) u[k] = next[k];
        i0 = i1;
    }
}

// Set bits among bits [b, e) of ebits, `stride` threads cooperating, U words
// of each in flight (a word past the end is the last one again, not counted).
template <int U>
__device__ __forceinline__ uint32_t count_bits(const uint32_t* __restrict__ ebits, int32_t b, int32_t e, int tid,
                                               int stride) {
    uint32_t c = 0u;
    const int32_t w1 = (int32_t)(((uint32_t)e + 31u) >> 5);
    for (int32_t w0 = (b >> 5) + tid; w0 < w1; w0 += stride * U) {
        uint32_t x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) x[u] = ebits[min(w0 + u * stride, w1 - 1)];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int32_t w = w0 + u * stride;
            if (w == (b >> 5)) x[u] &= 0xffffffffu << (b & 31);
            if (w == (e >> 5)) x[u] &= (1u << (e & 31)) - 1u;  // (not met when e is a multiple of 32)
            c += w < w1 ? (uint32_t)__popc(x[u]) : 0u;
        }
    }
    return c;
}
// Workgroups [0, nhubs) take a hub each (degrees above hub_deg, which may be
// less than kDomLaneDeg); the others 1,024 vertices each, hubs left out, one
// lane per vertex up to kDomLaneDeg edges, 16 lanes above.
// Ids in degree order put 64 of the larger ones in one wave, which then is a
// chain of dependent reads: four of them at a time, several words of each in
// flight, instead of one after another by the whole wave.  R-MAT scale 25,
// converged: 217 us a step with a whole wave per larger vertex, 172 with rows
// of 16 lanes, 140 with four vertices per lane, 470 MB; an undecided step's
// launch, which only ends, 31 -> 11 us.
constexpr int32_t kDomLaneDeg = 256;
constexpr int kDomVerts = 4;  // vertices per lane, their offsets loaded together
__global__ __launch_bounds__(256) void k_dominant_decide(StepArgs a, const uint32_t* __restrict__ ebits,
                                                         const int32_t* __restrict__ hubs, int32_t nhubs,
                                                         int32_t hub_deg, uint8_t* __restrict__ act) {
    if (a.fctl[0]) return;
    const int32_t label = __builtin_amdgcn_readfirstlane(a.fctl[2]);
    const int lane = lane_id();
    // act of vertex v with d edges, c of them showing the label; true when
    // the vertex is decided and its label changes
    auto settle = [&](int32_t v, int32_t d, uint32_t c) {
        const bool won = 2u * c > (uint32_t)d;
        act[v] = d > 0 && !won ? 1 : 0;
        if (!won) return false;
        a.Lw[v] = label;
        return a.keep[v] != label;
    };
    if ((int32_t)blockIdx.x < nhubs) {
        __shared__ uint32_t s_c[4];
        bool changed = false;
        const int32_t v = hubs[blockIdx.x];
        const int32_t b = a.off[v], e = a.off[v + 1];
        const uint32_t c = wave_sum_u32(count_bits<2>(ebits, b, e, threadIdx.x, 256));
        if (lane == 0) s_c[threadIdx.x >> 6] = c;
        __syncthreads();
        if (threadIdx.x == 0) changed = settle(v, e - b, s_c[0] + s_c[1] + s_c[2] + s_c[3]);
        if (threadIdx.x < 64) count_changes(a, changed);
        return;
    }
    const int64_t vw = (int64_t)(blockIdx.x - (uint32_t)nhubs) * (256 * kDomVerts) + (threadIdx.x & ~63);
    int32_t vb[kDomVerts], ve[kDomVerts];
#pragma unroll
    for (int k = 0; k < kDomVerts; ++k) {
        const int64_t v = min(vw + k * 256 + lane, (int64_t)a.n - 1);
        vb[k] = a.off[v];
        ve[k] = a.off[v + 1];
    }
    uint32_t nch = 0u;
#pragma unroll
    for (int k = 0; k < kDomVerts; ++k) {
        const int64_t v0 = vw + k * 256, v = v0 + lane;
        const int32_t b = vb[k], e = ve[k];
        const bool small = v < a.n && e - b <= min(kDomLaneDeg, hub_deg);
        uint32_t c = 0u;
        if (__ballot(small && e - b > 64) != 0ull) c = small ? count_bits<4>(ebits, b, e, 0, 1) : 0u;
        else if (small) c = count_bits<1>(ebits, b, e, 0, 1);
        bool changed = small && settle((int32_t)v, e - b, c);
        nch += (uint32_t)__popcll(__ballot(changed));
        unsigned long long q = __ballot(v < a.n && e - b > kDomLaneDeg && e - b <= hub_deg);
        while (q) {  // wave-uniform: the next four, a row of 16 lanes each
            int src = -1;
#pragma unroll
            for (int row = 0; row < 4; ++row) {
                if (lane >> 4 == row && q) src = (int)__builtin_ctzll(q);
                q &= q - 1ull;  // (0 stays 0)
            }
            const int32_t sb = shfl_i32(b, max(src, 0)), se = shfl_i32(e, max(src, 0));
            const int32_t rb = src < 0 ? 0 : sb, re = src < 0 ? 0 : se;  // no vertex: no words
            c = group_sum_u32<16>(count_bits<4>(ebits, rb, re, lane & 15, 16));
            changed = src >= 0 && (lane & 15) == 0 && settle((int32_t)(v0 + src), re - rb, c);
            nch += (uint32_t)__popcll(__ballot(changed));
        }
    }
    add_changes(a, nch);
}

void init_kernels() {
    static bool done = false;
    if (done) return;
    done = true;
    init_counting_kernels();
    init_tiers_classic();
    init_tiers_layered();
    init_tiers_layered_vol();
    init_tiers_slpa();
    init_tiers_user();
    init_tiers_seeded();
    init_tiers_first();
    init_tiers_multi();
    set_lds_limit((const void*)k_dominant_edges<true>);
    set_lds_limit((const void*)k_dominant_edges<false>);
    (void)hipGetLastError();
}

int launch_step(Method method, bool weighted, bool gathered, const DeviceGraph& g,
                const HubScratch& hs, const StepArgs& a, hipStream_t s, hipEvent_t* ev) {
    switch (method) {
        case Method::Classic: return launch_tiers_classic(weighted, gathered, g, hs, a, s, ev);
        case Method::First:
            if (gathered) return set_error(GLP_E_UNSUPPORTED, "first steps read the neighbour ids themselves");
            return launch_tiers_first(weighted, g, hs, a, s, ev);
        case Method::Layered: return launch_tiers_layered(weighted, gathered, g, hs, a, s, ev);
        case Method::LayeredVol:
            if (gathered || !a.LV)
                return set_error(GLP_E_UNSUPPORTED, "slot-scored layered steps need the (label, volume) records");
            return launch_tiers_layered_vol(weighted, g, hs, a, s, ev);
        case Method::Slpa: return launch_tiers_slpa(weighted, gathered, g, hs, a, s, ev);
        case Method::User: return launch_tiers_user(weighted, gathered, g, hs, a, s, ev);
        case Method::Seeded: return launch_tiers_seeded(weighted, gathered, g, hs, a, s, ev);
    }
    return set_error(GLP_E_ARG, "unknown method");
}

int launch_pick(Method method, const StepArgs& a, int32_t* shown, hipStream_t s) {
    const unsigned grid = grid_for(a.n, 256);
    switch (method) {
        case Method::Slpa:
            hipLaunchKernelGGL(k_pick<SlpaHooks>, dim3(grid), dim3(256), 0, s, a, shown);
            break;
        case Method::User:
            hipLaunchKernelGGL(k_pick<UserHooks>, dim3(grid), dim3(256), 0, s, a, shown);
            break;
        default:
            return set_error(GLP_E_ARG, "method has no pick kernel");
    }
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? GLP_OK : set_error(GLP_E_HIP, "pick launch: %s", hipGetErrorString(e));
}

int launch_gather(const StepArgs& a, int64_t m, int32_t* adj, hipStream_t s) {
    if (m == 0) return GLP_OK;
    const unsigned grid = (unsigned)std::min<int64_t>(grid_for(m / 4 + 1, 256), 256 * 64);
    hipLaunchKernelGGL(k_gather, dim3(grid), dim3(256), 0, s, a.nbr, a.L, adj, m);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? GLP_OK : set_error(GLP_E_HIP, "gather launch: %s", hipGetErrorString(e));
}

int launch_frontier_gather(const StepArgs& a, int64_t m, int32_t* adj, const InverseIndex& inv,
                           void* push, hipStream_t s) {
    if (m == 0) return GLP_OK;
    if (!a.chg_r || !a.fctl || !inv.off || !inv.pos || !push)
        return set_error(GLP_E_STATE, "frontier gather without its inverse index");
    const int64_t nwords = ((int64_t)a.n + 31) / 32;
    const int64_t nblocks = (nwords + 255) / 256;
    auto* psum = static_cast<int2*>(push);
    auto* ent = reinterpret_cast<PushEntry*>(psum + ((nblocks + 1) & ~(int64_t)1));
    int32_t* fctl = const_cast<int32_t*>(a.fctl);
    const int32_t need = a.lookahead ? 2 : 1;
    hipLaunchKernelGGL(k_push_count, dim3((unsigned)nblocks), dim3(256), 0, s, a.chg_r, nwords, inv.off,
                       psum, a.fctl, need);
    hipLaunchKernelGGL(k_push_scan, dim3(1), dim3(256), 0, s, psum, nblocks, fctl, need);
    hipLaunchKernelGGL(k_push_write, dim3((unsigned)nblocks), dim3(256), 0, s, a.chg_r, nwords, inv.off,
                       a.L, psum, ent, a.fctl, need);
    const unsigned grid = (unsigned)std::min<int64_t>(grid_for(m / 4 + 1, 256), 256 * 64);
    hipLaunchKernelGGL(k_gather_frontier, dim3(grid), dim3(256), 0, s, a.nbr, a.L, adj, m, inv.pos,
                       ent, a.fctl, need);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? GLP_OK : set_error(GLP_E_HIP, "gather launch: %s", hipGetErrorString(e));
}

int32_t push_edge_limit(int64_t m) {
    return (int32_t)std::min<int64_t>(m / kPushRatio, INT32_MAX);
}

size_t push_entry_bytes(int32_t n, int64_t m) {
    // per-workgroup sums (int2, padded to 16 bytes), then the entries
    const size_t nblocks = ((size_t)n / 32 + 1 + 255) / 256;
    return 8 * ((nblocks + 1) & ~(size_t)1) + sizeof(PushEntry) * ((size_t)n + (size_t)(m / kPushChunk) + 64);
}

int inverse_index_build(const int32_t* nbr, int32_t n, int64_t m, int32_t* cursor, InverseIndex& inv,
                        hipStream_t s) {
    // counts into inv.off[0..n], exclusive scan, then the fill (cursor = copy
    // of the offsets; n + 1 int32 of caller scratch)
    const int64_t cnt = (int64_t)n + 1;
    const int64_t nsums = (cnt + kScanBlock - 1) / kScanBlock;
    int32_t* sums = nullptr;
    GLP_HIP(hipMalloc(&sums, (size_t)nsums * 4));
    int rc = launch_fill_i32(inv.off, 0, cnt, s);
    const unsigned grid = (unsigned)std::min<int64_t>(grid_for(m, 256), 256 * 64);
    if (!rc && m > 0) hipLaunchKernelGGL(k_inv_count, dim3(grid), dim3(256), 0, s, nbr, m, inv.off);
    if (!rc) {
        hipLaunchKernelGGL(k_scan_sums, dim3((unsigned)nsums), dim3(256), 0, s, inv.off, cnt, sums);
        hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(256), 0, s, sums, nsums);
        hipLaunchKernelGGL(k_scan_apply, dim3((unsigned)nsums), dim3(256), 0, s, inv.off, cnt, sums);
        hipError_t e = hipMemcpyAsync(cursor, inv.off, (size_t)cnt * 4, hipMemcpyDeviceToDevice, s);
        if (e != hipSuccess) rc = set_error(GLP_E_HIP, "inverse index: %s", hipGetErrorString(e));
    }
    if (!rc && m > 0) hipLaunchKernelGGL(k_inv_fill, dim3(grid), dim3(256), 0, s, nbr, m, cursor, inv.pos);
    if (!rc) {
        hipError_t e = hipGetLastError();
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e != hipSuccess) rc = set_error(GLP_E_HIP, "inverse index: %s", hipGetErrorString(e));
    }
    (void)hipFree(sums);
    return rc;
}

int launch_volume_init(const int32_t* off, const int32_t* L, int32_t* V, int32_t n, hipStream_t s) {
    if (n <= 0) return GLP_OK;
    hipLaunchKernelGGL(k_volume_init, dim3((unsigned)std::min<int64_t>(grid_for(n, 256), 256 * 64)), dim3(256), 0, s,
                       off, L, V, n);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? GLP_OK : set_error(GLP_E_HIP, "volume launch: %s", hipGetErrorString(e));
}

int launch_volume(const int32_t* off, const int32_t* L, int32_t* V, int32_t n, hipStream_t s) {
    if (n <= 0) return GLP_OK;
    hipLaunchKernelGGL(k_volume, dim3(grid_for(n, kVolChunk)), dim3(kVolThreads), 0, s, off, L, V, n);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? GLP_OK : set_error(GLP_E_HIP, "volume launch: %s", hipGetErrorString(e));
}

int launch_fill_i32(int32_t* p, int32_t value, int64_t count, hipStream_t s) {
    if (count <= 0) return GLP_OK;
    const unsigned grid = (unsigned)std::min<int64_t>(grid_for(count, 256), 256 * 32);
    hipLaunchKernelGGL(k_fill_i32, dim3(grid), dim3(256), 0, s, p, value, count);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? GLP_OK : set_error(GLP_E_HIP, "fill launch: %s", hipGetErrorString(e));
}

int launch_label_volumes(const int32_t* off, const int32_t* L, const int32_t* Vr, int2* LV, int32_t* Vw, int32_t n,
                         hipStream_t s) {
    if (n <= 0) return GLP_OK;
    const unsigned grid = (unsigned)std::min<int64_t>(grid_for(n, 256), 256 * 64);
    hipLaunchKernelGGL(k_label_volumes, dim3(grid), dim3(256), 0, s, off, L, Vr, LV, Vw, n);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? GLP_OK : set_error(GLP_E_HIP, "label-volume launch: %s", hipGetErrorString(e));
}

int launch_iota(int32_t* p, int64_t count, hipStream_t s) {
    if (count <= 0) return GLP_OK;
    const unsigned grid = (unsigned)std::min<int64_t>(grid_for(count, 256), 256 * 32);
    hipLaunchKernelGGL(k_iota, dim3(grid), dim3(256), 0, s, p, count);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? GLP_OK : set_error(GLP_E_HIP, "iota launch: %s", hipGetErrorString(e));
}

// Whether every neighbour list is strictly ascending: the positions j with
// nbr[j] >= nbr[j + 1] (out[0]) must all be the last of their list (out[1]
// counts those).  Two streaming passes, once per graph.
__global__ __launch_bounds__(256) void k_descents(const int32_t* __restrict__ off, const int32_t* __restrict__ nbr,
                                                  int32_t n, int64_t m, unsigned long long* __restrict__ out) {
    const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    uint32_t all = 0u, ends = 0u;
    for (int64_t j = t0; j + 1 < m; j += stride) all += nbr[j] >= nbr[j + 1] ? 1u : 0u;
    for (int64_t v = t0; v < n; v += stride) {
        const int64_t e = off[v + 1];
        if (e > off[v] && e < m) ends += nbr[e - 1] >= nbr[e] ? 1u : 0u;
    }
    all = wave_sum_u32(all);
    ends = wave_sum_u32(ends);
    if (lane_id() == 0) {
        if (all) atomicAdd(&out[0], (unsigned long long)all);
        if (ends) atomicAdd(&out[1], (unsigned long long)ends);
    }
}

int neighbours_ascending(const int32_t* off, const int32_t* nbr, int32_t n, int64_t m, hipStream_t s,
                         unsigned long long* scratch, bool* yes) {
    *yes = true;
    if (m < 2) return GLP_OK;
    unsigned long long got[2] = {0, 0};
    const int rc = launch_zero_bytes(scratch, sizeof got, s);
    if (rc != GLP_OK) return rc;
    const unsigned grid = (unsigned)std::min<int64_t>(grid_for(m, 256), 256 * 32);
    hipLaunchKernelGGL(k_descents, dim3(grid), dim3(256), 0, s, off, nbr, n, m, scratch);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(got, scratch, sizeof got, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return set_error(GLP_E_HIP, "neighbour order check: %s", hipGetErrorString(e));
    *yes = got[0] == got[1];
    return GLP_OK;
}

// Random 4-byte reads of a table with uniform fmix32 indices (the label
// gather's access pattern without its CSR stream): four independent reads
// per lane per round, summed so the loads are kept.
__global__ __launch_bounds__(256) void k_calib_read(const int32_t* __restrict__ T, uint32_t mask,
                                                    int64_t reads, uint32_t seed,
                                                    int32_t* __restrict__ out) {
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    int32_t acc = 0;
    for (int64_t j = tid * 4; j < reads; j += stride * 4) {
        const uint32_t b = (uint32_t)j ^ seed;
        acc += T[fmix32(b) & mask] + T[fmix32(b + 1u) & mask] + T[fmix32(b + 2u) & mask] +
               T[fmix32(b + 3u) & mask];
    }
    out[tid] = acc;
}

int launch_calib_read(const int32_t* T, int64_t entries, int64_t reads, uint32_t seed, int32_t* out,
                      int64_t out_entries, hipStream_t s) {
    if (entries <= 0 || (entries & (entries - 1)) || entries > (int64_t)1 << 31)
        return set_error(GLP_E_ARG, "table entries must be a power of two <= 2^31");
    const int64_t grid = std::min<int64_t>(256 * 32, out_entries / 256);
    if (grid < 1) return set_error(GLP_E_ARG, "calibration output too small");
    hipLaunchKernelGGL(k_calib_read, dim3((unsigned)grid), dim3(256), 0, s, T, (uint32_t)(entries - 1),
                       reads, seed, out);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? GLP_OK : set_error(GLP_E_HIP, "calibration launch: %s", hipGetErrorString(e));
}

int launch_dominant(const DeviceGraph& g, const StepArgs& a, uint32_t* bits, uint32_t* ebits, uint8_t* act,
                    hipStream_t s) {
    if (g.n <= 0 || g.m <= 0) return GLP_OK;
    const int64_t words = ((int64_t)g.n + 31) / 32;
    uint32_t* blocks = bits + dominant_bytes(g.n) / 4;
    hipLaunchKernelGGL(k_dominant_bits, dim3(grid_for(g.n, 4 * 2048)), dim3(256), 0, s, a.L, g.n, a.fctl,
                       reinterpret_cast<unsigned long long*>(bits), blocks);
    static const int64_t resident = resident_blocks((const void*)k_dominant_edges<false>, kDomThreads, kDomLdsWords * 4);
    const dim3 grid((unsigned)std::min<int64_t>(grid_for(g.m, 4 * kDomThreads), resident));
    if (words <= kDomLdsWords) {
        hipLaunchKernelGGL((k_dominant_edges<true>), grid, dim3(kDomThreads), (size_t)words * 4, s, a.nbr, g.m, bits,
                           blocks, (int32_t)words, 0, a.fctl, ebits);
    } else {
        // blocks take at most half of LDS (up to 38M vertices)
        int32_t nblocks = (int32_t)((words + 63) / 64);
        if (nblocks > kDomLdsWords / 2) nblocks = 0;
        const int32_t fine = kDomLdsWords - std::max(nblocks, 1);
        hipLaunchKernelGGL((k_dominant_edges<false>), grid, dim3(kDomThreads), (size_t)kDomLdsWords * 4, s, a.nbr, g.m,
                           bits, blocks, fine, nblocks, a.fctl, ebits);
    }
    const int32_t nh = (int32_t)g.plan.hubs.size();
    hipLaunchKernelGGL(k_dominant_decide, dim3((unsigned)nh + grid_for(g.n, 256 * kDomVerts)), dim3(256), 0, s, a, ebits, g.d_hubs,
                       nh, nh ? g.plan.tune.block_max_deg : INT32_MAX, act);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? GLP_OK : set_error(GLP_E_HIP, "dominant label launch: %s", hipGetErrorString(e));
}

int launch_end_steps(unsigned long long* acc, int32_t rows, unsigned long long* ring, int32_t* step_ctr,
                     int32_t ring_size, hipStream_t s) {
    if (rows <= 0) return GLP_OK;
    hipLaunchKernelGGL(k_end_steps, dim3(1), dim3(1024), 0, s, acc, rows, ring, step_ctr, ring_size);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? GLP_OK : set_error(GLP_E_HIP, "end_steps launch: %s", hipGetErrorString(e));
}

int launch_reset(const ResetArgs& r, hipStream_t s) {
    int64_t work = r.n;
    for (int k = 0; k < 7; ++k) work = std::max(work, r.zero[k] ? r.zero_words[k] : 0);
    hipLaunchKernelGGL(k_reset, dim3((unsigned)std::min<int64_t>(grid_for(work, 256), 256 * 32)), dim3(256), 0, s, r);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? GLP_OK : set_error(GLP_E_HIP, "reset launch: %s", hipGetErrorString(e));
}

int launch_end_step(unsigned long long* acc, unsigned long long* ring, int32_t* step_ctr,
                    int32_t ring_size, hipStream_t s, int32_t* fctl, const int32_t* dom_nbr, const int32_t* dom_L,
                    int64_t dom_m, int32_t* dom_ctl) {
    hipLaunchKernelGGL(k_end_step, dim3(1), dim3(kChangeSlots), 0, s, acc, ring, step_ctr, ring_size,
                       fctl, DominantSample{dom_nbr, dom_L, dom_m, dom_ctl});
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? GLP_OK : set_error(GLP_E_HIP, "end_step launch: %s", hipGetErrorString(e));
}

}  // namespace glp
