// Wave64 / LDS primitives for gfx950 (CDNA4); a wavefront is 64 lanes.
// Shuffles to any lane go through ds_bpermute, reductions and scans over DPP
// moves and readlanes.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace glp {
namespace dev {

constexpr int kWave = 64;

__device__ __forceinline__ int lane_id() { return __lane_id(); }

__device__ __forceinline__ uint32_t shfl_u32(uint32_t x, int src) {
    return (uint32_t)__builtin_amdgcn_ds_bpermute(src << 2, (int)x);
}
__device__ __forceinline__ int32_t shfl_i32(int32_t x, int src) {
    return __builtin_amdgcn_ds_bpermute(src << 2, x);
}
__device__ __forceinline__ uint64_t shfl_u64(uint64_t x, int src) {
    uint32_t lo = shfl_u32((uint32_t)x, src);
    uint32_t hi = shfl_u32((uint32_t)(x >> 32), src);
    return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ uint64_t max_u64(uint64_t a, uint64_t b) { return a > b ? a : b; }

// Load of data read once per step (CSR neighbours, weights, gathered
// labels): marked nontemporal so it does not evict the label lines that the
// random gathers keep reusing from L2.
template <class T>
__device__ __forceinline__ T ld_stream(const T* p) {
    return __builtin_nontemporal_load(p);
}

// How many of the lanes below this one m holds.
__device__ __forceinline__ int32_t lanes_below(uint64_t m) {
    return (int32_t)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Reductions over the 64 lanes, every lane active; every lane receives the
// result.  DPP moves combine each row of 16 (quad pairs, quad with mirror
// quad, half-row with half-row), readlanes the four rows: about 15 vector and
// scalar instructions, where a shuffle tree waits for the LDS pipe six times
// (twelve for 64 bits).  (A lane whose DPP source is unavailable keeps its
// own value: old = x.)
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)x, (int)x, CTRL, 0xf, 0xf, false);
}
template <class F>
__device__ __forceinline__ uint32_t row_reduce(uint32_t x, F f) {  // over each row of 16 lanes
    x = f(x, dpp_u32<0xB1>(x));   // quad_perm [1,0,3,2]
    x = f(x, dpp_u32<0x4E>(x));   // quad_perm [2,3,0,1]
    x = f(x, dpp_u32<0x141>(x));  // row half-mirror
    return f(x, dpp_u32<0x140>(x));  // row mirror
}
template <class F>
__device__ __forceinline__ uint32_t wave_reduce(uint32_t x, F f) {
    x = row_reduce(x, f);
    const uint32_t r0 = (uint32_t)__builtin_amdgcn_readlane((int)x, 0);
    const uint32_t r1 = (uint32_t)__builtin_amdgcn_readlane((int)x, 16);
    const uint32_t r2 = (uint32_t)__builtin_amdgcn_readlane((int)x, 32);
    const uint32_t r3 = (uint32_t)__builtin_amdgcn_readlane((int)x, 48);
    return f(f(r0, r1), f(r2, r3));
}
__device__ __forceinline__ uint32_t wave_min_u32(uint32_t x) {
    return wave_reduce(x, [](uint32_t a, uint32_t b) { return min(a, b); });
}
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t x) {
    return wave_reduce(x, [](uint32_t a, uint32_t b) { return max(a, b); });
}
__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t x) {
    return wave_reduce(x, [](uint32_t a, uint32_t b) { return a + b; });
}
__device__ __forceinline__ uint64_t wave_max_u64(uint64_t x) {
    const uint32_t hi = wave_max_u32((uint32_t)(x >> 32));
    const uint32_t lo = wave_max_u32((uint32_t)(x >> 32) == hi ? (uint32_t)x : 0u);
    return ((uint64_t)hi << 32) | lo;
}
// The same over each group of S = 16 or 32 consecutive lanes (two rows meet
// through one shuffle).
template <int S, class F>
__device__ __forceinline__ uint32_t group_reduce(uint32_t x, F f) {
    static_assert(S == 16 || S == 32, "one row or two");
    x = row_reduce(x, f);
    if (S == 32) x = f(x, shfl_u32(x, lane_id() ^ 16));
    return x;
}
template <int S>
__device__ __forceinline__ uint32_t group_sum_u32(uint32_t x) {
    return group_reduce<S>(x, [](uint32_t a, uint32_t b) { return a + b; });
}
template <int S>
__device__ __forceinline__ uint64_t group_max_u64(uint64_t x) {
    auto mx = [](uint32_t a, uint32_t b) { return max(a, b); };
    const uint32_t hi = group_reduce<S>((uint32_t)(x >> 32), mx);
    const uint32_t lo = group_reduce<S>((uint32_t)(x >> 32) == hi ? (uint32_t)x : 0u, mx);
    return ((uint64_t)hi << 32) | lo;
}
// The group's lane I to all of its lanes.
template <int S, int I>
__device__ __forceinline__ uint32_t group_lane(uint32_t x) {
    if constexpr (S == 16) return dpp_u32<0x150 + I>(x);  // row_newbcast:I
    else return shfl_u32(x, (lane_id() & ~(S - 1)) + I);
}
// Inclusive prefix sum over the 64 lanes, every lane active: within rows by
// row shifts (a lane without a source adds 0), then each row's last lane into
// the next row, and lane 31 into the upper half.
__device__ __forceinline__ int32_t wave_incl_sum(int32_t x) {
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);  // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);  // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);  // row_shr:8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
    return x;
}

// Orders LDS traffic of one wavefront: LDS serves one wave's requests in
// issue order, so a compiler-level barrier is all that is needed between a
// lane's store and another lane's load in the same wave.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// murmur3 fmix32 finaliser; the slot hash of the LDS and HBM tables (the
// reference's GlobalHT uses the same finaliser, method/hashtable.cuh:19-26).
__device__ __forceinline__ uint32_t fmix32(uint32_t k) {
    k ^= k >> 16;
    k *= 0x85ebca6bu;
    k ^= k >> 13;
    k *= 0xc2b2ae35u;
    k ^= k >> 16;
    return k;
}

__host__ __device__ __forceinline__ uint32_t next_pow2(uint32_t x) {
    if (x <= 1) return 1;
    return 1u << (32 - __builtin_clz(x - 1));
}

}  // namespace dev
}  // namespace glp
