// Folded (multi-job) launches of the tier kernels: the serving path.

#include "tiers.h"

namespace glp {

template <class H, bool W, bool G, int L, int NT>
__global__ __launch_bounds__(NT) void k_multi(const JobDesc* __restrict__ jobs,
                                              const int32_t* __restrict__ cum, int32_t njobs,
                                              uint32_t cap_max) {
    const int32_t j = job_of(cum, njobs, blockIdx.x);
    const uint32_t blk = blockIdx.x - (uint32_t)cum[j];
    const JobDesc& jd = jobs[j];
    if constexpr (L == kLaunchPacked) {
        __shared__ PackedLds s_pk[4];
        packed_body<H, W, G, kFoldNG>(jd.a, jd.groups, jd.ngroups, jd.ngroups_e, wave_unit(blk),
                                      s_pk[threadIdx.x >> 6]);
    } else if constexpr (L == kLaunchHalf) {
        __shared__ HalfLds<32> s_half[4];
        half_body<H, W, G, kFoldNG>(jd.a, jd.half, jd.nhalf, wave_unit(blk), s_half[threadIdx.x >> 6]);
    } else if constexpr (L == kLaunchWave) {
        __shared__ unsigned long long s_tab[4][kWaveCap];
        wave_body<H, W, G>(jd.a, jd.wave, jd.nwave, wave_unit(blk), s_tab[threadIdx.x >> 6]);
    } else if constexpr (L >= kLaunchBlock0 && L < kLaunchBlock0 + kMaxBlockClasses) {
        block_body<H, W, G, NT>(jd.a, jd.block[L - kLaunchBlock0], cap_max, blk);
    } else if constexpr (L == kLaunchHubAgg) {
        hub_agg_body<H, W, G>(jd.a, jd.hub, blk);
    } else if constexpr (L == kLaunchHubPart) {
        hub_part_batch_body<H>(jd.a, jd.hub, blk);
    } else {
        hub_final_body<H>(jd.a, jd.hub, blk);
    }
}

// Folded launches of one step for `nj` jobs (the serving path).  cum holds
// kLaunches rows of nj+1 prefix sums; grid[L] = cum row L's last entry.
template <class H, bool W, int C>
static void launch_multi_block(const JobDesc* jobs, const int32_t* cum, int32_t nj,
                               const int32_t* grid, const Tuning& t, uint32_t cap, hipStream_t s) {
    constexpr int L = kLaunchBlock0 + C;
    if (!grid[L]) return;
    const size_t lds = (size_t)cap * 2 * sizeof(uint32_t);
    const int32_t* row = cum + (size_t)L * (nj + 1);
    if (t.block_threads == 1024)
        hipLaunchKernelGGL((k_multi<H, W, false, L, 1024>), dim3(grid[L]), dim3(1024), lds, s, jobs, row, nj, cap);
    else if (t.block_threads == 512)
        hipLaunchKernelGGL((k_multi<H, W, false, L, 512>), dim3(grid[L]), dim3(512), lds, s, jobs, row, nj, cap);
    else
        hipLaunchKernelGGL((k_multi<H, W, false, L, 256>), dim3(grid[L]), dim3(256), lds, s, jobs, row, nj, cap);
}

template <class H, bool W>
static int launch_multi_t(const JobDesc* jobs, const int32_t* cum, int32_t nj, const int32_t* grid,
                          const Tuning& t, const int32_t* class_cap, hipStream_t s) {
    auto row = [&](int L) { return cum + (size_t)L * (nj + 1); };
    if (grid[kLaunchPacked])
        hipLaunchKernelGGL((k_multi<H, W, false, kLaunchPacked, 256>), dim3(grid[kLaunchPacked]),
                           dim3(256), 0, s, jobs, row(kLaunchPacked), nj, 0u);
    if (grid[kLaunchHalf])
        hipLaunchKernelGGL((k_multi<H, W, false, kLaunchHalf, 256>), dim3(grid[kLaunchHalf]),
                           dim3(256), 0, s, jobs, row(kLaunchHalf), nj, 0u);
    if (grid[kLaunchWave])
        hipLaunchKernelGGL((k_multi<H, W, false, kLaunchWave, 256>), dim3(grid[kLaunchWave]),
                           dim3(256), 0, s, jobs, row(kLaunchWave), nj, 0u);
    launch_multi_block<H, W, 0>(jobs, cum, nj, grid, t, (uint32_t)class_cap[0], s);
    launch_multi_block<H, W, 1>(jobs, cum, nj, grid, t, (uint32_t)class_cap[1], s);
    launch_multi_block<H, W, 2>(jobs, cum, nj, grid, t, (uint32_t)class_cap[2], s);
    launch_multi_block<H, W, 3>(jobs, cum, nj, grid, t, (uint32_t)class_cap[3], s);
    launch_multi_block<H, W, 4>(jobs, cum, nj, grid, t, (uint32_t)class_cap[4], s);
    if (grid[kLaunchHubAgg]) {
        const size_t lds = hub_agg_lds(t.hub_chunk);
        hipLaunchKernelGGL((k_multi<H, W, false, kLaunchHubAgg, kHubThreads>), dim3(grid[kLaunchHubAgg]),
                           dim3(kHubThreads), lds, s, jobs, row(kLaunchHubAgg), nj, 0u);
    }
    if (grid[kLaunchHubPart]) {
        const size_t lds = (size_t)next_pow2(2u * (uint32_t)t.part_keys) * 2 * sizeof(uint32_t);
        hipLaunchKernelGGL((k_multi<H, W, false, kLaunchHubPart, kHubThreads>), dim3(grid[kLaunchHubPart]),
                           dim3(kHubThreads), lds, s, jobs, row(kLaunchHubPart), nj, 0u);
    }
    if (grid[kLaunchHubFinal])
        hipLaunchKernelGGL((k_multi<H, W, false, kLaunchHubFinal, 256>), dim3(grid[kLaunchHubFinal]),
                           dim3(256), 0, s, jobs, row(kLaunchHubFinal), nj, 0u);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? GLP_OK : set_error(GLP_E_HIP, "folded launch: %s", hipGetErrorString(e));
}

int launch_multi(bool weighted, bool slot_scores, const JobDesc* jobs, const int32_t* cum, int32_t nj,
                 const int32_t* grid, const Tuning& t, const int32_t* class_cap, hipStream_t s) {
    if (slot_scores) {
        if (weighted) return launch_multi_t<LayeredVolHooks, true>(jobs, cum, nj, grid, t, class_cap, s);
        return launch_multi_t<LayeredVolHooks, false>(jobs, cum, nj, grid, t, class_cap, s);
    }
    if (weighted) return launch_multi_t<LayeredHooks, true>(jobs, cum, nj, grid, t, class_cap, s);
    return launch_multi_t<LayeredHooks, false>(jobs, cum, nj, grid, t, class_cap, s);
}

// Workgroups each launch of a folded step needs for one job.
void job_blocks(const Plan& p, int32_t* blocks) {
    for (int L = 0; L < kLaunches; ++L) blocks[L] = 0;
    // folded jobs run the layered or slot-score hooks, which skip edge-less groups
    static_assert(LayeredHooks::kSkipIsolated && LayeredVolHooks::kSkipIsolated,
                  "folded launches run groups with edges only");
    blocks[kLaunchPacked] = (int32_t)((p.groups_with_edges + 4 * kFoldNG - 1) / (4 * kFoldNG));
    blocks[kLaunchHalf] = (int32_t)((p.half.size() + 8 * kFoldNG - 1) / (8 * kFoldNG));
    blocks[kLaunchWave] = (int32_t)((p.wave.size() + 4 * kWaveNV - 1) / (4 * kWaveNV));
    for (int c = 0; c < p.nclasses; ++c) blocks[kLaunchBlock0 + c] = (int32_t)p.block[c].size();
    blocks[kLaunchHubAgg] = (int32_t)p.hub_chunks.size();
    const int32_t pb = hub_part_batch((int64_t)p.hub_parts.size());
    blocks[kLaunchHubPart] = (int32_t)((p.hub_parts.size() + pb - 1) / pb);
    blocks[kLaunchHubFinal] = (int32_t)((p.hubs.size() + 255) / 256);
}

void init_tiers_multi() {
#define GLP_SETLDS_MULTI(W, L, NT)                                                              \
    set_lds_limit((const void*)k_multi<LayeredHooks, W, false, L, NT>);                          \
    set_lds_limit((const void*)k_multi<LayeredVolHooks, W, false, L, NT>);
#define GLP_SETLDS_MULTI_C(W, C) GLP_SETLDS_MULTI(W, kLaunchBlock0 + C, 256)                    \
    GLP_SETLDS_MULTI(W, kLaunchBlock0 + C, 512) GLP_SETLDS_MULTI(W, kLaunchBlock0 + C, 1024)
#define GLP_SETLDS_MULTI_W(W) GLP_SETLDS_MULTI_C(W, 0) GLP_SETLDS_MULTI_C(W, 1)                 \
    GLP_SETLDS_MULTI_C(W, 2) GLP_SETLDS_MULTI_C(W, 3) GLP_SETLDS_MULTI_C(W, 4)                   \
    GLP_SETLDS_MULTI(W, kLaunchHubAgg, kHubThreads) GLP_SETLDS_MULTI(W, kLaunchHubPart, kHubThreads)
    GLP_SETLDS_MULTI_W(false)
    GLP_SETLDS_MULTI_W(true)
#undef GLP_SETLDS_MULTI_W
#undef GLP_SETLDS_MULTI_C
#undef GLP_SETLDS_MULTI
}

}  // namespace glp
