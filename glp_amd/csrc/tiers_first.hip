// The tier kernels of first steps.

#include "tiers.h"

namespace glp {

// (fused gather only)
int launch_tiers_first(bool weighted, const DeviceGraph& g, const HubScratch& hs, const StepArgs& a, hipStream_t s,
                 hipEvent_t* ev) {
    return weighted ? launch_tiers<FirstHooks, true, false>(g, hs, a, s, ev)
                    : launch_tiers<FirstHooks, false, false>(g, hs, a, s, ev);
}
void init_tiers_first() { set_tier_limits<FirstHooks, false>(); }

}  // namespace glp
