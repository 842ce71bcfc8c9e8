// The tier kernels of layered LP with gamma > 0, scored in the table slots.

#include "tiers.h"

namespace glp {

// (fused gather only)
int launch_tiers_layered_vol(bool weighted, const DeviceGraph& g, const HubScratch& hs, const StepArgs& a, hipStream_t s,
                 hipEvent_t* ev) {
    return weighted ? launch_tiers<LayeredVolHooks, true, false>(g, hs, a, s, ev)
                    : launch_tiers<LayeredVolHooks, false, false>(g, hs, a, s, ev);
}
void init_tiers_layered_vol() { set_tier_limits<LayeredVolHooks, false>(); }

}  // namespace glp
