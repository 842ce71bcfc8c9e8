// The tier kernels of layered LP.

#include "tiers.h"

namespace glp {

int launch_tiers_layered(bool weighted, bool gathered, const DeviceGraph& g, const HubScratch& hs, const StepArgs& a,
                 hipStream_t s, hipEvent_t* ev) {
    return launch_hooks<LayeredHooks>(weighted, gathered, g, hs, a, s, ev);
}
void init_tiers_layered() { set_tier_limits<LayeredHooks, true>(); }

}  // namespace glp
