// The tier kernels of SLPA.

#include "tiers.h"

namespace glp {

int launch_tiers_slpa(bool weighted, bool gathered, const DeviceGraph& g, const HubScratch& hs, const StepArgs& a,
                 hipStream_t s, hipEvent_t* ev) {
    return launch_hooks<SlpaHooks>(weighted, gathered, g, hs, a, s, ev);
}
void init_tiers_slpa() { set_tier_limits<SlpaHooks, true>(); }

}  // namespace glp
