// The tier kernels of seeded LP.

#include "tiers.h"

namespace glp {

int launch_tiers_seeded(bool weighted, bool gathered, const DeviceGraph& g, const HubScratch& hs, const StepArgs& a,
                 hipStream_t s, hipEvent_t* ev) {
    return launch_hooks<SeededHooks>(weighted, gathered, g, hs, a, s, ev);
}
void init_tiers_seeded() { set_tier_limits<SeededHooks, true>(); }

}  // namespace glp
