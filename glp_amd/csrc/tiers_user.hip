// The tier kernels of the user hooks.

#include "tiers.h"

namespace glp {

int launch_tiers_user(bool weighted, bool gathered, const DeviceGraph& g, const HubScratch& hs, const StepArgs& a,
                 hipStream_t s, hipEvent_t* ev) {
    return launch_hooks<UserHooks>(weighted, gathered, g, hs, a, s, ev);
}
void init_tiers_user() { set_tier_limits<UserHooks, true>(); }

}  // namespace glp
