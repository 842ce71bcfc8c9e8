// The tier kernels of classic LP.

#include "tiers.h"

namespace glp {

int launch_tiers_classic(bool weighted, bool gathered, const DeviceGraph& g, const HubScratch& hs, const StepArgs& a,
                 hipStream_t s, hipEvent_t* ev) {
    return launch_hooks<ClassicHooks>(weighted, gathered, g, hs, a, s, ev);
}
void init_tiers_classic() { set_tier_limits<ClassicHooks, true>(); }

}  // namespace glp
