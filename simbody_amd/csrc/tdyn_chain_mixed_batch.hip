// Chain-evaluator rollout kernels: one model per batch, mixed precision.
#include "tdyn_rkm_chain.hpp"

namespace tdyn {

hipError_t launch_chain_mixed_batch(const RkmArgs& a, hipStream_t s, bool f0_only) {
    // (the derivative alone has one build, the general one: it agrees to rounding)
    if (a.idf && !f0_only) return launch_chain_t<chain::IdF<cdptr>, float>(a, s, false);
    return launch_chain_t<cdptr, float>(a, s, f0_only);
}

} // namespace tdyn
