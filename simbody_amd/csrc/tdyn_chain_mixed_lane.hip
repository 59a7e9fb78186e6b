// Chain-evaluator rollout kernels: one model per lane, mixed precision.
#include "tdyn_rkm_chain.hpp"

namespace tdyn {

// A launch for each kind of slot that occurs (a slot of the other kind is
// skipped): the two builds round differently, and a request's must not depend
// on its neighbours.
hipError_t launch_chain_mixed_lane(const RkmArgs& a, hipStream_t s) {
    hipError_t e = hipSuccess;
    if (a.kinds & 1 << SK_IDF) e = launch_chain_t<chain::IdF<chain::PrmL>, float>(a, s, false);
    if (e == hipSuccess && (a.kinds & 1)) e = launch_chain_t<chain::PrmL, float>(a, s, false);
    return e;
}

} // namespace tdyn
