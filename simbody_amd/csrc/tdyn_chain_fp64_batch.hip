// Chain rollout kernels in joint frames: one model per batch, FP64.
#include "tdyn_rkm_joint.hpp"

namespace tdyn {

hipError_t launch_chain_fp64_batch(const RkmArgs& a, hipStream_t s, bool f0_only) {
    // (rows of one pitch: batches whose blocks would not fit, joint_tiles)
    if (!a.tile) return launch_joint_i<cdptr, false, false>(a, s, f0_only);
    return a.jidf ? launch_joint_i<cdptr, true, true>(a, s, f0_only) : launch_joint_i<cdptr, false, true>(a, s, f0_only);
}

} // namespace tdyn
