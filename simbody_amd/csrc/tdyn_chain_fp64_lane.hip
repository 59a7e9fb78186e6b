// Chain rollout kernels in joint frames: one model per lane (serving slots,
// whose number is a multiple of 64), FP64.
#include "tdyn_rkm_joint.hpp"

namespace tdyn {

hipError_t launch_chain_fp64_lane(const RkmArgs& a, hipStream_t s, bool f0_only) {
    return a.jidf ? launch_joint_i<joint::PrmT, true, true>(a, s, f0_only)
                  : launch_joint_i<joint::PrmT, false, true>(a, s, f0_only);
}

} // namespace tdyn
