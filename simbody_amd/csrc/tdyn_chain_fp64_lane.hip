// Chain rollout kernels in joint frames: one model per lane (serving slots,
// whose number is a multiple of 64), FP64.
#include "tdyn_rkm_joint.hpp"

namespace tdyn {

hipError_t launch_chain_fp64_lane(const RkmArgs& a, hipStream_t s) {
    return a.kinds ? launch_joint_slots(a, s) : hipSuccess;
}

} // namespace tdyn
