// Instances of the FP32 filter kernel.
#define BLAMM_INSTANTIATE
#include "instances.hpp"

namespace blamm {
#define BLAMM_DEF_FP32(M, L) template __global__ void filter_fp32_kernel<M, L>(FilterArgs, WorkQueue, ListArgs);
BLAMM_SCAN_INSTANCES(BLAMM_DEF_FP32)
}  // namespace blamm
