// Instances of the split-BF16 filter kernel.
#define BLAMM_INSTANTIATE
#include "instances.hpp"

namespace blamm {
#define BLAMM_DEF_LO(M, L) template __global__ void filter_lo_kernel<M, L>(FilterArgs, WorkQueue, ListArgs);
BLAMM_SCAN_INSTANCES(BLAMM_DEF_LO)
}  // namespace blamm
