// Instances of the screen kernel (default and split-BF16 form).
#define BLAMM_INSTANTIATE
#include "instances.hpp"

namespace blamm {
#define BLAMM_DEF_SCREEN(M, L) template __global__ void screen_kernel<M, L, false>(ScreenArgs, WorkQueue, ListArgs);
#define BLAMM_DEF_LO(M, L) template __global__ void screen_kernel<M, L, true>(ScreenArgs, WorkQueue, ListArgs);
BLAMM_SCAN_INSTANCES(BLAMM_DEF_SCREEN)
BLAMM_SCAN_INSTANCES(BLAMM_DEF_LO)
}  // namespace blamm
