// Instances of the screen kernel.
#define BLAMM_INSTANTIATE
#include "instances.hpp"

namespace blamm {
#define BLAMM_DEF_SCREEN(M, L) template __global__ void screen_kernel<M, L>(ScreenArgs, WorkQueue, ListArgs);
BLAMM_SCAN_INSTANCES(BLAMM_DEF_SCREEN)
}  // namespace blamm
