// The filter and histogram kernels are compiled in translation units of their
// own (screen.hip, filter_fp32.hip, hist_filter.hip, hist_filter_hbm.hip) so that
// the library builds in parallel and a process loads only the code of the units
// it calls (about 2 ms per MB); the launching code sees these declarations and
// leaves the instantiation to those units.
#pragma once

#include "scan_kernels.hpp"
#include "hist_kernels.hpp"
#include "screen_kernels.hpp"

namespace blamm {

// (lowercase mask, list form)
#define BLAMM_SCAN_INSTANCES(X) X(false, false) X(false, true) X(true, false) X(true, true)
// (mask, LDS histograms, motifs longer than 32 positions)
#define BLAMM_HIST_LDS_INSTANCES(X) X(false, true, false) X(true, true, false) X(false, true, true) X(true, true, true)
#define BLAMM_HIST_HBM_INSTANCES(X) X(false, false, false) X(true, false, false) X(false, false, true) X(true, false, true)

#ifndef BLAMM_INSTANTIATE
#define BLAMM_EXTERN_SCREEN(M, L) extern template __global__ void screen_kernel<M, L, false>(ScreenArgs, WorkQueue, ListArgs);
#define BLAMM_EXTERN_FP32(M, L) extern template __global__ void filter_fp32_kernel<M, L>(FilterArgs, WorkQueue, ListArgs);
#define BLAMM_EXTERN_LO(M, L) extern template __global__ void screen_kernel<M, L, true>(ScreenArgs, WorkQueue, ListArgs);
#define BLAMM_EXTERN_HIST(M, L, W) extern template __global__ void hist_filter_kernel<M, L, W>(HistArgs);
BLAMM_SCAN_INSTANCES(BLAMM_EXTERN_SCREEN)
BLAMM_SCAN_INSTANCES(BLAMM_EXTERN_FP32)
BLAMM_SCAN_INSTANCES(BLAMM_EXTERN_LO)
BLAMM_HIST_LDS_INSTANCES(BLAMM_EXTERN_HIST)
BLAMM_HIST_HBM_INSTANCES(BLAMM_EXTERN_HIST)
#undef BLAMM_EXTERN_SCREEN
#undef BLAMM_EXTERN_FP32
#undef BLAMM_EXTERN_LO
#undef BLAMM_EXTERN_HIST
#endif

}  // namespace blamm
