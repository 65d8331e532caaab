// spx_few_f32.hip -- the FP32 step kernels for few resident waves (V = 1): the Parker family on the solar wind and the
// Cartesian grid.
//
// Same results as the kernels of spx_kernels_f32.hip, built with the same flags.  Not built for what gains nothing
// (the shocks and the uniform background have no stencil to split: 9% slower on the smooth shock) nor for the guiding
// centre: this unit contracts multiply-adds across statements, so the quad's straight-line sums of that stencil
// round differently from the loop's.
#include "spx_parker.h"

namespace spx {

hipError_t launch_few_f32(const spx_plan_desc& hp, const LaunchShape& S, const Launch* d_launch, hipStream_t st)
{
   switch (hp.bg.kind) {
   case SPX_BG_GRID: return dispatch_grid<float, LAUNCH_FEW>(hp, S, d_launch, st, nullptr);
   case SPX_BG_SOLARWIND: return dispatch_flow<float, SPX_BG_SOLARWIND, LAUNCH_FEW>(hp, S, d_launch, st, nullptr);
   default: return hipErrorInvalidValue;
   }
}

}  // namespace spx
