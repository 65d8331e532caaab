// spx_few_f64.hip -- the FP64 step kernels for few resident waves (V = 1): the Parker and guiding-centre families.
//
// Same results, bit for bit, as the kernels of spx_kernels_f64.hip, built with the same flags.
#include "spx_parker.h"
#include "spx_gc.h"

namespace spx {

hipError_t launch_few_f64(const spx_plan_desc& hp, const LaunchShape& S, const Launch* d_launch, hipStream_t st)
{
   if (hp.traj_type >= SPX_TRAJ_GUIDING_DIFF_SCATT && hp.traj_type <= SPX_TRAJ_GUIDING_DIFF)
      return dispatch_gc<double, LAUNCH_FEW>(hp, S, d_launch, st, nullptr);
   return dispatch_parker<double, LAUNCH_FEW>(hp, S, d_launch, st, nullptr);
}

}  // namespace spx
