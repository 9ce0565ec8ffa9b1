// bt_plan_flat_sums.hip -- the plan kernel for the kind set kKindsFlatSums.
#include <hip/hip_runtime.h>

#include "bt_plan.h"

namespace bt {

void launch_plan_flat_sums(int mode, dim3 grid, hipStream_t st, const bt_plan& plan,
                  const bt_rays& in, const bt_rays& out, int niter, int need_w)
{
    launch_plan_kinds<kKindsFlatSums>(mode, grid, st, plan, in, out, niter, need_w);
}

}  // namespace bt
