// bt_plan_sum_apb.hip -- the plan kernel for the kind set kKindsSumAPB.
#include <hip/hip_runtime.h>

#include "bt_plan.h"

namespace bt {

void launch_plan_sum_apb(int mode, dim3 grid, hipStream_t st, const bt_plan& plan,
                  const bt_rays& in, const bt_rays& out, int niter, int need_w)
{
    launch_plan_kinds<kKindsSumAPB>(mode, grid, st, plan, in, out, niter, need_w);
}

}  // namespace bt
