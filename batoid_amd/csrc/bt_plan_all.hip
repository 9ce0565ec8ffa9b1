// bt_plan_all.hip -- the plan kernel for the kind set kKindsAll.
#include <hip/hip_runtime.h>

#include "bt_plan.h"

namespace bt {

void launch_plan_all(int mode, dim3 grid, hipStream_t st, const bt_plan& plan,
                  const bt_rays& in, const bt_rays& out, int niter, int need_w)
{
    launch_plan_kinds<kKindsAll>(mode, grid, st, plan, in, out, niter, need_w);
}

}  // namespace bt
