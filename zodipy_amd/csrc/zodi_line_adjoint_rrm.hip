// The line adjoint and Jacobian kernels of the RRM layouts.

#include <hip/hip_runtime.h>

#include "zodi_line_rrm.hpp"

namespace zodi {

AdjKernel line_adjoint_rrm(bool split_layout, bool jac) {
  if (split_layout)
    return jac ? rrm_adjoint<LayoutRRMSplit, true> : rrm_adjoint<LayoutRRMSplit, false>;
  return jac ? rrm_adjoint<LayoutRRM, true> : rrm_adjoint<LayoutRRM, false>;
}

}  // namespace zodi
