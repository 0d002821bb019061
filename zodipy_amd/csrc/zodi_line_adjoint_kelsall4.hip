// The line adjoint and Jacobian kernels of the four-component Kelsall layout.

#include <hip/hip_runtime.h>

#include "zodi_line_adjoint.hpp"

namespace zodi {

AdjKernel line_adjoint_kelsall4(int scat, int pass) { return pick_line_adjoint<LayoutKelsall4>(scat, pass); }

}  // namespace zodi
