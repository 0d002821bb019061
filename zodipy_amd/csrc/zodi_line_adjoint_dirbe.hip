// The line adjoint and Jacobian kernels of the DIRBE layout.

#include <hip/hip_runtime.h>

#include "zodi_line_adjoint.hpp"

namespace zodi {

AdjKernel line_adjoint_dirbe(int scat, int pass) { return pick_line_adjoint<LayoutDirbe>(scat, pass); }

}  // namespace zodi
