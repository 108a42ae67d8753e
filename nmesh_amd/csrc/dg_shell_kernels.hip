// dg_shell_kernels.hip -- the DG stage kernels of dg_stage.h on CubedShell elements, dX/dx recomputed.
#include "dg_stage.h"

namespace nmx {

hipError_t launch_dg_shell(int np, int nmax, const AmrArgs &a, hipStream_t s) {
  return launch_dg_geom<2>(np, nmax, a, s);
}

}  // namespace nmx
