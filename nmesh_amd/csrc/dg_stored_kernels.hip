// dg_stored_kernels.hip -- the DG stage kernels of dg_stage.h on curvilinear elements whose dX/dx is read.
#include "dg_stage.h"

namespace nmx {

hipError_t launch_dg_stored(int np, int nmax, const AmrArgs &a, hipStream_t s) {
  return launch_dg_geom<1>(np, nmax, a, s);
}

}  // namespace nmx
