// dg_box_kernels.hip -- the DG stage kernels of dg_stage.h on Cartesian elements.
#include "dg_stage.h"

namespace nmx {

hipError_t launch_dg_box(int np, int nmax, const AmrArgs &a, hipStream_t s) {
  return launch_dg_geom<0>(np, nmax, a, s);
}

}  // namespace nmx
