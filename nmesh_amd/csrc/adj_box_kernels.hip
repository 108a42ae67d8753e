// adj_box_kernels.hip -- the adjoint stage kernels of adj_stage.h on Cartesian elements.
#include "adj_stage.h"

namespace nmx {

hipError_t launch_adj_jobs_box(const AdjArgs &a, hipStream_t s) { return launch_adj_jobs_geom<0>(a, s); }
hipError_t launch_adj_box(int np, int nmax, const AdjArgs &a, hipStream_t s) {
  return launch_adj_geom<0>(np, nmax, a, s);
}

}  // namespace nmx
