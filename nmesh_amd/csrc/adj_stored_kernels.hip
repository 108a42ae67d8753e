// adj_stored_kernels.hip -- the adjoint stage kernels of adj_stage.h on curvilinear elements whose dX/dx is read.
#include "adj_stage.h"

namespace nmx {

hipError_t launch_adj_jobs_stored(const AdjArgs &a, hipStream_t s) { return launch_adj_jobs_geom<1>(a, s); }
hipError_t launch_adj_stored(int np, int nmax, const AdjArgs &a, hipStream_t s) {
  return launch_adj_geom<1>(np, nmax, a, s);
}

}  // namespace nmx
