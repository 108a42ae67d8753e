// adj_shell_kernels.hip -- the adjoint stage kernels of adj_stage.h on CubedShell elements, dX/dx recomputed.
#include "adj_stage.h"

namespace nmx {

hipError_t launch_adj_jobs_shell(const AdjArgs &a, hipStream_t s) { return launch_adj_jobs_geom<2>(a, s); }
hipError_t launch_adj_shell(int np, int nmax, const AdjArgs &a, hipStream_t s) {
  return launch_adj_geom<2>(np, nmax, a, s);
}

}  // namespace nmx
