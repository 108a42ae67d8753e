// fvelm_llf_kernels.hip -- the FV element kernels (fvelm_stage.h) with LLF
// fluxes, which act on all of c: a translation unit of its own, so the upwind
// kernels hold only the components that their fluxes act on.
#include "fvelm_stage.h"

namespace nmx {

hipError_t launch_fvelm_llf(int np, int rec, int geom, const AmrArgs &a, const double *wc, hipStream_t s) {
  return launch_fvelm_v<false, true>(np, rec, geom, a, wc, s);
}

}  // namespace nmx
