// fvelm_kernels.hip -- the FV element kernels (fvelm_stage.h) with upwind
// fluxes and dnfn_extrap1's fixed weights, and the launcher that picks the
// variant with the fv_divf_extrap s1/s2/opt limit (fvelm_ex_kernels.hip) when
// it is on, or the one with LLF fluxes (fvelm_llf_kernels.hip).
#include "fvelm_stage.h"

namespace nmx {

hipError_t launch_fvelm(int np, int rec, int geom, const AmrArgs &a, const double *wc, hipStream_t s) {
  if (a.ex_on || a.recend != 0 || a.rec_first) return launch_fvelm_ex(np, rec, geom, a, wc, s);
  if (a.numflux) return launch_fvelm_llf(np, rec, geom, a, wc, s);
  return launch_fvelm_v<false, false>(np, rec, geom, a, wc, s);
}

}  // namespace nmx
