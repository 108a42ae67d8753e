// fvelm_ex_kernels.hip -- the FV element kernels (fvelm_stage.h) with the
// fv_divf_extrap_s1 / _s2 / _opt limit of dnfn_extrap1 (rec1d.c:542-609);
// a separate translation unit so the variants compile in parallel and the
// common one keeps its registers.
#include "fvelm_stage.h"

namespace nmx {

hipError_t launch_fvelm_ex(int np, int rec, int geom, const AmrArgs &a, const double *wc, hipStream_t s) {
  return launch_fvelm_v<true, true>(np, rec, geom, a, wc, s);
}

}  // namespace nmx
