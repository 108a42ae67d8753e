// fastmath.h -- reciprocal and reciprocal square root in FP64 for the
// VALU-bound FV kernels, gfx950.
//
// 1 / b from the hardware's reciprocal estimate r0 (relative error e = 1 - b r0
// below 2^-23) as r0 (1 + e + e^2), and 1 / sqrt(x) from its estimate y0 (e = 1
// - x y0^2) as y0 (1 + e/2 + 3/8 e^2): the next terms are below 2^-68, so both
// are within about an ulp for normal operands.  Three and five instructions
// after the estimate, where two Newton steps take four and eight and an IEEE
// division or square root about 10 and 20.  Callers keep their operands normal
// and nonzero.
#pragma once
#include <hip/hip_runtime.h>

namespace nmx {

__device__ __forceinline__ double rcp_nr(double b) {
  const double r = __builtin_amdgcn_rcp(b);
  const double e = fma(-b, r, 1.0);
  return fma(r, fma(e, e, e), r);
}

__device__ __forceinline__ double rsqrt_nr(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}

}  // namespace nmx
