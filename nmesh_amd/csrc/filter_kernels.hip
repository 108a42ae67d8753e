// filter_kernels.hip -- the exponential filter of the FILTER bin, applied in
// place to the state after each full step.
//
// Per element and filtered variable (expfilter_var, filter.c:75-92):
//   u <- u * J^jpow, with J = 1 / det(dXb/dx)  (var_to_var_times_JtoPower,
//        utilities.c:885-909; det_dXbdx as coordinates.c:173-203 sets it);
//   u <- F_z F_y F_x u, F = S diag(f) A per direction: the normalized
//        Legendre analysis A and synthesis S on the LGL nodes
//        (LGL_AT_ST_matrices, Legendre.c:257-307) around the coefficient
//        scaling f(i) = exp(-alp (i/N)^s) (expfilter_coeff_array,
//        filter.c:20-55).  The reference applies A, the scaling and S as six
//        directional passes; the product S diag(f) A is the same operator in
//        three, one LDS round trip each;
//   u <- u * J^-jpow (factors of J that are constant on the element cancel).
// One workgroup per element, one node per thread, the filtered variables in
// two LDS copies in turn: three barriers.  On few elements the chain load -
// three passes - store bounds it (384 shell elements of 7^3 points: 6.9 us, with
// one copy, seven barriers, the loads of the variables one after another and
// the metric's determinant by divisions 12.3 under the same profile).
#include <hip/hip_runtime.h>

#include "amr.h"
#include "dg_common.h"
#include "dg_stage.h"

namespace nmx {

// one thread per node
constexpr int filter_threads(int np) { return (np * np * np + 63) / 64 * 64; }

// ALL: every variable is filtered, so nothing branches on the mask
template <int NP, int GEOM, bool ALL>
__global__ __launch_bounds__(filter_threads(NP)) void filter_kernel(FilterArgs a) {
  constexpr int NP2 = NP * NP;
  constexpr int NP3 = NP * NP * NP;
  constexpr int NT = filter_threads(NP);
  __shared__ double s_u[2][5][NP3];
  __shared__ double s_F[NP2];
  const int it = xcd_block(a.nlist, a.xcd_map);
  if (it >= a.nlist) return;
  const int tid = threadIdx.x;
  const NMX_CONST SlotRec &R = as_const(a.rec)[it];
  const long noff = R.noff;
  double *u = a.u + 5 * noff;
  const int mask = ALL ? 31 : a.varmask;
  // lanes past the last node repeat it and store nothing
  const int node = min(tid, NP3 - 1);
  const int i = node % NP, j = (node / NP) % NP, k = node / NP2;
  double val[5];
#pragma unroll
  for (int v = 0; v < 5; ++v) val[v] = ALL || (mask >> v & 1) ? u[v * NP3 + node] : 0.0;
  for (int q = tid; q < NP2; q += NT) s_F[q] = a.F[q];
  // the weight w = J^jpow up to a factor constant on the element and 1 / w:
  // none on boxes; on shells det(dX/dx) = s^3 / ((s1 - s0) R^2) up to its sign
  // (NodeGeo, dg_stage.h)
  double w = 1.0, iw = 1.0;
  const bool weighted = GEOM != 0 && (a.jpow == 1 || a.jpow == -1);
  if (weighted) {
    if (GEOM == 1) {
      double M[3][3];
      const double *g = a.dXdx + 9 * noff;
#pragma unroll
      for (int m = 0; m < 3; ++m)
#pragma unroll
        for (int q = 0; q < 3; ++q) M[m][q] = g[(3 * m + q) * NP3 + node];
      w = det3(M);
      iw = rcp_nr(w);
    } else {
      const double A = patch_coord(R, 1, a.xb[j]), B = patch_coord(R, 2, a.xb[k]);
      const double r = R.s0 + (R.s1 - R.s0) * patch_coord(R, 0, a.xb[i]);
      const double t = 1.0 + A * A + B * B, rs = rsqrt_nr(t), ir = rcp_nr(r);
      w = t * t * rs * (ir * ir);
      iw = rcp_nr(w);
    }
    if (a.jpow == 1) {
      w = iw;
      iw = rcp_nr(w);
    }
#pragma unroll
    for (int v = 0; v < 5; ++v) val[v] *= w;
  }
  if (tid < NP3) {
#pragma unroll
    for (int v = 0; v < 5; ++v) s_u[0][v][node] = val[v];
  }
  __syncthreads();
  // F along x, y, z
#pragma unroll
  for (int dir = 0; dir < 3; ++dir) {
    const int im = dir == 0 ? i : dir == 1 ? j : k;
    const int stride = dir == 0 ? 1 : dir == 1 ? NP : NP2;
    const int base = node - im * stride;
#pragma unroll
    for (int v = 0; v < 5; ++v) val[v] = 0.0;
#pragma unroll
    for (int l = 0; l < NP; ++l) {
      const double Fl = s_F[im * NP + l];
#pragma unroll
      for (int v = 0; v < 5; ++v)
        if (ALL || (mask >> v & 1)) val[v] += Fl * s_u[dir & 1][v][base + l * stride];
    }
    if (dir == 2) break;
    if (tid < NP3) {
#pragma unroll
      for (int v = 0; v < 5; ++v) s_u[~dir & 1][v][node] = val[v];
    }
    __syncthreads();
  }
  // undo the weighting, back to HBM
  if (tid >= NP3) return;
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    if (weighted) {
      // val / w with its remainder: what the weighting rounds off, every step
      // rounds off again
      const double q = val[v] * iw;
      val[v] = fma(fma(-q, w, val[v]), iw, q);
    }
    if (ALL || (mask >> v & 1)) u[v * NP3 + node] = val[v];
  }
}

template <int NP, int GEOM>
static hipError_t launch_filter_t(const FilterArgs &a, hipStream_t s) {
  const dim3 grid(a.xcd_map ? 8 * ((a.nlist + 7) / 8) : a.nlist), block(filter_threads(NP));
  if (a.varmask == 31) hipLaunchKernelGGL((filter_kernel<NP, GEOM, true>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((filter_kernel<NP, GEOM, false>), grid, block, 0, s, a);
  return hipGetLastError();
}

hipError_t launch_filter(int np, int geom, const FilterArgs &a, hipStream_t s) {
  if (a.nlist == 0 || a.varmask == 0) return hipSuccess;
#define NMX_CASE(N)                                              \
  case N:                                                        \
    if (geom == 0) return launch_filter_t<N, 0>(a, s);           \
    if (geom == 1) return launch_filter_t<N, 1>(a, s);           \
    return launch_filter_t<N, 2>(a, s);
  switch (np) {
    NMX_CASE(2)
    NMX_CASE(3)
    NMX_CASE(4)
    NMX_CASE(5)
    NMX_CASE(6)
    NMX_CASE(7)
    NMX_CASE(8)
    NMX_CASE(9)
    NMX_CASE(10)
    default:
      return hipErrorInvalidValue;
  }
#undef NMX_CASE
}

}  // namespace nmx
