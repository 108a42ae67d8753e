// dg_stage.h -- the scalarwave1 DG right-hand side fused with the Runge-Kutta
// stage update, gfx950: one thread per (i, j) column of an element, or for
// few elements one thread per node.
// Instantiated by dg_box_kernels.hip, dg_stored_kernels.hip and
// dg_shell_kernels.hip (one geometry each, compiled in parallel).
//
// Per element:
//   - the tensor-product derivatives D_m q along the three directions
//     (src/main/amr/array.c:36-300 via basis_array_deriv1, basis.c:61-95),
//   - the non-conservative Cartesian divergence sum_m dXdx[m][i] dXbdX[m] D_m
//     (src/main/coordinates/derivs.c:102-181,756-815) of the scalarwave1 fluxes
//     f_pi^i = -c_i, f_cj^i = -pi delta_ij (scalarwave1.c:39-48,62-134),
//   - on face nodes the upwind or LLF numerical flux against the neighbour's
//     face value and the strong-form lift with sqrtgdiag / w_end
//     (scalarwave1.c:139-209,287-321,324-499; dg.c:30-151; numflux1d.c:85-112),
//   - the RHS r = -(div f + lift), r_phi = pi (scalarwave1.c:242-284),
//   - and the RK stage combination of evolve_RK4_mesh / evolve_sspRK3_mesh /
//     evolve_Euler_mesh (RungeKutta.c:19-188), so the RHS is never written
//     to HBM during a time step.
// Geometry (template GEOM): 0 Cartesian box (dXdx = 1), 1 dXdx streamed from
// HBM, 2 CubedShell dXdx recomputed from the element box and the cubed-sphere
// map (coordtrans_CubedSphere.c:259-509 with constant radii) instead of read.
// State layout: element blocks, element e at 5*off[e] doubles, variable v at
// +v*np, node ijk = i + n*(j + n*k) inside.
//
// Two shapes, chosen by order and number of elements (launch_dg_np).
//
// dg_node_kernel, one thread per node: every load (own fields, faces, D, the
// stage's other registers) is requested before the only barrier, and each
// thread has one node to finish after it.  A launch over a few elements costs
// one chain of waits.
//
// dg_col_kernel, one thread per (i, j) column: the column's 4 n values are
// requested at once and stay in registers, so the derivative along k needs no
// LDS, with D's row in scalar registers.  The planes k = 0, 1, .. go through a
// double-buffered LDS plane for the derivatives along i and j, whose rows of D
// the thread keeps.  Elements of up to 8 points per direction take one wave,
// which has no barriers; 9 and 10 take two and one barrier per plane.  4 to 12
// elements are in flight per CU.
// The stage's other registers are requested as a plane begins and used as it
// ends: a plane ahead, they cost registers and spills (n = 8 and 3072 elements,
// last RK4 stage: 52 us a launch, 50 without); held to three waves per SIMD, 66
// registers spill and steps take 2.5 times as long.
//
// One wave-wide pass over the mesh per stage is bound by its HBM traffic: on
// 3072 elements of 8 points a step moves 54 doubles per node in 146 us (4.65
// TB/s; a 2 GiB copy reaches 4.9).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "amr.h"
#include "dg_common.h"
#include "fastmath.h"

namespace nmx {

constexpr int col_threads(int np) { return (np * np + 63) / 64 * 64; }
// waves per SIMD that the registers are kept to (three for 7 points and the early
// stages measured the same: RK4 steps of 3072 elements 119 us either way)
constexpr int kColWaves = 2;
// row stride of an LDS plane: even, so rows of doubles load in pairs, and such
// that the rows read together by 16 lanes lie in different banks
constexpr int col_stride(int np) { return np == 7 || np == 8 ? 10 : (np + 1) / 2 * 2; }

// adjacent values (ajsurf) of pi and c at point q of face f, components in
// the order cmp: copied from a same-order neighbour (kind 1), interpolated
// this stage by face_interp_kernel (2), averaged over several neighbours
// where several hold the point (3, surface.c:1322-1337) or the exterior (0)
template <int NP>
__device__ __forceinline__ void stage_face(const AmrArgs &a, const NMX_CONST SlotRec &R, int f, int q, int fa, int fb,
                                         const int (&cmp)[4], double ua[4]) {
  constexpr int NP2 = NP * NP;
  constexpr int NP3 = NP * NP * NP;
  const int kind = R.fkind[f];
  if (kind == 1) {
    const double *p = a.win + R.foff[f] + fa * R.fs1[f] + fb * R.fs2[f];
#pragma unroll
    for (int v = 0; v < 4; ++v) ua[v] = p[cmp[v] * NP3];
  } else if (kind == 2) {
    const double *p = a.aj + R.foff[f] + q;
#pragma unroll
    for (int v = 0; v < 4; ++v) ua[v] = p[cmp[v] * NP2];
  } else if (kind == 3) {
    const int *md = a.mdesc + R.foff[f];
    const int ns = md[0];
    double sum[4] = {0.0, 0.0, 0.0, 0.0};
    int cnt = 0;
    for (int si = 0; si < ns; ++si) {
      const int *d = md + 1 + 5 * si;
      if (fa >= d[1] && fa <= d[2] && fb >= d[3] && fb <= d[4]) {
        const double *p = a.aj + d[0] + q;
#pragma unroll
        for (int v = 0; v < 4; ++v) sum[v] += p[cmp[v] * NP2];
        ++cnt;
      }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) ua[v] = cnt > 1 ? sum[v] / cnt : sum[v];
  } else {
#pragma unroll
    for (int v = 0; v < 4; ++v) ua[v] = 0.0;
    if (a.profile) {
      const int dir = f >> 1, pl = (f & 1) * (NP - 1);
      const int ii = (dir == 0) ? pl : fa;
      const int jj = (dir == 1) ? pl : ((dir == 0) ? fa : fb);
      const int kk = (dir == 2) ? pl : fb;
      const double *xp = a.xyz + 3 * R.noff + ii + NP * (jj + NP * kk);
      double w[4];
      plane_wave(a.k, a.om, xp[0], xp[NP3], xp[2 * NP3], a.tdev ? a.tdev[a.tidx] : a.t, w);
#pragma unroll
      for (int v = 0; v < 4; ++v) ua[v] = cmp[v] == 0 ? w[0] : cmp[v] == 1 ? w[1] : cmp[v] == 2 ? w[2] : w[3];
    }
  }
}

// The metric at one node.  GEOM 2: with s = sqrt(1 + A^2 + B^2), R = s0 + (s1
// - s0) lam and pm the patch's sign, the rows of dX/dx along (dir, ia, ib) are
// pm / ((s1 - s0) s) (1, A, B), pm s / R (-A, 1, 0) and pm s / R (-B, 0, 1)
// (shell_dXdx, dg_common.h).
struct NodeGeo {
  double g[3];           // dXb/dX
  double A, B, pm, idr;  // idr = 1 / (s1 - s0)
  double rs, sR;         // 1 / s, pm s / R
  double M[3][3];        // GEOM 1
};

template <int GEOM>
__device__ __forceinline__ void node_geo_elem(const NMX_CONST SlotRec &R, NodeGeo &m) {
  m.g[0] = R.dXbdX[0]; m.g[1] = R.dXbdX[1]; m.g[2] = R.dXbdX[2];
  if (GEOM == 2) {
    m.pm = (R.dom & 1) ? 1.0 : -1.0;
    m.idr = 1.0 / (R.s1 - R.s0);
  }
}
__device__ __forceinline__ double patch_coord(const NMX_CONST SlotRec &R, int d, double xb) {
  return 0.5 * ((R.bb[2 * d + 1] - R.bb[2 * d]) * xb + (R.bb[2 * d + 1] + R.bb[2 * d]));
}
// iR: pm / R at the node
__device__ __forceinline__ void node_geo_shell(NodeGeo &m, double A, double B, double iR) {
  m.A = A;
  m.B = B;
  const double t = 1.0 + A * A + B * B;
  m.rs = rsqrt_nr(t);
  m.sR = (t * m.rs) * iR;
}

// r from the derivatives of the fields along the element's directions.  GEOM
// 2: x[0] of pi, x[1] of c_n = c_r + A c_a + B c_b (A and B are constant along
// i, so one derivative serves the row (1, A, B)); y[0..2] of pi, c_r, c_a;
// z[0..2] of pi, c_r, c_b.  GEOM 0: x, y, z of pi and cx, cy or cz.  GEOM 1: of
// pi and all of c.
template <int GEOM>
__device__ __forceinline__ void node_rhs(const NodeGeo &m, const double x[4], const double y[4], const double z[4],
                                         double r[4]) {
  if (GEOM == 2) {
    const double c0 = m.g[0] * (m.pm * m.idr) * m.rs, c1 = m.g[1] * m.sR, c2 = m.g[2] * m.sR;
    const double xp = c0 * x[0], yp = c1 * y[0], zp = c2 * z[0];
    r[0] = c0 * x[1] + c1 * (y[2] - m.A * y[1]) + c2 * (z[2] - m.B * z[1]);
    r[1] = xp - m.A * yp - m.B * zp;
    r[2] = m.A * xp + yp;
    r[3] = m.B * xp + zp;
  } else if (GEOM == 0) {
    r[0] = m.g[0] * x[1] + m.g[1] * y[1] + m.g[2] * z[1];
    r[1] = m.g[0] * x[0];
    r[2] = m.g[1] * y[0];
    r[3] = m.g[2] * z[0];
  } else {
    const double *d[3] = {x, y, z};
#pragma unroll
    for (int v = 0; v < 4; ++v) r[v] = 0.0;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      r[0] += m.M[q][0] * (m.g[q] * d[q][1]) + m.M[q][1] * (m.g[q] * d[q][2]) + m.M[q][2] * (m.g[q] * d[q][3]);
#pragma unroll
      for (int c = 0; c < 3; ++c) r[1 + c] += m.M[q][c] * (m.g[q] * d[q][0]);
    }
  }
}

// outward unit normal of face 2 dir + side (sig -1 or 1) at a node on it and
// the lift's scale sqrtgdiag / w_end (dg.c:90-146,470-481 via
// node_normal_from_idXdx_at_ijk, utilities.c:48-81)
template <int GEOM>
__device__ __forceinline__ void node_face(const NodeGeo &m, int dir, double sig, double wend_inv, double nrm[3],
                                          double &scale) {
  if (GEOM == 2) {
    const double sg = sig * m.pm;
    if (dir == 0) {
      nrm[0] = sg * m.rs; nrm[1] = m.A * nrm[0]; nrm[2] = m.B * nrm[0];
      scale = m.g[0] * m.idr * wend_inv;
    } else {
      // row (-a, 1) over its length sqrt(1 + a^2)
      const double a = dir == 1 ? m.A : m.B, t = 1.0 + a * a, is = rsqrt_nr(t);
      const double n1 = sg * is;
      nrm[0] = -a * n1;
      nrm[1] = dir == 1 ? n1 : 0.0;
      nrm[2] = dir == 1 ? 0.0 : n1;
      scale = (fabs(m.sR) * m.g[dir]) * (t * is) * wend_inv;
    }
  } else if (GEOM == 0) {
    nrm[0] = dir == 0 ? sig : 0.0;
    nrm[1] = dir == 1 ? sig : 0.0;
    nrm[2] = dir == 2 ? sig : 0.0;
    scale = m.g[dir] * wend_inv;
  } else {
    face_normal<1>(m.M, m.g, 2 * dir + (sig > 0.0), wend_inv, nrm, scale);
  }
}

// lift of that face: r -= scale (fnum - f)(u - ua)
template <int GEOM>
__device__ __forceinline__ void node_lift(const NodeGeo &m, int dir, double sig, double wend_inv, int numflux,
                                          const double u[4], const double ua[4], double r[4]) {
  double nrm[3], scale;
  node_face<GEOM>(m, dir, sig, wend_inv, nrm, scale);
  const double dc[3] = {u[1] - ua[1], u[2] - ua[2], u[3] - ua[3]};
  double F[4];
  face_flux(numflux, nrm, u[0] - ua[0], dc, F);
#pragma unroll
  for (int v = 0; v < 4; ++v) r[v] -= F[v] * scale;
}

// What a stage with an accumulator (wmodes 0 to 2) reads at a node besides its
// own pi and c: u_p, the accumulator and its input's phi.
struct AccIn {
  double U[5], A[5], phi;
};
// ... and a right-hand side alone: nothing
struct RhsIn {};
template <int WM>
using NodeIn = std::conditional_t<WM == 0, AccIn, std::conditional_t<WM == 1, RhsIn, StageIn>>;

// the operands of node_out at the node whose first state double is gi,
// requested together: between node_out's stores, which they may alias, they were
// five round trips one after another (3072 shell elements of 8 points: Euler steps
// 62 us, 41 so, RK4 steps with the MRS limiter 556 and 440; 19,200 elements of 4
// to 10 points: Euler steps 555 and 453)
__device__ __forceinline__ void node_in(const AmrArgs &a, const StageRegs &, long gi, const int (&vo)[4], int po,
                                        AccIn &q) {
  if (a.wmode) {
#pragma unroll
    for (int v = 0; v < 5; ++v) q.U[v] = a.U[gi + (v < 4 ? vo[v] : po)];
  }
  if (a.Ain) {
#pragma unroll
    for (int v = 0; v < 5; ++v) q.A[v] = a.Ain[gi + (v < 4 ? vo[v] : po)];
  }
  if (a.wmode == 2 || (a.Aout && !a.Ain)) q.phi = a.win[gi + po];
}
__device__ __forceinline__ void node_in(const AmrArgs &, const StageRegs &, long, const int (&)[4], int, RhsIn &) {}
__device__ __forceinline__ void node_in(const AmrArgs &, const StageRegs &o, long gi, const int (&vo)[4], int po,
                                        StageIn &q) {
  stage_in(o, gi, vo, po, q);
}

// the stage's output there
__device__ __forceinline__ void node_out(const AmrArgs &a, const StageRegs &, const RhsIn &, long gi,
                                         const int (&vo)[4], int po, const double u[4], const double r[4]) {
#pragma unroll
  for (int v = 0; v < 4; ++v) a.R[gi + vo[v]] = r[v];
  a.R[gi + po] = u[0];
}
__device__ __forceinline__ void node_out(const AmrArgs &a, const StageRegs &, const AccIn &q, long gi,
                                         const int (&vo)[4], int po, const double u[4], const double r[4]) {
#pragma unroll
  for (int v = 0; v < 5; ++v) {
    const long g = gi + (v < 4 ? vo[v] : po);
    const double rv = v < 4 ? r[v] : u[0], w = v < 4 ? u[v] : q.phi;
    if (a.R) a.R[g] = rv;
    if (a.Aout) a.Aout[g] = (a.Ain ? q.A[v] : w) + a.cA * rv;
    if (a.wmode == 1) a.Wout[g] = q.U[v] + a.cW * rv;
    else if (a.wmode == 2) a.Wout[g] = 0.75 * q.U[v] + 0.25 * (w + a.cW * rv);
  }
}
__device__ __forceinline__ void node_out(const AmrArgs &a, const StageRegs &o, const StageIn &q, long gi,
                                         const int (&vo)[4], int po, const double u[4], const double r[4]) {
  double out[5];
  const bool end = stage_out<true>(o, q, u, r, out);
#pragma unroll
  for (int v = 0; v < 4; ++v) a.Wout[gi + vo[v]] = out[v];
  if (end) a.Wout[gi + po] = out[4];
}

// components of c along the patch's axes (dir, ia, ib): cmp[v] is the
// variable held as v (GEOM 2)
template <int GEOM>
__device__ __forceinline__ void node_cmp(const NMX_CONST SlotRec &R, int (&cmp)[4]) {
  cmp[0] = 0; cmp[1] = 1; cmp[2] = 2; cmp[3] = 3;
  if (GEOM == 2) {
    const int dir = R.dom >> 1, ia = dir == 1 ? 0 : 1;
    cmp[1] = 1 + dir;
    cmp[2] = 1 + ia;
    cmp[3] = 4 - dir - ia;
  }
}

template <int WM>
__device__ __forceinline__ StageRegs node_args(const AmrArgs &a) {
  return {a.win, a.U, a.Wa, a.Wb, a.cA, a.cW, WM};
}

// the workgroup's index in [0, nblk), contiguous ranges per XCD when mapped
// (workgroups are dispatched round-robin over the 8 XCDs), so neighbour faces
// are mostly read from the same XCD's L2; nblk and above: nothing to do
__device__ __forceinline__ int xcd_block(int nblk, int xcd_map) {
  if (!xcd_map) return blockIdx.x;
  const int chunk = (nblk + 7) >> 3, q = blockIdx.x >> 3;
  return q < chunk ? (blockIdx.x & 7) * chunk + q : nblk;
}

// WM: what the launch does with the RHS, wmode WM (3 to 6), 1 R alone, or for WM
// = 0 any of R, the accumulator and wmodes 1 and 2.  R alone holds no operands and
// so 20 to 40 registers less: right-hand sides of 4096 box elements take, with the
// kernel for all of them and alone, 33 and 28 us (7 points), 81 and 60 (9) and
// 107 and 92 (10), of 3072 shell elements 38 and 34 (8) and 85 and 75 (10).
inline int stage_kind(const AmrArgs &a) {
  return a.wmode >= 3 ? a.wmode : a.R && !a.Aout && !a.wmode ? 1 : 0;
}
template <int NP, int GEOM, int WM>
__global__ __launch_bounds__(col_threads(NP), kColWaves) void dg_col_kernel(AmrArgs a) {
  constexpr int NP2 = NP * NP;
  constexpr int NP3 = NP * NP * NP;
  constexpr int S = col_stride(NP);
  // fields in an LDS plane: GEOM 2 pi, c_n, c_r, c_a (node_rhs); GEOM 0 pi, cx,
  // cy; GEOM 1 pi, cx, cy, cz
  constexpr int NF = GEOM == 0 ? 3 : 4;
  __shared__ __attribute__((aligned(16))) double s_p[2][NF][NP * S];
  __shared__ double s_f[6][4][NP2];   // adjacent values on the faces

  const int it = xcd_block(a.nlist, a.xcd_map);
  if (it >= a.nlist) return;   // the whole workgroup
  // lanes past the last column repeat another one and store nothing
  const int tid = threadIdx.x;
  const int q = tid % NP2;
  const bool act = tid < NP2;
  const NMX_CONST SlotRec &R = as_const(a.rec)[it];
  const long gbase = 5 * R.noff;
  const int i = q % NP, j = q / NP;

  int cmp[4];
  node_cmp<GEOM>(R, cmp);
  int vo[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) vo[v] = cmp[v] * NP3;

  // every load of the element: the columns, the faces, D's rows
  const double *w = a.win + gbase + q;
  double col[4][NP];
#pragma unroll
  for (int k = 0; k < NP; ++k)
#pragma unroll
    for (int v = 0; v < 4; ++v) col[v][k] = w[vo[v] + k * NP2];
  double fv[6][4];
#pragma unroll
  for (int f = 0; f < 6; ++f) stage_face<NP>(a, R, f, q, i, j, cmp, fv[f]);
  double Di[NP], Dj[NP];
#pragma unroll
  for (int l = 0; l < NP; ++l) {
    Di[l] = a.D[i * NP + l];
    Dj[l] = a.D[j * NP + l];
  }
  const StageRegs o = node_args<WM>(a);
#pragma unroll
  for (int f = 0; f < 6; ++f)
#pragma unroll
    for (int v = 0; v < 4; ++v) s_f[f][v][q] = fv[f][v];

  NodeGeo m;
  node_geo_elem<GEOM>(R, m);
  double A = 0, iR = 0;
  if (GEOM == 2) {
    A = patch_coord(R, 1, a.xb[j]);
    iR = m.pm / (R.s0 + (R.s1 - R.s0) * patch_coord(R, 0, a.xb[i]));
  }

#pragma unroll
  for (int k = 0; k < NP; ++k) {
    const double u[4] = {col[0][k], col[1][k], col[2][k], col[3][k]};
    double(*P)[NP * S] = s_p[k & 1];
    const int pq = j * S + i;
    if (GEOM == 2) {
      node_geo_shell(m, A, patch_coord(R, 2, a.xb[k]), iR);
      P[0][pq] = u[0];
      P[1][pq] = u[1] + m.A * u[2] + m.B * u[3];
      P[2][pq] = u[1];
      P[3][pq] = u[2];
    } else {
#pragma unroll
      for (int v = 0; v < NF; ++v) P[v][pq] = u[v];
    }
    if (GEOM == 1) {
      const double *md = a.dXdx + 9 * R.noff + q + k * NP2;
#pragma unroll
      for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int c = 0; c < 3; ++c) m.M[d][c] = md[(3 * d + c) * NP3];
    }
    NodeIn<WM> in;
    node_in(a, o, gbase + q + k * NP2, vo, 4 * NP3, in);
    __syncthreads();

    // ---- derivatives along i (rows of the plane), j and k ----
    double x[4] = {0, 0, 0, 0}, y[4] = {0, 0, 0, 0}, z[4] = {0, 0, 0, 0};
    constexpr int NX = GEOM == 1 ? 4 : 2;
#pragma unroll
    for (int v = 0; v < NX; ++v) {
      const double2 *p = reinterpret_cast<const double2 *>(P[v] + j * S);
#pragma unroll
      for (int l = 0; l < NP / 2; ++l) {
        const double2 t = p[l];
        x[v] += Di[2 * l] * t.x;
        x[v] += Di[2 * l + 1] * t.y;
      }
      if (NP & 1) x[v] += Di[NP - 1] * P[v][j * S + NP - 1];
    }
#pragma unroll
    for (int l = 0; l < NP; ++l) {
      const double Dk = as_const(a.D)[k * NP + l];
      const int t = l * S + i;
      y[0] += Dj[l] * P[0][t];
      z[0] += Dk * col[0][l];
      if (GEOM == 0) {
        y[1] += Dj[l] * P[2][t];
        z[1] += Dk * col[3][l];
      } else if (GEOM == 2) {
        y[1] += Dj[l] * P[2][t];
        y[2] += Dj[l] * P[3][t];
        z[1] += Dk * col[1][l];
        z[2] += Dk * col[3][l];
      } else {
#pragma unroll
        for (int v = 1; v < 4; ++v) {
          y[v] += Dj[l] * P[v][t];
          z[v] += Dk * col[v][l];
        }
      }
    }
    double r[4];
    node_rhs<GEOM>(m, x, y, z, r);

    // ---- numerical flux and lift on the faces this node lies on ----
#pragma unroll
    for (int dir = 0; dir < 2; ++dir) {
      const int I = dir == 0 ? i : j, t = dir == 0 ? j : i;
      if (I == 0 || I == NP - 1) {
        const int side = I == 0 ? 0 : 1;
        const double(*sf)[NP2] = s_f[2 * dir + side];
        const double ua[4] = {sf[0][t + NP * k], sf[1][t + NP * k], sf[2][t + NP * k], sf[3][t + NP * k]};
        node_lift<GEOM>(m, dir, side ? 1.0 : -1.0, a.wend_inv, a.numflux, u, ua, r);
      }
    }
    if (k == 0 || k == NP - 1) {
      const double(*sf)[NP2] = s_f[k ? 5 : 4];
      const double ua[4] = {sf[0][q], sf[1][q], sf[2][q], sf[3][q]};
      node_lift<GEOM>(m, 2, k ? 1.0 : -1.0, a.wend_inv, a.numflux, u, ua, r);
    }
    if (act) node_out(a, o, in, gbase + q + k * NP2, vo, 4 * NP3, u, r);
  }
}

// ---------------------------------------------------------------------------
// one thread per node
// ---------------------------------------------------------------------------
constexpr int node_threads(int np) { return (np * np * np + 63) / 64 * 64; }
constexpr int node_fields(int geom) { return geom == 2 ? 5 : 4; }   // pi, c and for GEOM 2 c_n

// the element of record R with NT threads; D, xb, wend_inv of its order
template <int NP, int GEOM, int WM, int NT>
__device__ __forceinline__ void node_elem(const AmrArgs &a, const NMX_CONST SlotRec &R, const double *D,
                                          const double *xb, double wend_inv, double *l_u, double *l_f,
                                          double *s_D) {
  constexpr int NP2 = NP * NP;
  constexpr int NP3 = NP * NP * NP;
  constexpr int NQ = (6 * NP2 + NT - 1) / NT;   // face points per thread
  constexpr int NF = node_fields(GEOM);
  double(*s_u)[NP3] = reinterpret_cast<double(*)[NP3]>(l_u);
  double(*s_f)[4][NP2] = reinterpret_cast<double(*)[4][NP2]>(l_f);
  const int tid = threadIdx.x;
  const long gbase = 5 * R.noff;
  const bool act = tid < NP3;
  const int node = act ? tid : 0;
  const int i = node % NP, j = (node / NP) % NP, k = node / NP2;
  int cmp[4], vo[4];
  node_cmp<GEOM>(R, cmp);
#pragma unroll
  for (int v = 0; v < 4; ++v) vo[v] = cmp[v] * NP3;

  double u[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) u[v] = a.win[gbase + node + vo[v]];
  double fv[NQ][4];
#pragma unroll
  for (int c = 0; c < NQ; ++c) {
    const int p = min(tid + c * NT, 6 * NP2 - 1);
    const int f = p / NP2, q = p % NP2;
    stage_face<NP>(a, R, f, q, q % NP, q / NP, cmp, fv[c]);
  }
  const StageRegs o = node_args<WM>(a);
  NodeIn<WM> in;
  node_in(a, o, gbase + node, vo, 4 * NP3, in);
  NodeGeo m;
  node_geo_elem<GEOM>(R, m);
  if (GEOM == 1) {
    const double *md = a.dXdx + 9 * R.noff + node;
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int c = 0; c < 3; ++c) m.M[d][c] = md[(3 * d + c) * NP3];
  }
  for (int q = tid; q < NP2; q += NT) s_D[q] = D[q];
  if (GEOM == 2)
    node_geo_shell(m, patch_coord(R, 1, xb[j]), patch_coord(R, 2, xb[k]),
                   m.pm / (R.s0 + (R.s1 - R.s0) * patch_coord(R, 0, xb[i])));
  if (act) {
#pragma unroll
    for (int v = 0; v < 4; ++v) s_u[v][node] = u[v];
    if (GEOM == 2) s_u[NF - 1][node] = u[1] + m.A * u[2] + m.B * u[3];
  }
#pragma unroll
  for (int c = 0; c < NQ; ++c) {
    const int p = min(tid + c * NT, 6 * NP2 - 1);
#pragma unroll
    for (int v = 0; v < 4; ++v) s_f[p / NP2][v][p % NP2] = fv[c][v];
  }
  __syncthreads();
  if (!act) return;

  double x[4] = {0, 0, 0, 0}, y[4] = {0, 0, 0, 0}, z[4] = {0, 0, 0, 0};
#pragma unroll
  for (int l = 0; l < NP; ++l) {
    const double Di = s_D[i * NP + l], Dj = s_D[j * NP + l], Dk = s_D[k * NP + l];
    const int px = node + l - i, py = node + (l - j) * NP, pz = node + (l - k) * NP2;
    x[0] += Di * s_u[0][px];
    y[0] += Dj * s_u[0][py];
    z[0] += Dk * s_u[0][pz];
    if (GEOM == 0) {
      x[1] += Di * s_u[1][px];
      y[1] += Dj * s_u[2][py];
      z[1] += Dk * s_u[3][pz];
    } else if (GEOM == 2) {
      x[1] += Di * s_u[NF - 1][px];
      y[1] += Dj * s_u[1][py];
      y[2] += Dj * s_u[2][py];
      z[1] += Dk * s_u[1][pz];
      z[2] += Dk * s_u[3][pz];
    } else {
#pragma unroll
      for (int v = 1; v < 4; ++v) {
        x[v] += Di * s_u[v][px];
        y[v] += Dj * s_u[v][py];
        z[v] += Dk * s_u[v][pz];
      }
    }
  }
  double r[4];
  node_rhs<GEOM>(m, x, y, z, r);
#pragma unroll
  for (int dir = 0; dir < 3; ++dir) {
    const int I = dir == 0 ? i : dir == 1 ? j : k;
    if (I == 0 || I == NP - 1) {
      const int side = I == 0 ? 0 : 1, t = (dir == 0 ? j : i) + NP * (dir == 2 ? j : k);
      const double(*sf)[NP2] = s_f[2 * dir + side];
      const double ua[4] = {sf[0][t], sf[1][t], sf[2][t], sf[3][t]};
      node_lift<GEOM>(m, dir, side ? 1.0 : -1.0, wend_inv, a.numflux, u, ua, r);
    }
  }
  node_out(a, o, in, gbase + node, vo, 4 * NP3, u, r);
}

// waves per SIMD that the registers are kept to: with an accumulator and a stored
// metric 8 points take 130 without a bound, two too many for two workgroups per CU
// (Euler steps of 888 elements 31.1 us, 28.5 with it; the other modes, which
// would spill more, measured no faster)
constexpr int node_waves(int np, int geom, int wm) { return np == 8 && geom == 1 && wm == 0 ? 4 : 1; }

template <int NP, int GEOM, int WM>
__global__ __launch_bounds__(node_threads(NP), node_waves(NP, GEOM, WM)) void dg_node_kernel(AmrArgs a) {
  __shared__ double s_u[node_fields(GEOM) * NP * NP * NP];
  __shared__ double s_f[6 * 4 * NP * NP];
  __shared__ double s_D[NP * NP];
  const int it = xcd_block(a.nlist, a.xcd_map);
  if (it >= a.nlist) return;
  node_elem<NP, GEOM, WM, node_threads(NP)>(a, as_const(a.rec)[it], a.D, a.xb, a.wend_inv, s_u, s_f, s_D);
}

// Elements of every order in one launch, with the threads and LDS of the
// largest of two groups of orders (NMAX 8 or 10): on meshes of a few hundred
// elements the launches of the orders, forked and joined, take longer than the
// elements.
template <int NMAX, int GEOM, int WM>
__global__ __launch_bounds__(node_threads(NMAX)) void dg_mixed_kernel(AmrArgs a) {
  constexpr int NT = node_threads(NMAX);
  __shared__ double s_u[node_fields(GEOM) * NMAX * NMAX * NMAX];
  __shared__ double s_f[6 * 4 * NMAX * NMAX];
  __shared__ double s_D[NMAX * NMAX];
  const int it = xcd_block(a.nlist, a.xcd_map);
  if (it >= a.nlist) return;
  const NMX_CONST SlotRec &R = as_const(a.rec)[it];
  switch (R.n) {
#define NMX_CASE(N)                                                                                       \
  case N:                                                                                                 \
    if (N <= NMAX)                                                                                        \
      node_elem<N <= NMAX ? N : 2, GEOM, WM, NT>(a, R, a.Dall + batch_doff(N), a.xball + batch_xoff(N),   \
                                                 as_const(a.wall)[N], s_u, s_f, s_D);                     \
    break;
    NMX_CASE(2)
    NMX_CASE(3)
    NMX_CASE(4)
    NMX_CASE(5)
    NMX_CASE(6)
    NMX_CASE(7)
    NMX_CASE(8)
    NMX_CASE(9)
    NMX_CASE(10)
#undef NMX_CASE
    default:
      break;   // orders outside 2..10 are refused on the host
  }
}

// The column kernel from 7 points per direction on and above a number of
// elements, the node kernel below.  us for RK4 steps, column against node kernel
// (elements refined, so with the face pass, from 771 to 2052):
//   shell, n = 5, 24,576 elements 405 and 355, n = 6 688 and 630;
//   n = 7: box 512 38 and 27, 1023 94 and 81, 1534 114 and 106, 2052 140 and 124,
//     shell 1504 133 and 123, 3072 119 and 130, 24,576 964 and 1216;
//   n = 8: box 512 44 and 32, 1023 106 and 97, 1534 128 and 124, 2052 155 and 146,
//     shell 1504 142 and 131, 3072 142 and 146, 24,576 1272 and 1403;
//   n = 10: box 512 74 and 67, 771 126 and 148, 1023 149 and 181, 2052 291 and 322,
//     shell 384 84 and 66, 783 143 and 161, 1084 209 and 205, 1504 255 and 258,
//     3072 375 and 433, 24,576 2963 and 3612.
// So for 7 and 8 points the line lies at 2048, and for 9 and 10, whose node
// workgroups of 12 and 16 waves leave fewer in flight, at 1024: somewhat lower
// for one order alone, but beside other orders' launches the column kernel
// gains later (16 steps of 3744 elements of 4 to 10 points 5780, 5860 to 6220
// with it from 256 elements on).
constexpr int node_elems(int np) { return np <= 8 ? 2048 : 1024; }

template <int NP, int GEOM, int WM>
static hipError_t launch_dg_wm(const AmrArgs &a, hipStream_t s) {
  const dim3 grid(a.xcd_map ? 8 * ((a.nlist + 7) / 8) : a.nlist);
  if constexpr (NP >= 7) {
    if (a.nlist > node_elems(NP)) {
      hipLaunchKernelGGL((dg_col_kernel<NP, GEOM, WM>), grid, dim3(col_threads(NP)), 0, s, a);
      return hipGetLastError();
    }
  }
  hipLaunchKernelGGL((dg_node_kernel<NP, GEOM, WM>), grid, dim3(node_threads(NP)), 0, s, a);
  return hipGetLastError();
}

template <int NP, int GEOM>
static hipError_t launch_dg_np(const AmrArgs &a, hipStream_t s) {
  switch (stage_kind(a)) {
    case 1: return launch_dg_wm<NP, GEOM, 1>(a, s);
    case 3: return launch_dg_wm<NP, GEOM, 3>(a, s);
    case 4: return launch_dg_wm<NP, GEOM, 4>(a, s);
    case 5: return launch_dg_wm<NP, GEOM, 5>(a, s);
    case 6: return launch_dg_wm<NP, GEOM, 6>(a, s);
    default: return launch_dg_wm<NP, GEOM, 0>(a, s);
  }
}

template <int GEOM, int WM>
static hipError_t launch_mixed_wm(int nmax, const AmrArgs &a, hipStream_t s) {
  const dim3 grid(a.xcd_map ? 8 * ((a.nlist + 7) / 8) : a.nlist);
  if (nmax <= 8) hipLaunchKernelGGL((dg_mixed_kernel<8, GEOM, WM>), grid, dim3(node_threads(8)), 0, s, a);
  else hipLaunchKernelGGL((dg_mixed_kernel<10, GEOM, WM>), grid, dim3(node_threads(10)), 0, s, a);
  return hipGetLastError();
}

// np = 0: elements of any order up to nmax
template <int GEOM>
static hipError_t launch_dg_geom(int np, int nmax, const AmrArgs &a, hipStream_t s) {
  if (a.nlist <= 0) return hipSuccess;
  if (np == 0) {
    if (nmax < 2 || nmax > 10) return hipErrorInvalidValue;
    switch (stage_kind(a)) {
      case 1: return launch_mixed_wm<GEOM, 1>(nmax, a, s);
      case 3: return launch_mixed_wm<GEOM, 3>(nmax, a, s);
      case 4: return launch_mixed_wm<GEOM, 4>(nmax, a, s);
      case 5: return launch_mixed_wm<GEOM, 5>(nmax, a, s);
      case 6: return launch_mixed_wm<GEOM, 6>(nmax, a, s);
      default: return launch_mixed_wm<GEOM, 0>(nmax, a, s);
    }
  }
  switch (np) {
#define NMX_CASE(N) \
  case N:           \
    return launch_dg_np<N, GEOM>(a, s);
    NMX_CASE(2)
    NMX_CASE(3)
    NMX_CASE(4)
    NMX_CASE(5)
    NMX_CASE(6)
    NMX_CASE(7)
    NMX_CASE(8)
    NMX_CASE(9)
    NMX_CASE(10)
#undef NMX_CASE
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace nmx
