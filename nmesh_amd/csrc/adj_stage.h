// adj_stage.h -- discrete adjoint of the scalarwave1 DG right-hand side, fused
// with the RK stage combination, for conforming meshes and h-refined ones of
// mixed orders, gfx950.  Instantiated by adj_box_kernels.hip,
// adj_stored_kernels.hip and adj_shell_kernels.hip (one geometry each).
//
// The forward RHS (dg_stage.h) is linear in u:
//   r_pi(p) = sum_m sum_q M_p[m][q] g_m (D_m c_q)(p) - sum_{f at p} s_f(p) [A(n_f(p)) (u(p) - u_adj(p))]_pi
//   r_cq(p) = sum_m M_p[m][q] g_m (D_m pi)(p)        - sum_{f at p} s_f(p) [A(n_f(p)) (u(p) - u_adj(p))]_cq
//   r_phi(p) = pi(p)
// with g_m = dXb/dX of the element, M = dX/dx, D_m the LGL derivative along
// direction m, s_f the lift scale sqrtgdiag / w_end and A(n) the flux
// Jacobian of the upwind or LLF flux (scalarwave1.c:139-209,324-499;
// numflux1d.c:85-112; dg.c:90-146).  A(n) is symmetric for both fluxes
// (upwind: 1/2 [[1, n^T], [n, n n^T]]; LLF: 1/2 [[1, n^T], [n, I]]), so its
// transpose is applied with the forward face_flux.  The transpose y = L^T lam:
//   y_cq(s) = sum_m (D_m^T a_mq)(s),   a_mq = g_m M[m][q] lam_pi
//   y_pi(s) = sum_m (D_m^T b_m)(s) + lam_phi(s),  b_m = g_m sum_q M[m][q] lam_cq
//   face nodes: y(s) -= s_f(s) A(n_f(s)) lam(s), plus what the points that
//               read s hand back;
//   y_phi = 0.
// What the readers hand back to a face plane:
//   copy faces (the relation is mutual): the partner's s A(n) lam at the same
//     point.  Its normal is the opposite of this element's, and its scale
//     s this face's times a factor constant on the face (fg, AdjArgs: the
//     ratio of the two elements' dXb/dX, and at the interface of two shells, where
//     |dlam/dx| jumps, of their thicknesses): only the partner's values are
//     gathered;
//   interpolated faces (surface.c:1081-1337, interpolate.c:296-363): T = R1^T
//     (w G) R2 of every (receiving face, neighbour) job that reads the plane, G
//     = s A(n) lam at the receiving points, w = 1 / count where several
//     neighbours hold a point, summed in a fixed order.
// Two passes per stage: adj_jobs_kernel (T per job, one wave each) and one
// thread per node of every element.  Everything an element needs is requested
// before its only barrier, and all fields to be contracted are formed per node
// before it: on shells with c along the patch's axes (node_rhs, dg_stage.h) 7
// fields and 8 contractions instead of three rounds of 4 fields.
// Every sum runs in a fixed order, so the result is deterministic.
#pragma once
#include <hip/hip_runtime.h>

#include "amr.h"
#include "dg_stage.h"

namespace nmx {

// LDS fields of the contraction: GEOM 2 lam_pi, lam_n (x), f1 (y and z), f2,
// f3 (y), f4, f5 (z); GEOM 0 lam; GEOM 1 a_m0, a_m1, a_m2, b_m for each m
constexpr int adj_fields(int geom) { return geom == 2 ? 7 : geom == 0 ? 4 : 12; }

template <int NP, int GEOM, int WM, int NT>
__device__ __forceinline__ void adj_elem(const AdjArgs &a, int it, const double *D,
                                         const double *xb, double wend_inv, double *l_t, double *l_f,
                                         double *s_D) {
  constexpr int NP2 = NP * NP;
  constexpr int NP3 = NP * NP * NP;
  constexpr int NQ = (6 * NP2 + NT - 1) / NT;   // face points per thread
  const NMX_CONST SlotRec &R = as_const(a.rec)[it];
  double(*s_t)[NP3] = reinterpret_cast<double(*)[NP3]>(l_t);
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
  for (int v = 0; v < 4; ++v) u[v] = a.lam[gbase + node + vo[v]];
  const double ph = a.phi[gbase + node + 4 * NP3];
  // copy faces: the partner's lam; interpolated faces: the sum of the T planes
  double fv[NQ][4];
#pragma unroll
  for (int c = 0; c < NQ; ++c) {
    const int p = min(tid + c * NT, 6 * NP2 - 1);
    const int f = p / NP2, q = p % NP2;
    const int kind = R.fkind[f];
#pragma unroll
    for (int v = 0; v < 4; ++v) fv[c][v] = 0.0;
    if (kind == 1) {
      const double *lp = a.lam + R.foff[f] + (q % NP) * R.fs1[f] + (q / NP) * R.fs2[f];
#pragma unroll
      for (int v = 0; v < 4; ++v) fv[c][v] = lp[vo[v]];
    } else if (kind == 2) {
      const AdjRead *rd = a.reads + R.foff[f];
      const int n = R.fs1[f];
      for (int x = 0; x < n; ++x) {
        const double *T = a.T + rd[x].off + (q % NP) * rd[x].ca + (q / NP) * rd[x].cb;
#pragma unroll
        for (int v = 0; v < 4; ++v) fv[c][v] += T[cmp[v] * NP2];
      }
    }
  }
  const StageRegs o = {a.lam, a.U, a.Wa, a.Wb, a.cA, a.cW, WM};
  StageIn in;
  if (WM != 0) stage_in(o, gbase + node, vo, 4 * NP3, in);
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
    if (GEOM == 2) {
      const double f1 = m.sR * u[0];
      s_t[0][node] = u[0];
      s_t[1][node] = u[1] + m.A * u[2] + m.B * u[3];
      s_t[2][node] = f1;
      s_t[3][node] = m.A * f1;
      s_t[4][node] = m.sR * (u[2] - m.A * u[1]);
      s_t[5][node] = m.B * f1;
      s_t[6][node] = m.sR * (u[3] - m.B * u[1]);
    } else if (GEOM == 0) {
#pragma unroll
      for (int v = 0; v < 4; ++v) s_t[v][node] = u[v];
    } else {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
#pragma unroll
        for (int c = 0; c < 3; ++c) s_t[4 * d + c][node] = m.M[d][c] * u[0];
        s_t[4 * d + 3][node] = m.M[d][0] * u[1] + m.M[d][1] * u[2] + m.M[d][2] * u[3];
      }
    }
  }
#pragma unroll
  for (int c = 0; c < NQ; ++c) {
    const int p = min(tid + c * NT, 6 * NP2 - 1);
#pragma unroll
    for (int v = 0; v < 4; ++v) s_f[p / NP2][v][p % NP2] = fv[c][v];
  }
  __syncthreads();
  if (!act) return;

  // sums over the transposed derivatives along i, j, k of the fields above
  double x[4] = {0, 0, 0, 0}, y[4] = {0, 0, 0, 0}, z[4] = {0, 0, 0, 0};
#pragma unroll
  for (int l = 0; l < NP; ++l) {
    const double Di = s_D[l * NP + i], Dj = s_D[l * NP + j], Dk = s_D[l * NP + k];
    const int px = node + l - i, py = node + (l - j) * NP, pz = node + (l - k) * NP2;
    if (GEOM == 2) {
      x[0] += Di * s_t[0][px];
      x[1] += Di * s_t[1][px];
      y[0] += Dj * s_t[2][py];
      y[1] += Dj * s_t[3][py];
      y[2] += Dj * s_t[4][py];
      z[0] += Dk * s_t[2][pz];
      z[1] += Dk * s_t[5][pz];
      z[2] += Dk * s_t[6][pz];
    } else if (GEOM == 0) {
      x[0] += Di * s_t[0][px];
      x[1] += Di * s_t[1][px];
      y[0] += Dj * s_t[0][py];
      y[1] += Dj * s_t[2][py];
      z[0] += Dk * s_t[0][pz];
      z[1] += Dk * s_t[3][pz];
    } else {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        x[v] += Di * s_t[v][px];
        y[v] += Dj * s_t[4 + v][py];
        z[v] += Dk * s_t[8 + v][pz];
      }
    }
  }
  double r[4];
  if (GEOM == 2) {
    const double c0 = m.g[0] * (m.pm * m.idr) * m.rs, xp = c0 * x[0];
    r[0] = c0 * x[1] + m.g[1] * y[2] + m.g[2] * z[2];
    r[1] = xp - m.g[1] * y[1] - m.g[2] * z[1];
    r[2] = m.A * xp + m.g[1] * y[0];
    r[3] = m.B * xp + m.g[2] * z[0];
  } else if (GEOM == 0) {
    r[0] = m.g[0] * x[1] + m.g[1] * y[1] + m.g[2] * z[1];
    r[1] = m.g[0] * x[0];
    r[2] = m.g[1] * y[0];
    r[3] = m.g[2] * z[0];
  } else {
    r[0] = m.g[0] * x[3] + m.g[1] * y[3] + m.g[2] * z[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) r[1 + c] = m.g[0] * x[c] + m.g[1] * y[c] + m.g[2] * z[c];
  }
#pragma unroll
  for (int dir = 0; dir < 3; ++dir) {
    const int I = dir == 0 ? i : dir == 1 ? j : k;
    if (I == 0 || I == NP - 1) {
      const int side = I == 0 ? 0 : 1, t = (dir == 0 ? j : i) + NP * (dir == 2 ? j : k);
      const double(*sf)[NP2] = s_f[2 * dir + side];
      const double fa[4] = {sf[0][t], sf[1][t], sf[2][t], sf[3][t]};
      double nrm[3], scale, F[4];
      node_face<GEOM>(m, dir, side ? 1.0 : -1.0, wend_inv, nrm, scale);
      face_flux(a.numflux, nrm, u[0], u + 1, F);
#pragma unroll
      for (int v = 0; v < 4; ++v) r[v] -= scale * F[v];
      if (R.fkind[2 * dir + side] == 1) {
        const double opp[3] = {-nrm[0], -nrm[1], -nrm[2]};
        const double sc = scale * as_const(a.fg)[6 * it + 2 * dir + side];
        face_flux(a.numflux, opp, fa[0], fa + 1, F);
#pragma unroll
        for (int v = 0; v < 4; ++v) r[v] += sc * F[v];
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v) r[v] += fa[v];
      }
    }
  }
  r[0] += ph;

  const long gi = gbase + node;
  if (WM != 0) {
    double out[5];
    stage_out<false>(o, in, u, r, out);
#pragma unroll
    for (int v = 0; v < 4; ++v) a.Wout[gi + vo[v]] = out[v];
  } else {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      if (a.R) a.R[gi + vo[v]] = r[v];
      if (a.wmode == 1) a.Wout[gi + vo[v]] = a.U[gi + vo[v]] + a.cW * r[v];
    }
    if (a.R) a.R[gi + 4 * NP3] = 0.0;
    if (a.wmode == 1) a.Wout[gi + 4 * NP3] = a.U[gi + 4 * NP3];
  }
}

template <int NP, int GEOM, int WM>
__global__ __launch_bounds__(node_threads(NP)) void adj_node_kernel(AdjArgs a) {
  __shared__ double s_t[adj_fields(GEOM) * NP * NP * NP];
  __shared__ double s_f[6 * 4 * NP * NP];
  __shared__ double s_D[NP * NP];
  const int it = xcd_block(a.nlist, a.xcd_map);
  if (it >= a.nlist) return;
  adj_elem<NP, GEOM, WM, node_threads(NP)>(a, it, a.D, a.xb, a.wend_inv, s_t, s_f, s_D);
}

// elements of every order in one launch (dg_mixed_kernel, dg_stage.h)
template <int NMAX, int GEOM, int WM>
__global__ __launch_bounds__(node_threads(NMAX)) void adj_mixed_kernel(AdjArgs a) {
  __shared__ double s_t[adj_fields(GEOM) * NMAX * NMAX * NMAX];
  __shared__ double s_f[6 * 4 * NMAX * NMAX];
  __shared__ double s_D[NMAX * NMAX];
  const int it = xcd_block(a.nlist, a.xcd_map);
  if (it >= a.nlist) return;
  switch (as_const(a.rec)[it].n) {
#define NMX_CASE(N)                                                                                       \
  case N:                                                                                                 \
    if (N <= NMAX)                                                                                        \
      adj_elem<N <= NMAX ? N : 2, GEOM, WM, node_threads(NMAX)>(                                          \
          a, it, a.Dall + batch_doff(N), a.xball + batch_xoff(N), as_const(a.wall)[N], s_t, s_f, s_D);     \
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

// ---------------------------------------------------------------------------
// transposed interpolation, one wave per job:
//   W(x1, x2) = w(a, b) G(a, b) at the job's covered points,
//   S[x1][q2] = sum_x2 W(x1, x2) R2[x2][q2],
//   T(q1, q2) = sum_x1 R1[x1][q1] S[x1][q2]
// with (x1, x2) = (a, b), or (b, a) when the neighbour's first in-plane axis
// runs along the receiver's b: the transpose of face_interp_kernel's passes,
// with G taken from the receiver's lam as it is read.
// ---------------------------------------------------------------------------
constexpr int kAdjJobWaves = 4;   // jobs per workgroup

// One job with the receiver's order N known at compile time.  The covered
// ranges x1 < nx1, x2 < nx2 are padded to N with zero rows of W, R1, R2 and
// S, so the sums over x1 and x2 unroll without branches (their LDS reads are
// issued together) and add only exact zeros beyond the ranges.
template <int N, int GEOM>
__device__ __forceinline__ void adj_job(const AdjArgs &a, const NMX_CONST AdjJob &J, int tid, double *s_W,
                                        double *s_S, double *s_R1, double *s_R2) {
  constexpr int N2 = N * N, N3 = N * N * N;
  const int m = J.m, sw = J.sw;
  const int x1lo = sw ? J.b0 : J.a0, x2lo = sw ? J.a0 : J.b0;
  const int nx1 = (sw ? J.b1 - J.b0 : J.a1 - J.a0) + 1;
  const int nx2 = (sw ? J.a1 - J.a0 : J.b1 - J.b0) + 1;
  const double *R1 = a.Btab + (sw ? J.offB : J.offA) + x1lo * m;
  const double *R2 = a.Btab + (sw ? J.offA : J.offB) + x2lo * m;
  const NMX_CONST SlotRec &R = as_const(a.erec)[J.e];
  const double *lam = a.lam + 5 * R.noff;
  const double *xb = a.xball + batch_xoff(N);
  const double wend_inv = as_const(a.wall)[N];
  const int dir = J.g >> 1, pl = (J.g & 1) * (N - 1);
  const double sig = (J.g & 1) ? 1.0 : -1.0;
  int cmp[4];
  node_cmp<GEOM>(R, cmp);
  NodeGeo geo;
  node_geo_elem<GEOM>(R, geo);
  for (int idx = tid; idx < N * m; idx += 64) {
    s_R1[idx] = idx < nx1 * m ? R1[idx] : 0.0;
    s_R2[idx] = idx < nx2 * m ? R2[idx] : 0.0;
  }
  for (int r = tid; r < N2; r += 64) {
    const int x1 = r / N, x2 = r % N;
    double F[4] = {0.0, 0.0, 0.0, 0.0};
    if (x1 < nx1 && x2 < nx2) {
      const int fa = sw ? x2 + x2lo : x1 + x1lo, fb = sw ? x1 + x1lo : x2 + x2lo;
      double w = 1.0;
      if (J.md >= 0) {   // several neighbours: the averaging weight of this point
        const int *md = a.mdesc + J.md;
        int cnt = 0;
        for (int si = 0; si < md[0]; ++si) {
          const int *d = md + 1 + 5 * si;
          if (fa >= d[1] && fa <= d[2] && fb >= d[3] && fb <= d[4]) ++cnt;
        }
        if (cnt > 1) w = 1.0 / cnt;
      }
      const int i = dir == 0 ? pl : fa, jj = dir == 1 ? pl : (dir == 0 ? fa : fb), k = dir == 2 ? pl : fb;
      const int node = i + N * (jj + N * k);
      double u[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) u[v] = lam[cmp[v] * N3 + node];
      if (GEOM == 1) {
        const double *md = a.dXdx + 9 * R.noff + node;
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
          for (int c = 0; c < 3; ++c) geo.M[d][c] = md[(3 * d + c) * N3];
      } else if (GEOM == 2) {
        node_geo_shell(geo, patch_coord(R, 1, xb[jj]), patch_coord(R, 2, xb[k]),
                       geo.pm / (R.s0 + (R.s1 - R.s0) * patch_coord(R, 0, xb[i])));
      }
      double nrm[3], scale;
      if (dir == 0) node_face<GEOM>(geo, 0, sig, wend_inv, nrm, scale);
      else if (dir == 1) node_face<GEOM>(geo, 1, sig, wend_inv, nrm, scale);
      else node_face<GEOM>(geo, 2, sig, wend_inv, nrm, scale);
      face_flux(a.numflux, nrm, u[0], u + 1, F);
#pragma unroll
      for (int v = 0; v < 4; ++v) F[v] *= w * scale;
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) s_W[cmp[v] * N2 + r] = F[v];
  }
  wave_lds_fence();
  // idx < 400 and divisors up to 100: exact quotients from 16-bit reciprocals
  const int im = 65535 / m + 1, inm = 65535 / (N * m) + 1, imm = 65535 / (m * m) + 1;
  for (int idx = tid; idx < 4 * N * m; idx += 64) {
    const int v = (idx * inm) >> 16, r = idx - v * N * m;
    const int x1 = (r * im) >> 16, q2 = r - x1 * m;
    const double *W = s_W + (v * N + x1) * N;
    double t = 0.0;
#pragma unroll
    for (int x2 = 0; x2 < N; ++x2) t += W[x2] * s_R2[x2 * m + q2];
    s_S[idx] = t;
  }
  wave_lds_fence();
  double *T = a.T + J.toff;
  for (int idx = tid; idx < 4 * m * m; idx += 64) {
    const int v = (idx * imm) >> 16, r = idx - v * m * m;
    const int q2 = (r * im) >> 16, q1 = r - q2 * m;
    double t = 0.0;
#pragma unroll
    for (int x1 = 0; x1 < N; ++x1) t += s_R1[x1 * m + q1] * s_S[(v * N + x1) * m + q2];
    T[idx] = t;
  }
}

template <int GEOM>
__global__ __launch_bounds__(64 * kAdjJobWaves) void adj_jobs_kernel(AdjArgs a) {
  __shared__ double s_W[kAdjJobWaves][4 * kMaxFaceN * kMaxFaceN];
  __shared__ double s_S[kAdjJobWaves][4 * kMaxFaceN * kMaxFaceN];
  __shared__ double s_R1[kAdjJobWaves][kMaxFaceN * kMaxFaceN];
  __shared__ double s_R2[kAdjJobWaves][kMaxFaceN * kMaxFaceN];
  const int tid = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int chunk = (a.njobs + 7) >> 3, q = kAdjJobWaves * (blockIdx.x >> 3) + wv;
  const int ji = (blockIdx.x & 7) * chunk + q;
  if (q >= chunk || ji >= a.njobs) return;   // waves do not wait for one another
  const NMX_CONST AdjJob &J = as_const(a.jobs)[ji];
  switch (J.n) {
#define NMX_CASE(N_)                                                              \
  case N_:                                                                        \
    adj_job<N_, GEOM>(a, J, tid, s_W[wv], s_S[wv], s_R1[wv], s_R2[wv]);           \
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

template <int GEOM>
static hipError_t launch_adj_jobs_geom(const AdjArgs &a, hipStream_t s) {
  if (a.njobs <= 0) return hipSuccess;
  const int chunk = (a.njobs + 7) / 8;
  const int grid = 8 * ((chunk + kAdjJobWaves - 1) / kAdjJobWaves);
  hipLaunchKernelGGL(adj_jobs_kernel<GEOM>, dim3(grid), dim3(64 * kAdjJobWaves), 0, s, a);
  return hipGetLastError();
}

template <int NP, int GEOM, int WM>
static hipError_t launch_adj_wm(const AdjArgs &a, hipStream_t s) {
  hipLaunchKernelGGL((adj_node_kernel<NP, GEOM, WM>), dim3(a.xcd_map ? 8 * ((a.nlist + 7) / 8) : a.nlist),
                     dim3(node_threads(NP)), 0, s, a);
  return hipGetLastError();
}

template <int GEOM, int WM>
static hipError_t launch_adj_np(int np, int nmax, const AdjArgs &a, hipStream_t s) {
  if (np == 0) {
    if (nmax < 2 || nmax > 10) return hipErrorInvalidValue;
    const dim3 grid(a.xcd_map ? 8 * ((a.nlist + 7) / 8) : a.nlist);
    if (nmax <= 8) hipLaunchKernelGGL((adj_mixed_kernel<8, GEOM, WM>), grid, dim3(node_threads(8)), 0, s, a);
    else hipLaunchKernelGGL((adj_mixed_kernel<10, GEOM, WM>), grid, dim3(node_threads(10)), 0, s, a);
    return hipGetLastError();
  }
  switch (np) {
#define NMX_CASE(N) \
  case N:           \
    return launch_adj_wm<N, GEOM, WM>(a, s);
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

// np = 0: elements of any order up to nmax
template <int GEOM>
static hipError_t launch_adj_geom(int np, int nmax, const AdjArgs &a, hipStream_t s) {
  if (a.nlist <= 0) return hipSuccess;
  switch (a.wmode) {
    case 3: return launch_adj_np<GEOM, 3>(np, nmax, a, s);
    case 4: return launch_adj_np<GEOM, 4>(np, nmax, a, s);
    case 5: return launch_adj_np<GEOM, 5>(np, nmax, a, s);
    case 6: return launch_adj_np<GEOM, 6>(np, nmax, a, s);
    default: return launch_adj_np<GEOM, 0>(np, nmax, a, s);
  }
}

}  // namespace nmx
