// dg_common.h -- device code shared by the DG, adjoint and FV stage kernels:
// numerical flux, boundary profile, cubed-shell Jacobian and the RK stages.
#pragma once
#include <hip/hip_runtime.h>

namespace nmx {

// Tables that no kernel writes are read through the constant address space:
// wave-uniform reads from them become scalar loads issued together, instead
// of a chain of vector loads each waiting for the last.
#define NMX_CONST __attribute__((address_space(4)))
template <class T>
__device__ __forceinline__ const NMX_CONST T *as_const(const T *p) {
  return (const NMX_CONST T *)p;
}

// LDS written by some lanes of a wave, read by others of the same wave: the
// wave's LDS instructions are done in order, so only the compiler has to keep
// them so
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// upwind: F = fnum - f_inner for the 4 flux-carrying fields.  With A = f.n
// Jacobian [[0,-n^T],[-n,0]], A+/- = (A +- |A|)/2 gives
// F_pi = (dpi + n.dc)/2 and F_c = n F_pi with d = inner - adjacent
// (scalarwave1_numflux1d_upwind, scalarwave1.c:324-499).
// LLF (amax = 1): F_pi = (dpi + n.dc)/2, F_c = (dc + n dpi)/2
// (numflux1d_LLF, numflux1d.c:85-112).
__device__ __forceinline__ void face_flux(int numflux, const double n[3], double dpi,
                                          const double dc[3], double F[4]) {
  double ndc = n[0] * dc[0] + n[1] * dc[1] + n[2] * dc[2];
  double Fp = 0.5 * (dpi + ndc);
  F[0] = Fp;
  if (numflux == 0) {
    F[1] = n[0] * Fp; F[2] = n[1] * Fp; F[3] = n[2] * Fp;
  } else {
    F[1] = 0.5 * (dc[0] + n[0] * dpi);
    F[2] = 0.5 * (dc[1] + n[1] * dpi);
    F[3] = 0.5 * (dc[2] + n[2] * dpi);
  }
}

// plane wave of scalarwave1_set_profile_pt (scalarwave1.c:503-524)
__device__ __forceinline__ void plane_wave(const double k[3], double om, double x, double y,
                                           double z, double t, double u[4]) {
  double arg = k[0] * x + k[1] * y + k[2] * z - om * t;
  double s, c;
  sincos(arg, &s, &c);
  (void)s;
  u[0] = -om * c; u[1] = k[0] * c; u[2] = k[1] * c; u[3] = k[2] * c;
}

// dX/dx of a CubedShell (constant radii s0, s1, centre 0) at patch point X
// (lam, A, B) (coordtrans_CubedSphere.c:259-509 with dsigma = 0).  With
// s = sqrt(1 + A^2 + B^2), the radius-like coordinate r = (pm/s)(s0 + (s1 -
// s0) lam) along the patch axis dir and x_dir = r, x_ia = A r, x_ib = B r,
// the reference's rows reduce to
//   dlam/dx = pm / ((s1 - s0) s) (1, A, B),
//   dA/dx   = (pm s / R) (-A, 1, 0),   dB/dx = (pm s / R) (-B, 0, 1),
// R = s0 + (s1 - s0) lam, components ordered (dir, ia, ib): two divisions
// and one square root per point instead of nine divisions.  Written with
// compile-time component indices only: runtime-indexed private arrays would
// live in scratch memory.
__device__ __forceinline__ void shell_dXdx(int dom, double s0, double s1, const double X[3],
                                           double M[3][3]) {
  const double lam = X[0], A = X[1], B = X[2];
  const double pm = (dom & 1) ? 1.0 : -1.0;
  const double s = sqrt(1.0 + A * A + B * B);
  const double c0 = pm / ((s1 - s0) * s);
  const double c1 = pm * s / (s0 + (s1 - s0) * lam);
  const int dir = dom >> 1;
  const int ia = (dir == 1) ? 0 : 1;      // axis scaled by A
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const bool isr = (d == dir), isa = (d == ia);
    M[0][d] = isr ? c0 : (isa ? A * c0 : B * c0);
    M[1][d] = isr ? -A * c1 : (isa ? c1 : 0.0);
    M[2][d] = isr ? -B * c1 : (isa ? 0.0 : c1);
  }
}

// det of a 3x3 matrix (cofactor expansion along the first row)
__device__ __forceinline__ double det3(const double M[3][3]) {
  return M[0][0] * (M[1][1] * M[2][2] - M[1][2] * M[2][1]) -
         M[0][1] * (M[1][0] * M[2][2] - M[1][2] * M[2][0]) +
         M[0][2] * (M[1][0] * M[2][1] - M[1][1] * M[2][0]);
}

// What stage_in and stage_out take of a stage's arguments (kernels.h).
struct StageRegs {
  const double *win, *U, *Wa, *Wb;
  double cA, cW;
  int wmode;
};

// The operands of stage_out at one node.
struct StageIn {
  double U[5], a[4], b[4];
};

// Stages without an accumulator (wmodes 3 to 6), for right-hand sides in
// which phi does not appear.  An RK step keeps its stage inputs W1, W2, ..
// instead of accumulating u + sum_s b_s dt r_s, and the last stage recovers
// the earlier r_s from them:
//   RK4     W1 = U + dt/2 r1, W2 = U + dt/2 r2, W3 = U + dt r3, so the step
//           ends at U + ((W1 - U) + 2 (W2 - U) + (W3 - U))/3 + dt/6 r4;
//   sspRK3  W1 = U + dt r1, W2 = 0.75 U + 0.25 (W1 + dt r2), so it ends at
//           U + 2/3 ((W2 - U) + dt r3).
// phi is in no right-hand side and r_phi = pi, so its stage values are not
// kept: the last stage sums the stages' pi.  Per RK4 step and node that is
// 8 + 12 + 12 + 22 doubles moved instead of 15 + 25 + 25 + 15 (sspRK3: 8 +
// 12 + 15 instead of 15 + 25 + 15), and the state is stepped in place: the
// last stage reads U at its own nodes only.  W - U is exact where W is near
// U, so a step has the rounding of the stage inputs, thirds of ulps, and of
// one sum, where the accumulator had one rounding per stage.
// gi: the node's first state double; vo: the offsets of pi and c, in the
// order they are handed over; po: phi's.
template <class O>
__device__ __forceinline__ void stage_in(const O &o, long gi, const int (&vo)[4], int po, StageIn &q) {
  if (o.wmode <= 4) {
    if (o.U != o.win) {
#pragma unroll
      for (int v = 0; v < 4; ++v) q.U[v] = o.U[gi + vo[v]];
    }
  } else {
#pragma unroll
    for (int v = 0; v < 4; ++v) q.U[v] = o.U[gi + vo[v]];
    q.U[4] = o.U[gi + po];
    q.a[0] = o.Wa[gi + vo[0]];
    if (o.wmode == 5) {
#pragma unroll
      for (int v = 1; v < 4; ++v) q.a[v] = o.Wa[gi + vo[v]];
#pragma unroll
      for (int v = 0; v < 4; ++v) q.b[v] = o.Wb[gi + vo[v]];
    }
  }
}
template <class O>
__device__ __forceinline__ void stage_in(const O &o, long gi, int np3, StageIn &q) {
  const int vo[4] = {0, np3, 2 * np3, 3 * np3};
  stage_in(o, gi, vo, 4 * np3, q);
}

// own: the stage input's pi and c at the node; r: their RHS.  PHI: the
// system has r_phi = pi (else phi is left as it is).  Outputs in out[0..3],
// and phi in out[4] when the step ends (returns true then).
template <bool PHI, class O>
__device__ __forceinline__ bool stage_out(const O &o, const StageIn &q, const double own[4], const double r[4],
                                          double out[5]) {
  if (o.wmode == 3) {
    if (o.U == o.win) {
#pragma unroll
      for (int v = 0; v < 4; ++v) out[v] = own[v] + o.cW * r[v];
    } else {
#pragma unroll
      for (int v = 0; v < 4; ++v) out[v] = q.U[v] + o.cW * r[v];
    }
    return false;
  }
  if (o.wmode == 4) {
#pragma unroll
    for (int v = 0; v < 4; ++v) out[v] = 0.75 * q.U[v] + 0.25 * (own[v] + o.cW * r[v]);
    return false;
  }
  if (o.wmode == 5) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const double s = (q.a[v] - q.U[v]) + 2. * (q.b[v] - q.U[v]) + (own[v] - q.U[v]);
      out[v] = q.U[v] + (s * (1. / 3.) + o.cA * r[v]);
    }
    if (PHI) out[4] = q.U[4] + o.cA * (q.U[0] + 2. * (q.a[0] + q.b[0]) + own[0]);
    return PHI;
  }
#pragma unroll
  for (int v = 0; v < 4; ++v) out[v] = q.U[v] + (2. / 3.) * ((own[v] - q.U[v]) + o.cW * r[v]);
  if (PHI) out[4] = q.U[4] + o.cA * (q.U[0] + q.a[0] + 4. * own[0]);
  return PHI;
}

// outward unit normal and lift scale sqrtgdiag / w_end of face f at a node
// with metric M (dX/dx; unused on Cartesian elements, GEOM 0), as the
// stage kernels compute them (dg.c:90-146, utilities.c:48-81)
template <int GEOM>
__device__ __forceinline__ void face_normal(const double M[3][3], const double *dXbdX, int f,
                                            double wend_inv, double nrm[3], double &scale) {
  const int dir = f >> 1;
  const double sig = (f & 1) ? 1.0 : -1.0;
  if (GEOM == 0) {
    nrm[0] = (dir == 0) ? sig : 0.0;
    nrm[1] = (dir == 1) ? sig : 0.0;
    nrm[2] = (dir == 2) ? sig : 0.0;
    scale = dXbdX[dir] * wend_inv;
  } else {
    const double r0 = (dir == 0) ? M[0][0] : (dir == 1) ? M[1][0] : M[2][0];
    const double r1 = (dir == 0) ? M[0][1] : (dir == 1) ? M[1][1] : M[2][1];
    const double r2 = (dir == 0) ? M[0][2] : (dir == 1) ? M[1][2] : M[2][2];
    const double s = sqrt(r0 * r0 + r1 * r1 + r2 * r2);
    const double ism = 1.0 / (sig * s);
    nrm[0] = r0 * ism; nrm[1] = r1 * ism; nrm[2] = r2 * ism;
    scale = dXbdX[dir] * s * wend_inv;
  }
}

}  // namespace nmx
