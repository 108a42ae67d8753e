// fvelm_stage.h -- scalarwave1 RHS + RK stage on FV elements (uniform points
// including both faces) of a Cartesian or CubedShell mesh, gfx950.
// Instantiated by fvelm_kernels.hip (dnfn_extrap1 and fv_rec without the
// s1/s2/opt limits) and fvelm_ex_kernels.hip (with them), which compile in
// parallel.
//
// nmesh's fv_divf (src/main/dg/fv.c:115-624) with scalarwave1's callbacks
// (src/tests/scalarwave1/scalarwave1.c:211-237,755-790) and its default
// parameters (src/main/dg/nmesh_dg.c:26-66, dg.c:285-400): fv_flux = fnum,
// fv_divf_extrap = dnfn_extrap1 (so the face fluxes are set here and
// dg_add_surface_fluxes adds nothing), fv_divf_use_only_right_flux = yes,
// WENOm3 optimal weights (1, 2).  Per element:
//   own pi, c to LDS in one coalesced pass, the adjacent face values to the
//     line that ends there;
//   the three directions side by side, one lane per line: reconstruct every
//     midpoint from both sides (WENOm5, WENOmZ, WENOmT or WENOm3, rec1d.c:
//     115-232,875-1370,1412-1798), take upwind / LLF fnum with the midpoint
//     normal, the face fluxes against ajsurf at both ends, df_i = Jg_R fnumR_i
//     - Jg_L fnumR_{i-1} with Jg = sqrtgdiag / (ooJ dXb_i), dnfn_extrap1 at
//     both ends (rec1d.c:542-626) and divf_d = df ooJ into LDS;
//   r_{pi,c} = -(divf_x + divf_y + divf_z), r_phi = pi, the RK stage.
// A line's midpoints are unrolled, one code for the three directions.  The
// reconstructions are those of the reference in differences of neighbouring
// points: the nonlinear weights of a point's three stencils serve the midpoint
// on its left from the right and the one on its right from the left, so their
// products are computed once; they are normalised with one reciprocal.  Only
// rounding differs from the reference's per-weight divisions.
// The upwind fnum of a face acts on c along its normal only, so components of
// c that a direction's normal has none of are not reconstructed there: of pi
// and c, 2 variables per direction on boxes, and 4, 3 and 3 on shells.
//
// What bounds it: on many elements the FP64 VALU and HBM alike (4096 box
// elements of 8^3 points, WENO5: 62 us a stage, about 45 us of memory traffic
// at the rate of a large copy and 38 us of arithmetic at the rate of a large
// FP64 product), on few the chain load - line - store (192 shell elements of
// 6^3 points: 9 us).  With the directions one after another on one group of
// lanes, each line streamed from HBM through a sliding window and every
// weight computed twice, these were 150 and 39 us; with the sums in
// differences and the fields in LDS, but the directions still in turn and all of
// c held, 8 steps of the box took 4.23 ms (side by side 2.92, with the needed
// components alone 2.13) and 16 steps of the shell with its DG elements 1.87
// (1.40).  Of 10^3 points: 9.50 ms for 8 steps in turn, 6.55 side by side,
// though only two workgroups then fit a CU's LDS.
#pragma once
#include <hip/hip_runtime.h>

#include "amr.h"
#include "dg_common.h"
#include "dg_stage.h"
#include "fastmath.h"

namespace nmx {

constexpr double kWeno3Eps = 1e-6 / 36.;    // WENO3_epsilon (rec1d.c:35), u_scale = 1, over 36
constexpr double kWeno5EpsE = 1e-40 / 9.;   // WENO5_epsilon (rec1d.c:1193) over 9

// The differences are h_k = (u[k+1] - u[k])/6.  A smoothness indicator of the
// stencil with differences (p, q), by the position of the midpoint it
// reconstructs (right end, centre, left end), is 9 times
//   13/3 (q - p)^2 + (3 q - p)^2, (p + q)^2 or (q - 3 p)^2;
// weights depend on ratios only, so the factor goes into the epsilon.
__device__ __forceinline__ double fve_curv(double p, double q) {
  const double s = q - p;
  return fma(13. / 3. * s, s, kWeno5EpsE);
}
// the unnormalised weights of the stencils (h0, h1), (h1, h2), (h2, h3) before
// the ideal weights, E[1] times 6: WENO5 (REC 5) 1 / b_k^2, WENOT (9: (1 + |b0 -
// b2|) / b_k normalises to 1 / b_k) and WENO-Z (7) 1 + |b0 - b2| / b_k, times
// the product that clears the denominators
template <int REC>
__device__ __forceinline__ void fve_weights(double h0, double h1, double h2, double h3, double (&E)[3]) {
  const double s0 = fma(3., h1, -h0), s1 = h1 + h2, s2 = fma(-3., h2, h3);
  double e0 = fma(s0, s0, fve_curv(h0, h1)), e1 = fma(s1, s1, fve_curv(h1, h2)), e2 = fma(s2, s2, fve_curv(h2, h3));
  const double tau = REC == 7 ? fabs(e0 - e2) : 0.0;
  if (REC == 5) { e0 *= e0; e1 *= e1; e2 *= e2; }
  E[0] = e1 * e2;
  E[1] = 6. * (e0 * e2);
  E[2] = e0 * e1;
  if (REC == 7) { E[0] *= e0 + tau; E[1] *= e1 + tau; E[2] *= e2 + tau; }
}
// midpoint right of u from the left, ideal weights (1, 6, 3), and left of u
// from the right, (3, 6, 1); h0 .. h3 the differences around u
__device__ __forceinline__ double fve_left(double u, double h0, double h1, double h2, double h3, const double (&E)[3]) {
  const double E2 = 3. * E[2];
  const double q = E[0] * fma(5., h1, -2. * h0) + E[1] * fma(2., h2, h1) + E2 * fma(4., h2, -h3);
  return fma(q, rcp_nr(E[0] + E[1] + E2), u);
}
__device__ __forceinline__ double fve_right(double u, double h0, double h1, double h2, double h3, const double (&E)[3]) {
  const double E0 = 3. * E[0];
  const double q = E0 * fma(-4., h1, h0) - E[1] * fma(2., h1, h2) + E[2] * fma(2., h3, -5. * h2);
  return fma(q, rcp_nr(E0 + E[1] + E[2]), u);
}
// WENOm3: the midpoint beyond u from the differences on its far side (hf) and
// across the midpoint (hm), ideal weights 1 and 2, towards u + 3 ...
__device__ __forceinline__ double fve_weno3(double hf, double hm) {
  const double bf = fma(hf, hf, kWeno3Eps), bm = fma(hm, hm, kWeno3Eps);
  const double wf = bm * bm, wm = 2. * (bf * bf);
  return 3. * fma(wf, hf, wm * hm) * rcp_nr(wf + wm);
}

// fv_divf_extrap_s1, _s2, _opt of dnfn_extrap1 (fv.c:147-150, 558-573)
// and the end-midpoint reconstruction of fv_rec (dg.c:295-326):
// recend 0 for the _2 modes (average of the two end points), 1 for the _1
// modes (the end point), 2 for WENOm3 / WENOm5 / WENOmZ (the average unless
// fv_rec_WENOm_s1 / _s2 / _opt take the end point, rec1d.c:1096-1186, which
// then also keeps that end's df from dnfn_extrap1, fv.c:45-79, 558-573)
struct FvEx {
  double s1, s2;
  int opt, on;   // on: s1 > 0 or s2 < DBL_MAX
  int recend;
  double rs1, rs2;
  int ropt, ron; // ron: fv_rec_WENOm_s1 > 0 or _s2 < DBL_MAX
  int first;     // fv_rec = 1: the point left / right of each midpoint (rec1d.c:16-27)
};

// rec at an end midpoint from the end point u0 and the next two inward
// (rec1d_p_WENOm3 / rec1d_m_WENOm3 with rec1d_u_in1_weightfac,
// rec1d.c:1096-1186; the _1 and _2 modes, rec1d.c:1032-1090, 909-1030);
// *kept: the end point itself was taken under the WENOm limit
template <bool EX>
__device__ __forceinline__ double rec_end(double u0, double u1, double u2, const FvEx &ex, bool *kept) {
  *kept = false;
  if (!EX || ex.recend == 0) return 0.5 * u0 + 0.5 * u1;
  if (ex.recend == 1) return u0;
  double w1fac = 1.;
  if (ex.ron) {
    const double d2 = u2 - u1, d1 = u1 - u0;
    const double s = fabs(d1) / (fabs(d2) + 1e-100);
    if (s < ex.rs1 || s >= ex.rs2) w1fac = 0.;
    if (ex.ropt == -1) w1fac = 0.;
    else if (ex.ropt == 1 && d1 * d2 <= 0.) w1fac = 0.;
    else if (ex.ropt == 2 && d1 * d2 >= 0.) w1fac = 0.;
  }
  const double w1 = 0.5 * w1fac, w0 = 1. - w1;
  const double r = w0 * u0 + w1 * u1;
  *kept = ex.ron && r == u0;   // fv_stat_WENOm_1or2: the rec equals the end point
  return r;
}

// The face value of df from the end value u0 and the next two inward, u1
// and u2 (rec1d_compute_1s1_u with forward = 0, rec1d.c:542-609): u0 sits a
// quarter spacing inside the face, so u_face = u0 / 0.75 + (1 - 1 / 0.75) u1,
// unless s = (4/3)|u1 - u0| / |u2 - u1| falls outside [s1, s2) or opt says
// otherwise, which keeps u0 (0th order).
template <bool EX>
__device__ __forceinline__ double fv_extrap1(double u0, double u1, double u2, const FvEx &ex) {
  double w0 = 1. / 0.75;
  double w1 = 1. - w0;
  if (EX && ex.on) {
    const double d2 = u2 - u1, d1 = u1 - u0;
    const double s = 1.3333333333 * fabs(d1) / (fabs(d2) + 1e-100);
    if (s < ex.s1 || s >= ex.s2) w1 = 0.;
    if (ex.opt == -1) w1 = 0.;
    else if (ex.opt == 1 && d1 * d2 <= 0.) w1 = 0.;
    else if (ex.opt == 2 && d1 * d2 >= 0.) w1 = 0.;
    w0 = 1. - w1;
  }
  return w0 * u0 + w1 * u1;
}

// Place of point (i, j, k) in an LDS field: rows along i of odd stride, or for
// 8 points rows permuted, so that the lanes of a sweep in any direction spread
// over the banks; for 10 points rows of 10, whose two-way conflicts cost less
// than a workgroup per CU (4096 box elements: 6.55 ms for 8 steps, 6.86 with
// rows of 11).
constexpr int fve_stride(int np) { return np == 8 || np == 10 ? np : np | 1; }
constexpr int fve_field(int np) { return fve_stride(np) * np * np; }
template <int NP>
__device__ __forceinline__ int fve_at(int i, int j, int k) {
  if (NP == 8) return (i ^ k) + 8 * (((j + k) & 7) + 8 * k);
  return i + fve_stride(NP) * (j + NP * k);
}

// LDS fields of the directions' divf: direction d has variables of its own
// fluxes only, so on boxes with upwind fluxes pi and c_d, and on shells pi, c_r
// and for d > 0 its own axis' c (all four for d = 0).
template <int GEOM, bool LLF>
__host__ __device__ constexpr int fve_slots(int d) { return LLF ? 4 : GEOM == 0 ? 2 : d == 0 ? 4 : 3; }
template <int GEOM, bool LLF>
constexpr int fve_slabs() { return LLF ? 12 : GEOM == 0 ? 6 : 10; }
template <int GEOM, bool LLF>
__device__ __forceinline__ int fve_slab(int d, int slot) {
  return LLF ? 4 * d + slot : GEOM == 0 ? 2 * d + slot : d == 0 ? slot : 1 + 3 * d + slot;
}

// One direction d of the element, one lane per line at (la, lb) (along the
// other two directions in order), points s = 0 .. NP-1.  The variables are held
// in slots: 0 pi; on boxes 1 c along d; on shells 1 c_r, then c along d's own
// axis for d > 0 (all three matter for d = 0).  lo, hi: the adjacent values at
// the line's ends, fields in the order of s_u.  Writes divf_d into d's fields of
// acc, in the order of the slots.
template <int NP, int REC, int GEOM, bool EX, bool LLF>
__device__ __forceinline__ void fve_sweep(const AmrArgs &a, const NMX_CONST SlotRec &R, const double *wc,
                                          const FvEx &ex, int d, int la, int lb, const double lo[4],
                                          const double hi[4], const double (*s_u)[fve_field(NP)],
                                          double (*acc)[fve_field(NP)]) {
  static_assert(NP >= 3, "FV lines have at least 3 points");
  auto at = [&](int s) {
    return d == 0 ? fve_at<NP>(s, la, lb) : d == 1 ? fve_at<NP>(la, s, lb) : fve_at<NP>(la, lb, s);
  };
  const int d1 = d == 2 ? 0 : d + 1, d2 = d == 0 ? 2 : d - 1;
  const int sl[4] = {0, GEOM == 0 ? 1 + d : 1, GEOM == 0 ? 1 + d1 : d == 2 ? 3 : 2, GEOM == 0 ? 1 + d2 : d == 2 ? 2 : 3};
  constexpr int NA = GEOM == 0 && !LLF ? 2 : 4;      // slots held
  const bool llf = LLF && (!EX || a.numflux != 0);   // EX: either flux
  const int na = fve_slots<GEOM, LLF>(d);
  const NMX_CONST double *xb = as_const(a.xb);

  // ---- metric ----
  // Boxes: Jg = dXb/dX[d] / ooJ constant.  Shells (NodeGeo, dg_stage.h): with t =
  // s^2 = 1 + A^2 + B^2, sqrtgdiag / ooJ = dXb/dX[d] |dX_d/dx| / ooJ is K R^2 along
  // lam and K (1 + a^2)^(1/2) / t along A or B (a the coordinate along the line),
  // ooJ = K' / R^2 or K' t^(3/2), and the normal pm (1, A, B)/s or pm (-a, 1)/(1 +
  // a^2)^(1/2) (coordinates.c:133-224,284-415,728-802; utilities.c:48-81).
  const double gd = d == 0 ? R.dXbdX[0] : d == 1 ? R.dXbdX[1] : R.dXbdX[2];
  const double detb = R.dXbdX[0] * R.dXbdX[1] * R.dXbdX[2];
  double K = gd / detb, Kp = detb, b2 = 0, pm = 1, nc[3] = {1, 0, 0};
  const double c0 = d == 0 ? R.bb[0] : d == 1 ? R.bb[2] : R.bb[4], c1 = d == 0 ? R.bb[1] : d == 1 ? R.bb[3] : R.bb[5];
  const double cm = 0.5 * (c1 + c0), ch = 0.5 * (c1 - c0);
  if (GEOM == 2) {
    pm = (R.dom & 1) ? 1.0 : -1.0;
    const double dr = R.s1 - R.s0;
    if (d == 0) {
      const double A = patch_coord(R, 1, xb[la]), B = patch_coord(R, 2, xb[lb]);
      const double t = 1. + A * A + B * B, rs = rsqrt_nr(t);
      K = R.dXbdX[0] * (rs * rs * rs) / detb;
      Kp = detb / dr * (t * t * rs);
      nc[0] = pm * rs; nc[1] = A * nc[0]; nc[2] = B * nc[0];
    } else {
      const double r = R.s0 + dr * patch_coord(R, 0, xb[la]);
      const double b = d == 1 ? patch_coord(R, 2, xb[lb]) : patch_coord(R, 1, xb[lb]);
      b2 = 1. + b * b;
      K = gd * r * dr / detb;
      Kp = detb / (dr * r * r);
    }
  }
  // at element coordinate x along the line: sqrtgdiag / ooJ and the normal, and ooJ
  auto flux_metric = [&](double x, double &soj, double n[3]) {
    soj = K;
    n[0] = nc[0]; n[1] = nc[1]; n[2] = nc[2];
    if (GEOM == 2) {
      const double c = fma(ch, x, cm);
      if (d == 0) {
        const double r = R.s0 + (R.s1 - R.s0) * c;
        soj = K * (r * r);
      } else {
        const double t = fma(c, c, 1.), ra = rsqrt_nr(t);
        soj = K * (t * ra) * rcp_nr(fma(c, c, b2));
        n[0] = -pm * c * ra; n[1] = pm * ra;
      }
    }
  };
  auto node_ooJ = [&](double x) {
    if (GEOM == 0) return Kp;
    const double c = fma(ch, x, cm);
    if (d == 0) {
      const double ir = rcp_nr(R.s0 + (R.s1 - R.s0) * c);
      return Kp * (ir * ir);
    }
    const double t = fma(c, c, b2);
    return Kp * (t * t * rsqrt_nr(t));
  };

  // fnum = f(ui).n + F(ui - ua) for a unit normal n (scalarwave1 fluxes,
  // scalarwave1.c:39-48; F as in face_flux)
  auto fnum = [&](const double n[3], const double ui[4], const double ua[4], double fn[4]) {
    double un, dn;
    if (GEOM == 0) {
      un = n[0] * ui[1];
      dn = n[0] * (ui[1] - ua[1]);
    } else {
      un = n[0] * ui[1] + n[1] * ui[2];
      dn = n[0] * (ui[1] - ua[1]) + n[1] * (ui[2] - ua[2]);
      if (d == 0) {
        un += n[2] * ui[3];
        dn += n[2] * (ui[3] - ua[3]);
      }
    }
    const double dp = ui[0] - ua[0];
    const double Fp = 0.5 * (dp + dn);
    fn[0] = Fp - un;
    if (!llf) {
      const double G = Fp - ui[0];
#pragma unroll
      for (int q = 0; q < 3; ++q) fn[1 + q] = n[q] * G;
    } else {
#pragma unroll
      for (int q = 0; q < 3; ++q) fn[1 + q] = 0.5 * ((ui[1 + q] - ua[1 + q]) + n[q] * dp) - n[q] * ui[0];
    }
  };

  double u[NA][NP], h[NA][NP], E[NA][3], dd[NA][NP];
  bool keepL[4] = {false, false, false, false}, keepR[4] = {false, false, false, false};
  double loS[4], hiS[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    loS[v] = sl[v] == 0 ? lo[0] : sl[v] == 1 ? lo[1] : sl[v] == 2 ? lo[2] : lo[3];
    hiS[v] = sl[v] == 0 ? hi[0] : sl[v] == 1 ? hi[1] : sl[v] == 2 ? hi[2] : hi[3];
  }
  auto load = [&](int s) {
    const int p = at(s);
#pragma unroll
    for (int v = 0; v < NA; ++v) {
      u[v][s] = v < na ? s_u[sl[v]][p] : 0.0;
      if (s > 0) h[v][s - 1] = (u[v][s] - u[v][s - 1]) * (1. / 6.);
    }
  };
#pragma unroll
  for (int s = 0; s < (NP < 4 ? NP : 4); ++s) load(s);
  double fL[4], fR[4], sojL = 0, dL[4], dR[4];
#pragma unroll
  for (int i0 = 0; i0 < NP; ++i0) {
    if (i0 + 4 < NP) load(i0 + 4);
    double sojR, nR[3];
    const bool mid = GEOM == 2 && a.fv_mid && i0 < NP - 1;
    flux_metric(mid ? 0.5 * (xb[i0] + xb[i0 + 1 < NP ? i0 + 1 : i0]) : xb[i0], sojR, nR);
    if (i0 == 0) {
      double n0[3];
      if (GEOM == 2) {
        flux_metric(xb[0], sojL, n0);
      } else {
        sojL = sojR;
        n0[0] = nR[0]; n0[1] = nR[1]; n0[2] = nR[2];
      }
      const double nL[3] = {-n0[0], -n0[1], -n0[2]};
      double ue[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) ue[v] = v < NA ? u[v % NA][0] : 0.0;
      fnum(nL, ue, loS, fL);
    } else {
#pragma unroll
      for (int l = 0; l < 4; ++l) fL[l] = -fR[l];
    }
    double ui[4], ua[4];
    if (i0 < NP - 1) {
      // both sides of the midpoint between points i0 and i0 + 1
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        ui[v] = ua[v] = 0.0;
        if (v >= NA || v >= na) continue;
        if (EX && ex.first) {
          ui[v] = u[v][i0];
          ua[v] = u[v][i0 + 1];
          continue;
        }
        if (REC != 3 && i0 >= 2 && i0 <= NP - 3)
          ui[v] = fve_left(u[v][i0], h[v][i0 - 2], h[v][i0 - 1], h[v][i0], h[v][i0 + 1], E[v]);
        else if (i0 >= 1) ui[v] = u[v][i0] + fve_weno3(h[v][i0 - 1], h[v][i0]);
        else ui[v] = rec_end<EX>(u[v][0], u[v][1], u[v][2], ex, &keepL[v]);
        if (REC != 3 && i0 >= 1 && i0 <= NP - 4) {
          // the weights around point i0 + 1, for its left and its right midpoint
          fve_weights<REC>(h[v][i0 - 1], h[v][i0], h[v][i0 + 1], h[v][i0 + 2], E[v]);
          ua[v] = fve_right(u[v][i0 + 1], h[v][i0 - 1], h[v][i0], h[v][i0 + 1], h[v][i0 + 2], E[v]);
        } else if (i0 <= NP - 3) ua[v] = u[v][i0 + 1] - fve_weno3(h[v][i0 + 1], h[v][i0]);
        else ua[v] = rec_end<EX>(u[v][NP - 1], u[v][NP - 2], u[v][NP - 3], ex, &keepR[v]);
      }
    } else {
#pragma unroll
      for (int v = 0; v < 4; ++v) { ui[v] = v < NA ? u[v % NA][i0] : 0.0; ua[v] = hiS[v]; }
    }
    fnum(nR, ui, ua, fR);
    const double iwc = rcp_nr(as_const(wc)[i0]);
    const double JR = sojR * iwc, JL = sojL * iwc;
    sojL = sojR;
#pragma unroll
    for (int l = 0; l < NA; ++l) dd[l][i0] = JR * fR[l] + JL * fL[l];
    if (i0 == 2) {
      // the left end (rec1d_LR_uface_to_uin_1_Carray, left first)
#pragma unroll
      for (int l = 0; l < NA; ++l)
        dL[l] = (EX && keepL[l]) ? dd[l][0] : fv_extrap1<EX>(dd[l][0], dd[l][1], dd[l][2], ex);
    }
    if (i0 == NP - 1) {
      // the right end; with 3 points its inner neighbours are point 1 and the
      // extrapolated point 0
#pragma unroll
      for (int l = 0; l < NA; ++l)
        dR[l] = (EX && keepR[l]) ? dd[l][NP - 1]
                                 : fv_extrap1<EX>(dd[l][NP - 1], dd[l][NP - 2], NP == 3 ? dL[l] : dd[l][NP - 3], ex);
    }
    auto put = [&](int s, const double *val, int stride) {
      const int p = at(s);
      const double oj = node_ooJ(xb[s]);
#pragma unroll
      for (int l = 0; l < NA; ++l)
        if (l < na) acc[fve_slab<GEOM, LLF>(d, l)][p] = val[l * stride] * oj;
    };
    if (i0 == 2) put(0, dL, 1);
    if (i0 >= 1 && i0 < NP - 1) put(i0, &dd[0][i0], NP);
    if (i0 == NP - 1) put(NP - 1, dR, 1);
  }
}

// Lanes of one direction; the three directions run side by side.
constexpr int fve_line_threads(int np) { return (np * np + 63) / 64 * 64; }

template <int NP, int REC, int GEOM, bool EX, bool LLF>
__global__ __launch_bounds__(3 * fve_line_threads(NP), 2) void fvelm_kernel(AmrArgs a, const double *wc) {
  constexpr int NP2 = NP * NP;
  constexpr int NP3 = NP * NP * NP;
  constexpr int NL = fve_line_threads(NP), NT = 3 * NL;
  constexpr int NC = (NP3 + NT - 1) / NT;
  constexpr int F = fve_field(NP);
  __shared__ double s_u[4][F];
  __shared__ double acc[fve_slabs<GEOM, LLF>()][F];
  const int it = xcd_block(a.nlist, a.xcd_map);
  if (it >= a.nlist) return;
  const NMX_CONST SlotRec &R = as_const(a.rec)[it];
  const int tid = threadIdx.x;
  const long gbase = 5 * R.noff;
  int cmp[4], vo[4];
  node_cmp<GEOM>(R, cmp);
#pragma unroll
  for (int v = 0; v < 4; ++v) vo[v] = cmp[v] * NP3;
  const FvEx ex = {a.ex_s1, a.ex_s2, a.ex_opt, a.ex_on, a.recend, a.rec_s1, a.rec_s2, a.rec_opt, a.rec_on, a.rec_first};

  // own fields and the line's faces; lanes past the last node or line repeat it
  double own[NC][4];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int node = min(tid + c * NT, NP3 - 1);
#pragma unroll
    for (int v = 0; v < 4; ++v) own[c][v] = a.win[gbase + node + vo[v]];
  }
  const int d = __builtin_amdgcn_readfirstlane(tid / NL);
  const int line = min(tid % NL, NP2 - 1);
  const int la = line % NP, lb = line / NP;
  double lo[4], hi[4];
  stage_face<NP>(a, R, 2 * d, line, la, lb, cmp, lo);
  stage_face<NP>(a, R, 2 * d + 1, line, la, lb, cmp, hi);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int node = min(tid + c * NT, NP3 - 1);
    const int p = fve_at<NP>(node % NP, (node / NP) % NP, node / NP2);
#pragma unroll
    for (int v = 0; v < 4; ++v) s_u[v][p] = own[c][v];
  }
  __syncthreads();
  if (tid % NL < NP2) fve_sweep<NP, REC, GEOM, EX, LLF>(a, R, wc, ex, d, la, lb, lo, hi, s_u, acc);
  // r_{pi,c} = -divf, r_phi = pi, the RK stage; the next node's registers
  // requested a node ahead, but for the operands of stages with an accumulator,
  // whose loop of its own leaves the other's registers as they are
  const StageRegs o = {a.win, a.U, a.Wa, a.Wb, a.cA, a.cW, a.wmode};
  StageIn in;
  if (a.wmode >= 3 && tid < NP3) node_in(a, o, gbase + tid, vo, 4 * NP3, in);
  __syncthreads();
  auto rhs_at = [&](int node, double u[4], double r[4]) {
    const int p = fve_at<NP>(node % NP, (node / NP) % NP, node / NP2);
#pragma unroll
    for (int v = 0; v < 4; ++v) u[v] = s_u[v][p];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      double div = 0;
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        // field v's slot in direction e
        const int slot = v == 0 || (GEOM == 2 && (v == 1 || e < 2)) ? v : GEOM == 2 ? 5 - v : 1 + (v + 2 - e) % 3;
        if (slot < fve_slots<GEOM, LLF>(e)) div += acc[fve_slab<GEOM, LLF>(e, slot)][p];
      }
      r[v] = -div;
    }
  };
  if (a.wmode < 3) {
#pragma unroll 1
    for (int node = tid; node < NP3; node += NT) {
      AccIn q;
      double u[4], r[4];
      node_in(a, o, gbase + node, vo, 4 * NP3, q);
      rhs_at(node, u, r);
      node_out(a, o, q, gbase + node, vo, 4 * NP3, u, r);
    }
    return;
  }
#pragma unroll 1
  for (int node = tid; node < NP3; node += NT) {
    double u[4], r[4];
    rhs_at(node, u, r);
    const StageIn q = in;
    if (node + NT < NP3) node_in(a, o, gbase + node + NT, vo, 4 * NP3, in);
    node_out(a, o, q, gbase + node, vo, 4 * NP3, u, r);
  }
}

template <int NP, int REC, bool EX, bool LLF>
static hipError_t launch_fvelm_t(int geom, const AmrArgs &a, const double *wc, hipStream_t s) {
  const dim3 grid(a.xcd_map ? 8 * ((a.nlist + 7) / 8) : a.nlist), block(3 * fve_line_threads(NP));
  if (geom == 0)
    hipLaunchKernelGGL((fvelm_kernel<NP, REC, 0, EX, LLF>), grid, block, 0, s, a, wc);
  else
    hipLaunchKernelGGL((fvelm_kernel<NP, REC, 2, EX, LLF>), grid, block, 0, s, a, wc);
  return hipGetLastError();
}

// the FV launch of one variant: EX with the s1/s2/opt limits (and LLF, which
// then serves both fluxes), LLF with the LLF flux
template <bool EX, bool LLF>
static hipError_t launch_fvelm_v(int np, int rec, int geom, const AmrArgs &a, const double *wc, hipStream_t s) {
  if (a.nlist <= 0) return hipSuccess;
#define NMX_CASE(N)                                                                 \
  case N:                                                                           \
    return rec == 5   ? launch_fvelm_t<N, 5, EX, LLF>(geom, a, wc, s)               \
           : rec == 7 ? launch_fvelm_t<N, 7, EX, LLF>(geom, a, wc, s)               \
           : rec == 9 ? launch_fvelm_t<N, 9, EX, LLF>(geom, a, wc, s)               \
                      : launch_fvelm_t<N, 3, EX, LLF>(geom, a, wc, s);
  switch (np) {
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

// defined in fvelm_ex_kernels.hip and fvelm_llf_kernels.hip
hipError_t launch_fvelm_ex(int np, int rec, int geom, const AmrArgs &a, const double *wc, hipStream_t s);
hipError_t launch_fvelm_llf(int np, int rec, int geom, const AmrArgs &a, const double *wc, hipStream_t s);

}  // namespace nmx
