// fv_kernels.hip -- FV WENO5 + LLF for special-relativistic Euler (ideal
// gas) on a periodic grid of 16^3-cell blocks, gfx950, FP64.
//
// fv_stage_kernel, once per RK stage: one 64-lane wave per 8^3-cell tile and
// direction.  A lane walks one line of the tile along the direction with a
// window of primitives in registers, reconstructs both face states with WENO5
// (rec1d_p_WENO5 / rec1d_m_WENO5 with uniform weights, rec1d.c:1190-1352,
// u_scale = 1 as in fv.c:141), takes the LLF flux (numflux1d.c:85-112) and
// accumulates the flux difference of each cell in LDS; the epilogue applies
// the RK stage combination (RungeKutta.c:19-188) and solves for the next
// stage's primitives (rho, v, p): Newton on the pressure, guessed from this
// stage's value.  fv_c2p_kernel does that solve alone, before the first stage.
// The WENO5 formulas are the reference's in differences of neighbouring cells
// (weno5_*, below).
// The SR-Euler flux, eigenvalues and c2p are textbook (Marti & Mueller,
// Living Rev. Relativ. 6 (2003) 7); the reference has no SR-Euler system.
#include <hip/hip_runtime.h>

#include "fastmath.h"
#include "fv.h"

namespace nmx {

constexpr int kFvB = 16;                     // cells per block edge
constexpr int kFvB3 = kFvB * kFvB * kFvB;
constexpr int kFvT = 8;                      // cells per tile edge
constexpr int kFvT3 = kFvT * kFvT * kFvT;
constexpr int kC2pMaxIt = 100;
// up to this many tiles a tile gets three waves (fv_stage_kernel): sspRK3 and
// RK4 steps of 48^3 cells (216 tiles) take 107 us with three and 187 with one,
// of 64^3 (512) 185 and 234, of 96^3 (1728) 622 and 611, of 256^3 6.21 and
// 5.94 ms
constexpr int kFvSplitTiles = 1024;

// WENO5 in the differences h_k = (u[k+1] - u[k])/6 of neighbouring cells.  A
// smoothness indicator of the stencil with differences (p, q) by the position
// of the midpoint it reconstructs (right end: role 0, centre 1, left end 2;
// rec1d.c:1195-1300) is 9 times
//   13/3 (q - p)^2 + (3 q - p)^2, (p + q)^2 or (q - 3 p)^2,
// and the weights depend only on the indicators' ratios, so the factor goes
// into the epsilon (1e-40 over 9).  The first term is shared by the three
// roles a stencil takes at successive midpoints; the squared indicators E of a
// midpoint's right side are those of the next one's left side, so their
// products are kept.  Normalised with one reciprocal: the weights g_k / E_k
// over their sum equal g_k prod_{j != k} E_j over theirs (for the data here
// every product stays between 1e-170 and 1e+60).
constexpr double kWeno5Eps = 1e-40 / 9.;

__device__ __forceinline__ double weno_curv(double p, double q) {
  const double s = q - p;
  return fma(13. / 3. * s, s, kWeno5Eps);
}
// the products E1 E2, 6 E0 E2, E0 E1 of the stencils (h0, h1), (h1, h2), (h2,
// h3) with curvature terms c0, c1, c2
__device__ __forceinline__ void weno_products(double h0, double h1, double h2, double h3, double c0, double c1,
                                              double c2, double (&E)[3]) {
  const double s0 = fma(3., h1, -h0), s1 = h1 + h2, s2 = fma(-3., h2, h3);
  double e0 = fma(s0, s0, c0), e1 = fma(s1, s1, c1), e2 = fma(s2, s2, c2);
  e0 *= e0; e1 *= e1; e2 *= e2;
  E[0] = e1 * e2;
  E[1] = 6. * (e0 * e2);
  E[2] = e0 * e1;
}
// midpoint right of u from its left side: ideal weights (1, 6, 3), h0 .. h3
// the differences from two cells left of u on
__device__ __forceinline__ double weno_left(double u, double h0, double h1, double h2, double h3,
                                            const double (&E)[3]) {
  const double E2 = 3. * E[2];
  const double q = E[0] * fma(5., h1, -2. * h0) + E[1] * fma(2., h2, h1) + E2 * fma(4., h2, -h3);
  return fma(q, rcp_nr(E[0] + E[1] + E2), u);
}
// midpoint left of u from its right side: ideal weights (3, 6, 1), h1 .. h4
// the differences from two cells left of u on
__device__ __forceinline__ double weno_right(double u, double h1, double h2, double h3, double h4,
                                             const double (&E)[3]) {
  const double E0 = 3. * E[0];
  const double q = E0 * fma(-4., h2, h1) - E[1] * fma(2., h2, h3) + E[2] * fma(2., h4, -5. * h3);
  return fma(q, rcp_nr(E0 + E[1] + E[2]), u);
}

__device__ __forceinline__ void sr_p2c(double gam, const double P[5], double U[5]) {
  const double rho = P[0], vx = P[1], vy = P[2], vz = P[3], p = P[4];
  const double v2 = vx * vx + vy * vy + vz * vz;
  const double W = 1. / sqrt(1. - v2);
  const double h = 1. + gam / (gam - 1.) * p / rho;
  const double rhW2 = rho * h * W * W;
  U[0] = rho * W;
  U[1] = rhW2 * vx;
  U[2] = rhW2 * vy;
  U[3] = rhW2 * vz;
  U[4] = rhW2 - p - U[0];
}

// flux along the normal, conserved state and max |acoustic eigenvalue| of P =
// (rho, v_n, v_t, v_t', p); v2 = v^2, g1 = gam / (gam - 1).  With w = rho h =
// rho + g1 p and a = gam p (c_s^2 = a / w) the eigenvalues
//   (v_n (1 - c_s^2) +- c_s sqrt((1 - v2) (1 - v2 c_s^2 - v_n^2 (1 - c_s^2)))) / (1 - v2 c_s^2)
// become (v_n (w - a) +- sqrt(a (1 - v2) (w - v2 a - v_n^2 (w - a)))) / (w - v2 a).
__device__ __forceinline__ double sr_flux(double gam, double g1, const double P[5], double v2, double F[5],
                                          double U[5]) {
  const double rho = P[0], vn = P[1], p = P[4];
  const double iW2 = 1. - v2;
  const double W = rsqrt_nr(iW2);
  const double w = fma(g1, p, rho);
  const double D = rho * W, q = w * (W * W), t = q - D;
  U[0] = D;
  U[1] = q * vn;
  U[2] = q * P[2];
  U[3] = q * P[3];
  U[4] = t - p;
  F[0] = D * vn;
  F[1] = fma(U[1], vn, p);
  F[2] = U[2] * vn;
  F[3] = U[3] * vn;
  F[4] = t * vn;
  const double a = gam * p, wa = w - a, den = fma(-v2, a, w);
  const double rad = a * iW2 * fma(-vn * vn, wa, den);
  const double root = rad * rsqrt_nr(rad + 1e-300);   // 0 at 0
  return fma(fabs(vn), wa, root) * rcp_nr(den);
}

__device__ __forceinline__ double speed2(const double P[5]) { return P[1] * P[1] + P[2] * P[2] + P[3] * P[3]; }

// ---------------------------------------------------------------------------
// c2p
// ---------------------------------------------------------------------------

// primitives of U, p the pressure guess; false if Newton did not converge
__device__ __forceinline__ bool sr_c2p(double gam, double tol, const double U[5], double p, double P[5]) {
  const double D = U[0], E = U[4] + D;
  const double S2 = U[1] * U[1] + U[2] * U[2] + U[3] * U[3];
  const double pmin = fmax(sqrt(S2) - E, 0.0);
  if (!(p > pmin)) p = pmin + 1e-10 * E;
  int it;
  // (the reciprocals and 1/sqrt by rcp_nr / rsqrt_nr: 1/W = (1 - v^2) W)
  for (it = 1; it <= kC2pMaxIt; ++it) {
    const double iEp = rcp_nr(E + p);
    const double v2 = S2 * iEp * iEp;
    const double W = rsqrt_nr(1. - v2);
    const double iW = (1. - v2) * W;
    const double f = (gam - 1.) * (E - S2 * iEp - D * iW) - p;
    const double df = (gam - 1.) * v2 * (1. - D * W * iEp) - 1.;
    double pn = p - f * rcp_nr(df);
    if (pn <= pmin) pn = 0.5 * (p + pmin);
    const double dp = fabs(pn - p);
    p = pn;
    if (dp <= tol * p) break;
  }
  const double iEp = rcp_nr(E + p);
  const double v2 = S2 * iEp * iEp;
  const double iW = (1. - v2) * rsqrt_nr(1. - v2);
  P[0] = D * iW;
  P[1] = U[1] * iEp;
  P[2] = U[2] * iEp;
  P[3] = U[3] * iEp;
  P[4] = p;
  return it <= kC2pMaxIt;
}

__global__ __launch_bounds__(256) void fv_c2p_kernel(FvC2pArgs a) {
  const long ncell = (long)a.g.nbx * a.g.nbx * a.g.nbx * kFvB3;
  for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < ncell; c += (long)gridDim.x * blockDim.x) {
    const long b = c / kFvB3, q = c % kFvB3;
    const long base = b * 5 * kFvB3 + q;
    double U[5], P[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) U[v] = a.U[base + v * kFvB3];
    if (!sr_c2p(a.g.gam, a.tol, U, a.guess[base + 4 * kFvB3], P)) a.bad[b] = 1;
#pragma unroll
    for (int v = 0; v < 5; ++v) a.P[base + v * kFvB3] = P[v];
  }
}

hipError_t launch_fv_c2p(const FvC2pArgs &a, hipStream_t s) {
  const long ncell = (long)a.g.nbx * a.g.nbx * a.g.nbx * kFvB3;
  long grid = (ncell + 255) / 256;
  if (grid > 1 << 20) grid = 1 << 20;
  hipLaunchKernelGGL(fv_c2p_kernel, dim3((unsigned)grid), dim3(256), 0, s, a);
  return hipGetLastError();
}

__global__ __launch_bounds__(256) void fv_p2c_kernel(FvGrid g, const double *P, double *U) {
  const long ncell = (long)g.nbx * g.nbx * g.nbx * kFvB3;
  for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < ncell; c += (long)gridDim.x * blockDim.x) {
    const long b = c / kFvB3, q = c % kFvB3;
    const long base = b * 5 * kFvB3 + q;
    double Q[5], V[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) Q[v] = P[base + v * kFvB3];
    sr_p2c(g.gam, Q, V);
#pragma unroll
    for (int v = 0; v < 5; ++v) U[base + v * kFvB3] = V[v];
  }
}

hipError_t launch_fv_p2c(const FvGrid &g, const double *P, double *U, hipStream_t s) {
  const long ncell = (long)g.nbx * g.nbx * g.nbx * kFvB3;
  long grid = (ncell + 255) / 256;
  if (grid > 1 << 20) grid = 1 << 20;
  hipLaunchKernelGGL(fv_p2c_kernel, dim3((unsigned)grid), dim3(256), 0, s, g, P, U);
  return hipGetLastError();
}

__global__ __launch_bounds__(256) void fv_layout_kernel(FvGrid g, const double *src, double *dst, int to_blocks) {
  const int N = g.nbx * kFvB;
  const long ncell = (long)N * N * N;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < 5 * ncell;
       idx += (long)gridDim.x * blockDim.x) {
    const int v = (int)(idx / ncell);
    const long c = idx % ncell;
    const int i = (int)(c % N), j = (int)((c / N) % N), k = (int)(c / ((long)N * N));
    const long b = (i / kFvB) + (long)g.nbx * ((j / kFvB) + (long)g.nbx * (k / kFvB));
    const long q = (i % kFvB) + kFvB * ((j % kFvB) + kFvB * (k % kFvB));
    const long bi = b * 5 * kFvB3 + (long)v * kFvB3 + q;
    if (to_blocks) dst[bi] = src[idx];
    else dst[idx] = src[bi];
  }
}

hipError_t launch_fv_layout(const FvGrid &g, const double *src, double *dst, int to_blocks, hipStream_t s) {
  const long n = 5L * g.nbx * g.nbx * g.nbx * kFvB3;
  long grid = (n + 255) / 256;
  if (grid > 1 << 20) grid = 1 << 20;
  hipLaunchKernelGGL(fv_layout_kernel, dim3((unsigned)grid), dim3(256), 0, s, g, src, dst, to_blocks);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// fused RHS + RK stage on 8^3 tiles
// ---------------------------------------------------------------------------

// Cell (cx, cy, cz) of a tile in the accumulator: rows along x, permuted so
// that the lanes of a sweep along x, y or z (8 x 8 of the other two) spread
// over the banks.
__device__ __forceinline__ int acc_cell(int cx, int cy, int cz) {
  return (cx ^ cz) + kFvT * (((cy + cz) & (kFvT - 1)) + kFvT * cz);
}

// One direction d of the tile at block (bx, by, bz), cells t[0..2] on of it:
// lane (ta, tb) walks the tile line along d.  FIRST writes the accumulator
// (twice the flux difference), later directions add to it.  The code is the
// same for the three directions (velocities are held as normal and tangential
// ones), so that it can be unrolled over the line's 9 faces: the windows then
// move through registers without copies.
// STAGED (d = 0): the tile's own cells come from the accumulator, where the
// caller has put them; a lane reads a cell before it writes the difference there.
template <bool FIRST, bool STAGED>
__device__ __forceinline__ void fv_sweep(const FvStageArgs &a, int d, const int (&bl)[3], const int (&t)[3],
                                         double (*acc)[kFvT3]) {
  const int lane = threadIdx.x & 63;
  const int ta = lane % kFvT, tb = lane / kFvT;
  const double gam = a.g.gam, g1 = gam / (gam - 1.);
  const int nbx = a.g.nbx;
  // Along d the tile's 8 cells lie in its own block, and so do the 3 cells
  // beyond one of its ends; the 3 beyond the other end lie in the next block
  // (or the one before).  Cell s of the line: base(s) + off + s * st.
  const int st = d == 0 ? 1 : d == 1 ? kFvB : kFvB * kFvB;
  auto block = [&](int shift) {
    int c[3] = {bl[0], bl[1], bl[2]};
    c[d] += shift;
    c[d] = c[d] < 0 ? nbx - 1 : c[d] >= nbx ? 0 : c[d];
    return a.P + (c[0] + (long)nbx * (c[1] + (long)nbx * c[2])) * (5L * kFvB3);
  };
  const bool upper = t[d] != 0;   // the tile is the upper half of its block along d
  const double *own = block(0);
  const double *lo = upper ? own : block(-1) + kFvB * st;
  const double *hi = upper ? block(1) - kFvB * st : own;
  const int off = (t[0] + (d == 0 ? 0 : ta)) + kFvB * ((t[1] + (d == 1 ? 0 : d == 0 ? ta : tb)) +
                                                        kFvB * (t[2] + (d == 2 ? 0 : tb)));
  // variables held as (rho, v_n, v_t, v_t', p)
  const int d1 = d == 2 ? 0 : d + 1, d2 = d == 0 ? 2 : d - 1;
  const int vi[5] = {0, 1 + d, 1 + d1, 1 + d2, 4};
  // cells f .. f + 5 (counted from 3 before the tile) surround face f
  double u[5][kFvT + 6], h[5][kFvT + 5], c[5][kFvT + 4], E[5][3];
  auto load = [&](int k) {
    const int s = k - 3;
    if (STAGED && s >= 0 && s < kFvT) {
#pragma unroll
      for (int v = 0; v < 5; ++v) u[v][k] = acc[v][acc_cell(s, ta, tb)];
      return;
    }
    const double *p = (s < 0 ? lo : s < kFvT ? own : hi) + s * st;
#pragma unroll
    for (int v = 0; v < 5; ++v) u[v][k] = (p + vi[v] * kFvB3)[off];
  };
#pragma unroll
  for (int k = 0; k < 7; ++k) load(k);
#pragma unroll
  for (int v = 0; v < 5; ++v) {
#pragma unroll
    for (int k = 0; k < 4; ++k) h[v][k] = (u[v][k + 1] - u[v][k]) * (1. / 6.);
#pragma unroll
    for (int k = 0; k < 3; ++k) c[v][k] = weno_curv(h[v][k], h[v][k + 1]);
    weno_products(h[v][0], h[v][1], h[v][2], h[v][3], c[v][0], c[v][1], c[v][2], E[v]);
  }
  double Fprev[5];
#pragma unroll
  for (int f = 0; f <= kFvT; ++f) {   // face between tile cells f-1 and f
    if (f + 7 < kFvT + 6) load(f + 7);
    double PL[5], PR[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      const double *q = h[v] + f;
      PL[v] = weno_left(u[v][f + 2], q[0], q[1], q[2], q[3], E[v]);
      h[v][f + 4] = (u[v][f + 5] - u[v][f + 4]) * (1. / 6.);
      c[v][f + 3] = weno_curv(h[v][f + 3], h[v][f + 4]);
      weno_products(q[1], q[2], q[3], q[4], c[v][f + 1], c[v][f + 2], c[v][f + 3], E[v]);
      PR[v] = weno_right(u[v][f + 3], q[1], q[2], q[3], q[4], E[v]);
    }
    // unphysical face states fall back to the cell's
    double vL = speed2(PL), vR = speed2(PR);
    if (!(PL[0] > 0. && PL[4] > 0. && vL < 1.)) {
#pragma unroll
      for (int v = 0; v < 5; ++v) PL[v] = u[v][f + 2];
      vL = speed2(PL);
    }
    if (!(PR[0] > 0. && PR[4] > 0. && vR < 1.)) {
#pragma unroll
      for (int v = 0; v < 5; ++v) PR[v] = u[v][f + 3];
      vR = speed2(PR);
    }
    double FL[5], FR[5], UL[5], UR[5], F[5];
    const double aL = sr_flux(gam, g1, PL, vL, FL, UL);
    const double aR = sr_flux(gam, g1, PR, vR, FR, UR);
    const double am = fmax(aL, aR);
#pragma unroll
    for (int v = 0; v < 5; ++v) F[v] = fma(-am, UR[v] - UL[v], FL[v] + FR[v]);   // twice the flux
    if (f > 0) {
      const int s = f - 1;
      const int cell = d == 0 ? acc_cell(s, ta, tb) : d == 1 ? acc_cell(ta, s, tb) : acc_cell(ta, tb, s);
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        if (FIRST) acc[vi[v]][cell] = Fprev[v] - F[v];
        else acc[vi[v]][cell] += Fprev[v] - F[v];
      }
    }
#pragma unroll
    for (int v = 0; v < 5; ++v) Fprev[v] = F[v];
  }
}

// W waves per tile: 1, or 3 with one direction each, which finish a tile of a
// small grid in about a third of the time.  The accumulators take 20 KB per
// wave: 8 waves per CU, two per SIMD, which is also what 246 VGPRs allow.
// 256^3 cells take 1.33 ms per stage, primitives included, at 27 TFLOP/s
// (2,150 operations per cell by the counters; 13,140 VALU instructions per
// tile, 85% of them FP64; VALU 60% busy, the rest waits on memory and issue).
// Weights and fluxes as they stood, by cell values with two IEEE square roots
// per state, windows moved by copies and the primitives in a launch of their
// own, took 2.09 ms.
// The line's 9 faces are unrolled: 61 KB of code, of the 64 KB that two CUs
// share.  One copy of the sweep for all directions, a nontemporal epilogue and
// tiles in 2^3-block bricks measured no faster (5.5% slower, and within 0.5%).
template <int W>
__global__ __launch_bounds__(64 * W, 2) void fv_stage_kernel(FvStageArgs a) {
  __shared__ double acc[W][5][kFvT3];
  const int nbx = a.g.nbx;
  const int ntiles = nbx * nbx * nbx * 8;
  int tile = blockIdx.x;
  if (a.xcd_map) {
    const int chunk = (ntiles + 7) >> 3, q = blockIdx.x >> 3;
    tile = q < chunk ? (blockIdx.x & 7) * chunk + q : ntiles;
  }
  if (tile >= ntiles) return;
  const int b = tile >> 3, sub = tile & 7;
  const int bl[3] = {b % nbx, (b / nbx) % nbx, b / (nbx * nbx)};
  const int t[3] = {(sub & 1) * kFvT, ((sub >> 1) & 1) * kFvT, (sub >> 2) * kFvT};
  const int tid = threadIdx.x;
  if (W == 1) {
    // Along x the lanes' lines lie 128 bytes apart, so that each load of the
    // sweep would fetch 64 lines for 8 bytes of each, more than the L1 keeps:
    // the tile's own cells go through LDS, in the accumulator.
    const double *own = a.P + (long)b * 5 * kFvB3 + t[0] + kFvB * (t[1] + kFvB * t[2]);
    const int cx = tid % kFvT, cy = tid / kFvT;
#pragma unroll
    for (int v = 0; v < 5; ++v)
#pragma unroll
      for (int cz = 0; cz < kFvT; ++cz)
        acc[0][v][acc_cell(cx, cy, cz)] = own[v * kFvB3 + cx + kFvB * (cy + kFvB * cz)];
    __syncthreads();
    fv_sweep<true, true>(a, 0, bl, t, acc[0]);
    __syncthreads();
#pragma unroll 1
    for (int d = 1; d < 3; ++d) {
      fv_sweep<false, false>(a, d, bl, t, acc[0]);
      __syncthreads();
    }
  } else {
    const int d = __builtin_amdgcn_readfirstlane(tid >> 6);
    fv_sweep<true, false>(a, d, bl, t, acc[d]);
    __syncthreads();
  }
  // stage combination and the next primitives, the next cell's registers
  // requested while this one's primitives are solved for
  const long g0 = (long)b * 5 * kFvB3 + t[0] + kFvB * (t[1] + kFvB * t[2]);
  auto place = [&](int cell) {
    return g0 + cell % kFvT + kFvB * ((cell / kFvT) % kFvT + kFvB * (cell / (kFvT * kFvT)));
  };
  struct Regs {
    double U[5], w[5], Wa[5], Wb[5], p;
  } in;
  auto request = [&](int cell) {
    const long gi = place(cell);
#pragma unroll
    for (int v = 0; v < 5; ++v) in.U[v] = a.U[gi + v * kFvB3];
    if (a.wmode > 1) {
#pragma unroll
      for (int v = 0; v < 5; ++v) in.w[v] = a.win[gi + v * kFvB3];
    }
    if (a.wmode == 3) {
#pragma unroll
      for (int v = 0; v < 5; ++v) {
        in.Wa[v] = a.Wa[gi + v * kFvB3];
        in.Wb[v] = a.Wb[gi + v * kFvB3];
      }
    }
    if (a.Pout) in.p = a.P[gi + 4 * kFvB3];
  };
  if (a.Wout) request(tid);
#pragma unroll 1
  for (int cell = tid; cell < kFvT3; cell += 64 * W) {
    const int ac = acc_cell(cell % kFvT, (cell / kFvT) % kFvT, cell / (kFvT * kFvT));
    const long gi = place(cell);
    double r[5], out[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      double s = acc[0][v][ac];
      if (W == 3) s = (s + acc[1][v][ac]) + acc[2][v][ac];
      r[v] = 0.5 * s;
    }
    if (a.R) {
#pragma unroll
      for (int v = 0; v < 5; ++v) a.R[gi + v * kFvB3] = r[v];
    }
    if (!a.Wout) continue;
#pragma unroll
    for (int v = 0; v < 5; ++v) {
      const double U = in.U[v];
      if (a.wmode == 1) out[v] = U + a.cW * r[v];
      else if (a.wmode == 2) out[v] = 0.75 * U + 0.25 * (in.w[v] + a.cW * r[v]);
      else if (a.wmode == 3) {
        const double s = (in.Wa[v] - U) + 2. * (in.Wb[v] - U) + (in.w[v] - U);
        out[v] = U + (s * (1. / 3.) + a.cW * r[v]);
      } else out[v] = U + (2. / 3.) * ((in.w[v] - U) + a.cW * r[v]);
    }
    const double p = in.p;
    if (cell + 64 * W < kFvT3) request(cell + 64 * W);
#pragma unroll
    for (int v = 0; v < 5; ++v) a.Wout[gi + v * kFvB3] = out[v];
    if (a.Pout) {
      double P[5];
      if (!sr_c2p(a.g.gam, a.tol, out, p, P)) a.bad[b] = 1;
#pragma unroll
      for (int v = 0; v < 5; ++v) a.Pout[gi + v * kFvB3] = P[v];
    }
  }
}

// ---------------------------------------------------------------------------
// CFL: the largest |lambda+-| over cells and directions (the eigenvalues of
// sr_flux), reduced with lane shuffles, then per workgroup and over the grid
// ---------------------------------------------------------------------------
constexpr int kSpeedThreads = 256;

__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v = fmax(v, __shfl_xor(v, m, 64));
  return v;
}

__device__ __forceinline__ double sr_speed(double gam, double g1, const double P[5], int d) {
  const double rho = P[0], p = P[4];
  const double v2 = P[1] * P[1] + P[2] * P[2] + P[3] * P[3];
  const double ph = p / rho;
  const double h = 1. + g1 * ph;
  const double cs2 = gam * ph / h;
  const double cs = sqrt(cs2);
  const double vd = P[1 + d];
  const double oden = 1. / (1. - v2 * cs2);
  const double root = cs * sqrt((1. - v2) * (1. - v2 * cs2 - vd * vd * (1. - cs2)));
  const double lm = (vd * (1. - cs2) - root) * oden;
  const double lp = (vd * (1. - cs2) + root) * oden;
  return fmax(fabs(lm), fabs(lp));
}

__global__ __launch_bounds__(kSpeedThreads) void fv_speed_kernel(FvGrid g, const double *P, double *part) {
  __shared__ double s_max[kSpeedThreads / 64];
  const long ncell = (long)g.nbx * g.nbx * g.nbx * kFvB3;
  const double gam = g.gam, g1 = gam / (gam - 1.);
  double m = 0.0;
  for (long c = (long)blockIdx.x * kSpeedThreads + threadIdx.x; c < ncell; c += (long)gridDim.x * kSpeedThreads) {
    const long b = c / kFvB3, q = c % kFvB3;
    const double *pc = P + b * 5 * kFvB3 + q;
    const double Pc[5] = {pc[0], pc[kFvB3], pc[2 * kFvB3], pc[3 * kFvB3], pc[4 * kFvB3]};
#pragma unroll
    for (int d = 0; d < 3; ++d) m = fmax(m, sr_speed(gam, g1, Pc, d));
  }
  m = wave_max(m);
  if ((threadIdx.x & 63) == 0) s_max[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double r = s_max[0];
    for (int w = 1; w < kSpeedThreads / 64; ++w) r = fmax(r, s_max[w]);
    part[blockIdx.x] = r;
  }
}

__global__ __launch_bounds__(kSpeedThreads) void fv_speed_max_kernel(const double *part, int n, double *out) {
  __shared__ double s_max[kSpeedThreads / 64];
  double m = 0.0;
  for (int i = threadIdx.x; i < n; i += kSpeedThreads) m = fmax(m, part[i]);
  m = wave_max(m);
  if ((threadIdx.x & 63) == 0) s_max[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double r = s_max[0];
    for (int w = 1; w < kSpeedThreads / 64; ++w) r = fmax(r, s_max[w]);
    out[0] = r;
  }
}

int fv_speed_grid(const FvGrid &g) {
  const long ncell = (long)g.nbx * g.nbx * g.nbx * kFvB3;
  const long gr = (ncell + kSpeedThreads - 1) / kSpeedThreads;
  return gr < 4096 ? (int)gr : 4096;
}

hipError_t launch_fv_max_speed(const FvGrid &g, const double *P, double *part, double *out, hipStream_t s) {
  const int grid = fv_speed_grid(g);
  hipLaunchKernelGGL(fv_speed_kernel, dim3(grid), dim3(kSpeedThreads), 0, s, g, P, part);
  hipLaunchKernelGGL(fv_speed_max_kernel, dim3(1), dim3(kSpeedThreads), 0, s, part, grid, out);
  return hipGetLastError();
}

hipError_t launch_fv_stage(const FvStageArgs &a, hipStream_t s) {
  const int ntiles = a.g.nbx * a.g.nbx * a.g.nbx * 8;
  const int grid = a.xcd_map ? 8 * ((ntiles + 7) / 8) : ntiles;
  if (ntiles <= kFvSplitTiles) hipLaunchKernelGGL(fv_stage_kernel<3>, dim3(grid), dim3(192), 0, s, a);
  else hipLaunchKernelGGL(fv_stage_kernel<1>, dim3(grid), dim3(64), 0, s, a);
  return hipGetLastError();
}

}  // namespace nmx
