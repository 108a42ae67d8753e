// fv.h -- launch interface of the FV WENO5 + LLF kernels (special-relativistic
// Euler, ideal gas) on a periodic grid of cubic cell blocks.
#pragma once
#include <hip/hip_runtime.h>

namespace nmx {

// Grid: nbx^3 blocks of B^3 cells (cell size 1, periodic).  A state register
// holds [block][var][B^3] doubles, block b = bx + nbx (by + nbx bz), cell
// i + B (j + B k) inside; conserved vars (D, Sx, Sy, Sz, tau), primitive vars
// (rho, vx, vy, vz, p).
struct FvGrid {
  int B = 16;        // cells per block edge
  int nbx = 16;      // blocks per grid edge
  double gam = 2.0;  // ideal-gas Gamma
};

// c2p of every cell: P = primitives of U, guess's pressure as the Newton guess
// (guess may be P); blocks whose solve fails get bad[b] = 1 (never cleared here)
struct FvC2pArgs {
  FvGrid g;
  const double *U = nullptr, *guess = nullptr;
  double *P = nullptr;
  int *bad = nullptr;
  double tol = 1e-12;
};

// fused RHS + RK stage on 8^3-cell tiles:
//   r = -sum_d (F_{i+1/2} - F_{i-1/2}) from the primitives P (WENO5 + LLF)
//   R = r and, by wmode,
//   1: Wout = U + cW r
//   2: Wout = 0.75 U + 0.25 (win + cW r)
//   3: Wout = U + ((Wa - U) + 2 (Wb - U) + (win - U))/3 + cW r, the end of an
//      RK4 step with the stage inputs Wa, Wb, win
//   4: Wout = U + 2/3 ((win - U) + cW r), the end of an sspRK3 step
// (the sum of the earlier stages' r recovered from their inputs; Wout may be
// U), then Pout = the primitives of Wout, solved as c2p does from P's pressure
struct FvStageArgs {
  FvGrid g;
  const double *P = nullptr;
  const double *win = nullptr, *U = nullptr, *Wa = nullptr, *Wb = nullptr;
  double *Wout = nullptr, *R = nullptr, *Pout = nullptr;
  int *bad = nullptr;
  double cW = 0, tol = 1e-12;
  int wmode = 0;
  int xcd_map = 1;
};

hipError_t launch_fv_c2p(const FvC2pArgs &a, hipStream_t s);
// the largest characteristic speed |lambda+-| over all cells and directions
// of primitives P: per-workgroup maxima in part[grid], the grid's in out[0]
int fv_speed_grid(const FvGrid &g);
hipError_t launch_fv_max_speed(const FvGrid &g, const double *P, double *part, double *out, hipStream_t s);
hipError_t launch_fv_p2c(const FvGrid &g, const double *P, double *U, hipStream_t s);
hipError_t launch_fv_stage(const FvStageArgs &a, hipStream_t s);
// flat [v][cell] (cell = i + N (j + N k), N = B nbx) <-> block layout
hipError_t launch_fv_layout(const FvGrid &g, const double *src, double *dst, int to_blocks, hipStream_t s);

}  // namespace nmx
