// amr.h -- launch interface of the batched (order-bucketed) DG stage kernel.
#pragma once
#include <hip/hip_runtime.h>

namespace nmx {

// face interpolation job, kJobInts ints per (face, neighbour):
//   [0] n (my points per direction), [1] m (neighbour's), [2] offset of the
//   job's region in the face buffer ([v][n*n]), [3] 16-bit reciprocals of n*n
//   (low) and n (high), rounded up, [4] base, [5] t1,
//   [6] t2 (neighbour plane node = base + q1*t1 + q2*t2 inside the
//   neighbour), [7] swap, [8..11] a0,a1,b0,b1 covered point ranges, [12]
//   offset of the rows for my a, [13] for my b, in Btab (rows of m doubles),
//   [14..15] the neighbour's first state double (a long)
constexpr int kJobInts = 16;
// LDS of the face interpolation kernel, in doubles: first-pass results
// (4 * covered rows * m) and the rows of each pass (covered rows or columns
// * m); covered rows and columns <= kMaxFaceN.
constexpr int kFaceT1 = 4 * 10 * 10, kFaceR1 = 10 * 10;
constexpr int kMaxFaceN = 10;
// Faces with several neighbours (a coarse face against finer ones): one
// region per neighbour; mdesc[foff] = ns, then per neighbour {region, a0,
// a1, b0, b1}.
constexpr int kMaxFaceNb = 4;

// One element of an order bucket, everything its stage needs besides the
// state: read with wave-uniform loads, so no load of the kernel waits on
// another table lookup first.
struct SlotRec {
  long noff;            // first node of the element (state at 5 * noff)
  double dXbdX[3];      // 2 / box widths
  double bb[6];         // element box in patch coordinates
  double s0, s1;        // CubedShell radii of the patch
  long foff[6];         // kind 1: the neighbour's first state double + base
                        // node; kind 2: the face's values in the face buffer;
                        // kind 3: the face's entry in mdesc
  int fkind[6];         // 0 outer boundary, 1 conforming copy, 2 interpolated
                        // from one neighbour, 3 from several
  int fs1[6], fs2[6];   // kind 1: neighbour node = base + a*fs1 + b*fs2
  int dom;              // CubedShell patch direction and sign
  int n;                // points per direction
  int pad[8];
};
static_assert(sizeof(SlotRec) == 256, "SlotRec is 256 bytes");

constexpr int kBatchMaxN = 10;
// offsets of order n (2 <= n <= 10) in the concatenated D and node tables
__host__ __device__ constexpr int batch_doff(int n) { return (n - 1) * n * (2 * n - 1) / 6 - 1; }
__host__ __device__ constexpr int batch_xoff(int n) { return n * (n - 1) / 2 - 1; }

struct AmrArgs {
  const double *win = nullptr, *U = nullptr, *Wa = nullptr, *Wb = nullptr, *Ain = nullptr;
  double *Aout = nullptr, *Wout = nullptr, *R = nullptr;
  const SlotRec *rec = nullptr;   // this bucket's elements
  int nlist = 0;
  const double *aj = nullptr;     // interpolated face values
  const int *mdesc = nullptr;     // faces with several neighbours
  const double *dXdx = nullptr;   // element blocks of 9*np
  const double *xyz = nullptr;    // element blocks of 3*np
  const double *D = nullptr;      // this bucket's D[i*n + l]
  const double *xb = nullptr;     // this bucket's LGL nodes
  // launches over several orders: D and nodes of order n at batch_doff(n) and
  // batch_xoff(n), 1 / (end weight) at [n]
  const double *Dall = nullptr, *xball = nullptr, *wall = nullptr;
  const double *tdev = nullptr;   // the stage's time is tdev[tidx], t without tdev
  int tidx = 0;
  double t = 0;
  double cA = 0, cW = 0, wend_inv = 0;
  double k[3] = {0, 0, 0};
  double om = 0;
  int wmode = 0, numflux = 0, profile = 0, xcd_map = 0;
  int fv_mid = 0;                 // FV buckets: metric and normal at the midpoints
  // FV buckets: fv_divf_extrap_s1, _s2, _opt (ex_on: s1 > 0 or s2 < DBL_MAX)
  double ex_s1 = 0, ex_s2 = 1.7976931348623157e308;
  int ex_opt = 0, ex_on = 0;
  // fv_rec's end midpoints: recend 0 (_2 modes), 1 (_1), 2 (WENOm3/5/Z with
  // fv_rec_WENOm_s1/_s2/_opt; rec_on: s1 > 0 or s2 < DBL_MAX)
  int recend = 0, rec_opt = 0, rec_on = 0;
  int rec_first = 0;               // fv_rec = 1 (first order)
  double rec_s1 = 0, rec_s2 = 1.7976931348623157e308;
};

struct FaceArgs {
  const double *win = nullptr;
  const int *jobs = nullptr;      // [job][kJobInts]
  int nfaces = 0;                 // jobs
  const double *Btab = nullptr;
  double *aj = nullptr;
};

// The exponential filter, in place, over a list of elements of one order.
struct FilterArgs {
  double *u = nullptr;            // register filtered in place
  const SlotRec *rec = nullptr;
  int nlist = 0;
  const double *F = nullptr;      // F[i*np + l]: the filter along one direction
  const double *xb = nullptr;     // LGL nodes of this order
  const double *dXdx = nullptr;   // element blocks of 9*np (stored geometry)
  int varmask = 0;                // bit v: pi, cx, cy, cz, phi
  int jpow = 0;                   // filter u J^jpow, J = 1/det(dXb/dx)
  int xcd_map = 0;                // as the stages', whose output is in the XCDs' L2s
};

// ---------------------------------------------------------------------------
// Discrete adjoint (adj_stage.h)
// ---------------------------------------------------------------------------

// a transposed plane [4][n*n] that belongs to a face: the value of variable v
// at face point (a, b) is T[off + v n n + a ca + b cb]
struct AdjRead {
  int off, ca, cb;
};

// one (receiving face, neighbour) interpolation job, transposed
struct AdjJob {
  int e, g;             // receiving element (its record in AdjArgs::erec) and face
  int n, m;             // points per direction of the receiver and of the neighbour
  int sw, a0, a1, b0, b1;   // the forward job's axis swap and covered points
  int offA, offB;       // rows for the receiver's a and b points in Btab (m doubles each)
  int md;               // the receiving face's mdesc entry (several neighbours), -1 for one
  int toff;             // this job's transposed plane [4][m*m] in Tbuf
  // neighbour face coordinates (a, b) -> plane indices: q1 = A1 (a - A0) +
  // B1 (b - B0), q2 = A2 (a - A0) + B2 (b - B0)
  int A0, B0, A1, A2, B1, B2;
  int pad;
};
static_assert(sizeof(AdjJob) == 80, "AdjJob is 80 bytes");

// One adjoint stage: y = L^T lam (L the Jacobian of the scalarwave1 DG RHS with
// respect to u), then R = y or Wout as StageArgs' wmodes 1 and 3 to 6 with r = y
// and win = lam.  The RHS is linear and the same at every stage, so the
// transpose of an RK step is that RK step with L^T.  y_phi = 0 and y_pi has +
// lam_phi, which stays what it is through a step: it is read from phi.  Wout
// must not alias lam: neighbours read lam.
struct AdjArgs {
  const double *lam = nullptr, *phi = nullptr;
  const double *U = nullptr, *Wa = nullptr, *Wb = nullptr;
  double *Wout = nullptr, *R = nullptr;
  double cA = 0, cW = 0;
  int wmode = 0;
  int numflux = 0, xcd_map = 0;
  // this launch's elements: fkind 0 outer boundary; 1 copy, the partner as the
  // forward stage gathers it; 2 interpolated: foff the face's first entry in
  // reads, fs1 their number.  fg[6 el + f]: at a copy face the partner's lift
  // scale over this element's
  const SlotRec *rec = nullptr;
  const double *fg = nullptr;
  int nlist = 0;
  const SlotRec *erec = nullptr;  // every element, for the jobs
  const AdjRead *reads = nullptr;
  const double *dXdx = nullptr;   // element blocks of 9*np (stored geometry)
  // the order's D, LGL nodes and 1 / (end weight); for launches over several
  // orders and the jobs those of order n at batch_doff(n), batch_xoff(n) and [n]
  const double *D = nullptr, *xb = nullptr;
  double wend_inv = 0;
  const double *Dall = nullptr, *xball = nullptr, *wall = nullptr;
  const AdjJob *jobs = nullptr;
  int njobs = 0;
  const int *mdesc = nullptr;
  const double *Btab = nullptr;
  double *T = nullptr;
};

// the transposed interpolation jobs into T
hipError_t launch_adj_jobs_box(const AdjArgs &a, hipStream_t s);
hipError_t launch_adj_jobs_stored(const AdjArgs &a, hipStream_t s);
hipError_t launch_adj_jobs_shell(const AdjArgs &a, hipStream_t s);
inline hipError_t launch_adj_jobs(int geom, const AdjArgs &a, hipStream_t s) {
  return geom == 0 ? launch_adj_jobs_box(a, s) : geom == 1 ? launch_adj_jobs_stored(a, s) : launch_adj_jobs_shell(a, s);
}
// the stage over a.nlist elements of order np, or of any order up to nmax (np = 0)
hipError_t launch_adj_box(int np, int nmax, const AdjArgs &a, hipStream_t s);
hipError_t launch_adj_stored(int np, int nmax, const AdjArgs &a, hipStream_t s);
hipError_t launch_adj_shell(int np, int nmax, const AdjArgs &a, hipStream_t s);
inline hipError_t launch_adj(int np, int nmax, int geom, const AdjArgs &a, hipStream_t s) {
  return geom == 0   ? launch_adj_box(np, nmax, a, s)
         : geom == 1 ? launch_adj_stored(np, nmax, a, s)
                     : launch_adj_shell(np, nmax, a, s);
}

// the DG stage kernels (dg_stage.h) over a.nlist elements of order np, or of
// any order up to nmax (np = 0); geom 0 Cartesian, 1 stored dX/dx, 2
// CubedShell recomputed
hipError_t launch_dg_box(int np, int nmax, const AmrArgs &a, hipStream_t s);
hipError_t launch_dg_stored(int np, int nmax, const AmrArgs &a, hipStream_t s);
hipError_t launch_dg_shell(int np, int nmax, const AmrArgs &a, hipStream_t s);
inline hipError_t launch_dg(int np, int nmax, int geom, const AmrArgs &a, hipStream_t s) {
  return geom == 0   ? launch_dg_box(np, nmax, a, s)
         : geom == 1 ? launch_dg_stored(np, nmax, a, s)
                     : launch_dg_shell(np, nmax, a, s);
}
hipError_t launch_face_interp(const FaceArgs &a, hipStream_t s);
hipError_t launch_filter(int np, int geom, const FilterArgs &a, hipStream_t s);
// the FV element kernel (fv_divf on uniform points, fvelm_stage.h) over
// a.nlist elements of np points; rec: the interior scheme, 5 WENO5, 7 WENO-Z,
// 9 WENOT, 3 WENOm3 (the end midpoints by AmrArgs::recend); geom 0 Cartesian,
// 2 CubedShell; wc[np]: distances between the midpoints around each uniform
// point; a.xb the uniform points
hipError_t launch_fvelm(int np, int rec, int geom, const AmrArgs &a, const double *wc, hipStream_t s);

}  // namespace nmx
