// amr_kernels.hip -- the face values of meshes with mixed refinement levels
// and mixed element orders: face_interp_kernel, once per RK stage before the
// stage kernels (dg_stage.h), computes ajsurf (the neighbour's values at a
// face's points) of every interpolated face by 2D tensor Lagrange
// interpolation of the neighbour's face plane (surface.c:1081-1337,
// interpolate.c:296-363) into a compact face buffer.
#include <hip/hip_runtime.h>

#include "amr.h"
#include "dg_common.h"

namespace nmx {

// ---------------------------------------------------------------------------
// face interpolation, one wave per (face, neighbour) job:
//   pass 1: T[v][x1][q2] = sum_q1 P[v](q1, q2) R1[x1][q1]; a lane owns one
//           (v, q2) line of the neighbour plane and keeps the x1 sums in
//           registers;
//   pass 2: V[v][a][b] = sum_q2 T[v][x1][q2] R2[x2][q2], (x1, x2) = (a, b),
//           or (b, a) when the neighbour's first in-plane axis runs along my
//           b, for the points this neighbour covers (0 elsewhere).
// The plane lines and both passes' rows are requested together, so a job
// waits on one round trip to memory.  A face with several neighbours has
// one region per neighbour, averaged by the stage kernel.
// The jobs are in the order of the elements whose planes they read, so the
// lines of a plane normal to x (every line of the element's block) come from
// HBM once, and four jobs, of which a CU mostly finds the plane in its L1, make
// a workgroup (one wave per workgroup: the 100,318 jobs of 19,200 elements of 4
// to 10 points take 118 us instead of 106, 282 MB fetched and 171 written).
// ---------------------------------------------------------------------------
constexpr int kFaceWaves = 4;   // jobs per workgroup

struct JobView {
  int n, m, ajoff, inn, in, base, t1, t2, sw, a0, a1, b0, b1, offA, offB;
  long soff;
  __device__ JobView(const NMX_CONST int *j) {
    n = j[0]; m = j[1]; ajoff = j[2]; inn = (unsigned)j[3] & 0xffff; in = (unsigned)j[3] >> 16; base = j[4]; t1 = j[5]; t2 = j[6];
    sw = j[7]; a0 = j[8]; a1 = j[9]; b0 = j[10]; b1 = j[11]; offA = j[12]; offB = j[13];
    soff = (long)(unsigned)j[14] | ((long)j[15] << 32);
  }
  __device__ int x1lo() const { return sw ? b0 : a0; }
  __device__ int nx1() const { return (sw ? b1 - b0 : a1 - a0) + 1; }
  __device__ int x2lo() const { return sw ? a0 : b0; }
  __device__ int nx2() const { return (sw ? a1 - a0 : b1 - b0) + 1; }
};

// One job with the neighbour's order M known at compile time: the loops
// over its points are unrolled without branches, so the LDS reads of a row
// are issued together instead of one round trip per term.  The lanes of pass 2
// take the face's points in order, whole lines of the face buffer at a time,
// with their places from multiplications (divisions by n took a third of the
// kernel's instructions; a lane per line of points instead of per point has
// none, but writes every line in pieces: 138 us for the faces of 19,200
// elements).
template <int M>
__device__ __forceinline__ void face_job(const FaceArgs &a, const JobView &J, int tid, double *s_T, double *s_R1,
                                         double *s_R2) {
  const int n = J.n, nx1 = J.nx1(), nx2 = J.nx2();
  const int n1 = nx1 * M, n2 = nx2 * M;
  // every load of this face: rows (at most 100 doubles each, two per lane)
  // and my (v, q2) line of the plane
  const double *R1 = a.Btab + (J.sw ? J.offB : J.offA) + J.x1lo() * M;
  const double *R2 = a.Btab + (J.sw ? J.offA : J.offB) + J.x2lo() * M;
  const double r1a = tid < n1 ? R1[tid] : 0.0, r1b = tid + 64 < n1 ? R1[tid + 64] : 0.0;
  const double r2a = tid < n2 ? R2[tid] : 0.0, r2b = tid + 64 < n2 ? R2[tid + 64] : 0.0;
  const bool act = tid < 4 * M;
  const int v = act ? tid / M : 0, q2 = act ? tid % M : 0;
  const double *P = a.win + J.soff + J.base + (long)v * M * M * M + q2 * J.t2;
  double p[M];
#pragma unroll
  for (int q1 = 0; q1 < M; ++q1) p[q1] = act ? P[q1 * J.t1] : 0.0;
  if (tid < n1) s_R1[tid] = r1a;
  if (tid + 64 < n1) s_R1[tid + 64] = r1b;
  if (tid < n2) s_R2[tid] = r2a;
  if (tid + 64 < n2) s_R2[tid + 64] = r2b;
  wave_lds_fence();
  if (act) {
    double *T = s_T + v * nx1 * M + q2;
    for (int x = 0; x < nx1; ++x) {
      const double *row = s_R1 + x * M;
      double t = 0.0;
#pragma unroll
      for (int q1 = 0; q1 < M; ++q1) t += p[q1] * row[q1];
      T[x * M] = t;
    }
  }
  wave_lds_fence();
  const int nn = n * n;
  double *out = a.aj + J.ajoff;
  for (int idx = tid; idx < 4 * nn; idx += 64) {
    // idx < 400 and n <= 10: exact quotients from 16-bit reciprocals
    const int vv = (idx * J.inn) >> 16, q = idx - vv * nn;
    const int fb = (q * J.in) >> 16, fa = q - fb * n;
    double t = 0.0;
    if (fa >= J.a0 && fa <= J.a1 && fb >= J.b0 && fb <= J.b1) {
      const int x1 = (J.sw ? fb : fa) - J.x1lo(), x2 = (J.sw ? fa : fb) - J.x2lo();
      const double *T = s_T + (vv * nx1 + x1) * M;
      const double *row = s_R2 + x2 * M;
#pragma unroll
      for (int k = 0; k < M; ++k) t += T[k] * row[k];
    }
    out[idx] = t;
  }
}

__global__ __launch_bounds__(64 * kFaceWaves) void face_interp_kernel(FaceArgs a) {
  __shared__ double s_T[kFaceWaves][kFaceT1];    // [v][x1][m]
  __shared__ double s_R1[kFaceWaves][kFaceR1];   // [x1][m]
  __shared__ double s_R2[kFaceWaves][kFaceR1];   // [x2][m]
  const int tid = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // contiguous ranges of jobs per XCD, kFaceWaves of them per workgroup
  const int chunk = (a.nfaces + 7) >> 3, q = kFaceWaves * (blockIdx.x >> 3) + wv;
  const int fi = (blockIdx.x & 7) * chunk + q;
  if (q >= chunk || fi >= a.nfaces) return;   // waves do not wait for one another
  const JobView J(as_const(a.jobs) + kJobInts * fi);
  switch (J.m) {
#define NMX_CASE(M_)                                       \
  case M_:                                                 \
    face_job<M_>(a, J, tid, s_T[wv], s_R1[wv], s_R2[wv]);  \
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

hipError_t launch_face_interp(const FaceArgs &a, hipStream_t s) {
  if (a.nfaces == 0) return hipSuccess;
  const int chunk = (a.nfaces + 7) / 8;
  const int grid = 8 * ((chunk + kFaceWaves - 1) / kFaceWaves);
  hipLaunchKernelGGL(face_interp_kernel, dim3(grid), dim3(64 * kFaceWaves), 0, s, a);
  return hipGetLastError();
}

}  // namespace nmx
