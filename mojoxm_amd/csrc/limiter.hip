// limiter.hip -- Barth-Jespersen slope limiter with Venkatakrishnan
// smoothing, split into a per-element theta and an apply that the readers
// of the state perform.
//
//   cell means     sum_i w_i q_i per (element, component), and the
//                  smallest and largest node value per (element,
//                  component), computed by the stage kernel's epilogue
//                  from the values it stores (compute_cell_averages_kernel,
//                  src/solver.mojo:384-407; cell_mean_kernel_2d,
//                  src/local_mesh_2d_gpu.mojo:246-264)
//   theta          one theta per element from the face neighbours' means
//                  (3D: all components, boundary self-neighbour counted,
//                  src/solver.mojo:410-530; 2D: component 0, boundary
//                  faces skipped, src/local_mesh_2d_gpu_limiter.mojo:74-153)
//   apply          q = mean + theta (q - mean) when theta < 1
//
// Both are done by the next stage kernel as it loads the state: each block
// computes theta for its tile and for the elements behind the tile's faces
// (bj.hpp), and applies it to the q_in tile and the partner traces; q_a takes
// the factors that stage 1 stored.  As a launch of its own between two stages
// theta took 3 to 5 us, latency for the most part, against 1 to 5 % more work
// in the stage (us per limited stage, both before -> after: 75^2 P = 2 dam
// break 10.9 -> 7.9, 48^2 Sod FP32 11.6 -> 7.6, 192^2 Sod FP64 33.3 -> 33.1;
// in 3D, where all components are limited, 18^3 P = 3 Euler 66 -> 53, MHD 125
// -> 109, two-fluid 432 -> 320, 28^3 P = 1 Euler 66 -> 58, two-fluid 391 -> 331;
// dg_stage_kernel says how the block shares that work).
// The kernel here limits a stored state in place for its other readers.
//
// The reference takes the minimum of the Venkatakrishnan factor
//   g(x) = (D^2 + 2 D x + eps^2) / (D^2 + 2 x^2 + D x + eps^2)
// over the nodes, x = |q_i - mean|, D the bound on the side of q_i.  For
// x <= D/2, g >= 1 (D x >= 2 x^2), and beyond D/2 g decreases (the
// numerator of g' is D^3 + D eps^2 - 4 D x^2 - 4 D^2 x - 4 eps^2 x, which
// is negative there and falls with x), so the minimum over the nodes with
// q_i above the mean is g at the largest value, and below the mean g at
// the smallest: theta needs only the two extrema, and no pass over the
// state.  g is evaluated on those two nodes' own differences, as the
// per-node loop would.
#include <hip/hip_runtime.h>

#include "bj.hpp"
#include "limiter.hpp"

namespace mxm {
namespace {

// The limited state written in place, then extrema of NaN and theta = 1 (a
// stage takes q_a's theta as it is stored).  A block holds whole elements:
// its threads take one limited component of an element each and form the
// element's factor in LDS (as the stage kernel does), then one node each.
// One launch instead of one for the factors and one for the nodes: a limited
// instance of a batch is read in 4 to 5 us less, of 4^3 cubes in 12 less.
template <class R, int NC, bool ALL>
__global__ __launch_bounds__(256) void bj_limit_kernel(R *__restrict__ q, double *__restrict__ theta,
                                                       const double *__restrict__ mean, R *__restrict__ ext,
                                                       const int *__restrict__ conn, int e0, int n, int NP,
                                                       double eps2) {
  constexpr int NCL = ALL ? NC : 1, NF = ALL ? 4 : 3;
  __shared__ double sTh[256 / 3];  // at least 3 nodes per element
  const int epb = 256 / NP, first = blockIdx.x * epb, elems = min(epb, n - first);
  const int tid = threadIdx.x;
  if (tid < elems) sTh[tid] = 1.0;
  __syncthreads();
  for (int t = tid; t < elems * NCL; t += 256) {
    const int el = t / NCL, e = e0 + first + el;
    int nb[NF];
    bj_neighbours<NF>(e, conn, nb);
    const double th = bj_theta_comp<NC, ALL, NF>(e, t - el * NCL, nb, mean, ext, eps2, 1.0);
    if (th < 1.0)
      atomicMin(reinterpret_cast<unsigned long long *>(&sTh[el]), (unsigned long long)__double_as_longlong(th));
  }
  __syncthreads();
  for (int t = tid; t < elems * NCL * 2; t += 256)
    ext[(size_t)(e0 + first) * NCL * 2 + t] = R(__builtin_nan(""));
  const int el = tid / NP, node = tid - el * NP;
  if (el >= elems) return;
  const size_t e = (size_t)e0 + first + el;
  if (node == 0) theta[e] = 1.0;
  const double th = sTh[el];
  if (!(th < 1.0)) return;
  R *qn = q + (e * NP + node) * NC;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const double bm = mean[e * NC + c];
    qn[c] = R(bm + th * (double(qn[c]) - bm));
  }
}

__global__ void fill_kernel(double *p, long long n, double v) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = v;
}

template <class R, int NC, bool ALL>
void limit_nc(R *q, double *theta, const double *mean, R *ext, const int *conn, int e0, int n, int NP,
              double eps2, hipStream_t s) {
  const int epb = 256 / NP;
  hipLaunchKernelGGL((bj_limit_kernel<R, NC, ALL>), dim3((n + epb - 1) / epb), dim3(256), 0, s, q, theta, mean, ext,
                     conn, e0, n, NP, eps2);
}

}  // namespace

template <class R>
hipError_t launch_bj_limit(R *q, double *theta, const double *mean, R *ext, const int *conn, int e0, int n,
                           int NP, int NC, int NF, int dim, double eps, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  if (NP < 3 || NP > 256 || NF != dim + 1) return hipErrorInvalidValue;
  const double e2 = eps * eps;
#define MXM_LIMIT(N)                                                          \
  case N:                                                                     \
    if (dim == 3)                                                             \
      limit_nc<R, N, true>(q, theta, mean, ext, conn, e0, n, NP, e2, s);      \
    else                                                                      \
      limit_nc<R, N, false>(q, theta, mean, ext, conn, e0, n, NP, e2, s);     \
    break;
  switch (NC) {
    MXM_LIMIT(1) MXM_LIMIT(3) MXM_LIMIT(4) MXM_LIMIT(5) MXM_LIMIT(6) MXM_LIMIT(7) MXM_LIMIT(9) MXM_LIMIT(17)
    default: return hipErrorInvalidValue;
  }
#undef MXM_LIMIT
  return hipGetLastError();
}

hipError_t launch_fill(double *p, long long n, double v, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(fill_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n, v);
  return hipGetLastError();
}

template hipError_t launch_bj_limit<double>(double *, double *, const double *, double *, const int *, int, int, int,
                                            int, int, int, double, hipStream_t);
template hipError_t launch_bj_limit<float>(float *, double *, const double *, float *, const int *, int, int, int,
                                           int, int, int, double, hipStream_t);

}  // namespace mxm
