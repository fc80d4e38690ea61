// bj.hpp -- the Barth-Jespersen factor of one element with Venkatakrishnan
// smoothing, from the cell means of the element and its face neighbours and
// the element's smallest and largest node value (limiter.hip says why those
// suffice).  The stage kernels compute it for the elements they read; the
// limiter's own kernel computes the same bits for readers of a stored state.
#pragma once

#include <hip/hip_runtime.h>

namespace mxm {

// n / d correctly rounded, as the division sequence of the ISA's own
// instructions: the stage kernels are compiled to refine reciprocals for
// their divisions, and theta must not depend on where it is computed.
__device__ __forceinline__ double div_rounded(double n, double d) {
  bool scaled, unused;
  const double ds = __builtin_amdgcn_div_scale(n, d, false, &unused);
  const double ns = __builtin_amdgcn_div_scale(n, d, true, &scaled);
  double r = __builtin_amdgcn_rcp(ds);
  r = fma(r, fma(-ds, r, 1.0), r);
  r = fma(r, fma(-ds, r, 1.0), r);
  const double q = ns * r;
  return __builtin_amdgcn_div_fixup(__builtin_amdgcn_div_fmas(fma(-ds, q, ns), r, q, scaled), d, n);
}

// mean [slots][NC], ext [slots][NCL][2] (NCL = NC with ALL, else component 0
// only) in the state's precision, whose values they are (NaN: nothing pending,
// no factor below 1), nb = conn[e] of conn [slots][NF], the partner slot of each face (the
// element's own on a boundary, which constrains only with ALL)
template <int NF>
__device__ __forceinline__ void bj_neighbours(int e, const int *conn, int (&nb)[NF]) {
#pragma unroll
  for (int f = 0; f < NF; ++f) nb[f] = conn[(size_t)e * NF + f];
}
// the smaller of th and the factor that component c asks for
template <int NC, bool ALL, int NF, class R>
__device__ __forceinline__ double bj_theta_comp(int e, int c, const int (&nb)[NF], const double *mean,
                                                const R *ext, double eps2, double th) {
  constexpr int NCL = ALL ? NC : 1;
  const double bm = mean[(size_t)e * NC + c];
  double mn = bm, mx = bm;
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const double v = mean[(size_t)nb[f] * NC + c];
    if (ALL || nb[f] != e) {  // (its own mean constrains nothing)
      mn = v < mn ? v : mn;
      mx = v > mx ? v : mx;
    }
  }
  const double pD = mx - bm < 0.0 ? 0.0 : mx - bm;
  const double nD = bm - mn < 0.0 ? 0.0 : bm - mn;
#pragma unroll
  for (int s = 0; s < 2; ++s) {  // the smallest and the largest node value
    const double d = double(ext[((size_t)e * NCL + c) * 2 + s]) - bm;
    const double da = d >= 0.0 ? d : -d;
    if (da <= 1.0e-30) continue;
    const double D = d > 0.0 ? pD : nD;
    const double D2 = D * D, d2 = da * da, Dd = D * da;
    const double al = div_rounded(D2 + 2.0 * Dd + eps2, D2 + 2.0 * d2 + Dd + eps2);
    th = al < th ? al : th;
  }
  return th;
}
template <int NC, bool ALL, int NF, class R>
__device__ __forceinline__ double bj_theta(int e, const int (&nb)[NF], const double *mean, const R *ext,
                                           double eps2) {
  double th = 1.0;
#pragma unroll
  for (int c = 0; c < (ALL ? NC : 1); ++c) th = bj_theta_comp<NC, ALL, NF>(e, c, nb, mean, ext, eps2, th);
  return th;
}

}  // namespace mxm
