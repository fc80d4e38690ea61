// limiter.hpp -- the Barth-Jespersen limiter of a stored state.  The stage
// kernel writes the cell means and node extrema of what it stores
// (StageArgs::mean, StageArgs::ext); the next stage kernel computes the
// factors from them and applies them as it reads (StageArgs::lim_*).  This
// does the same for every other reader of the state.
#pragma once
#include <hip/hip_runtime.h>

namespace mxm {
constexpr int kLimMaxNC = 17;  // the widest state (two-fluid)
// The limited values written in place for slots [e0, e0 + n) of q, whose
// factors are computed from mean [slots][NC] (sum_i w_i q_i), ext
// [slots][NCL][2] (smallest, largest node value of the limited components:
// all NC in 3D, component 0 in 2D) and the neighbours' means through conn
// (the partner slot of each of an element's NF faces); FP64 whatever the
// state precision.  Afterwards nothing is pending on these slots: their
// extrema are NaN, which makes their factor 1, and theta [slots], which a
// stage reads for its q_a, is 1.  The range covers every element of a mesh it
// touches.
template <class R>
hipError_t launch_bj_limit(R *q, double *theta, const double *mean, R *ext, const int *conn, int e0, int n,
                           int NP, int NC, int NF, int dim, double eps, hipStream_t s);
// Extrema that leave nothing pending, as launch_fill's value: a NaN in FP64,
// and two of them in FP32
inline double no_extrema() { return __builtin_bit_cast(double, ~0ull); }
// p[0..n) = v (a kernel, so that it can sit in a captured graph)
hipError_t launch_fill(double *p, long long n, double v, hipStream_t s);
}  // namespace mxm
