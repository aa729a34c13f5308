// Exact (float64) assignment of one row to its nearest centre by a whole wave: what every assignment kernel falls back
// to for the rows that its own evaluation cannot decide.
#pragma once

#include <cfloat>
#include <climits>

#include "common.hpp"

namespace f2cgt {

// Squared L2 or cosine distance of a row and a centre in float64.  kx <= k: how many values the row has; it counts as
// zero in the dimensions after them.  xn: |row|^2 (cosine).
__device__ __forceinline__ double exact_distance(const float* __restrict__ xrow, const float* __restrict__ cr, int k, int kx,
                                                 bool cosine, double xn) {
  if (cosine) {
    double dot = 0.0, cn = 0.0;
    for (int t = 0; t < kx; ++t) {
      dot += (double)xrow[t] * (double)cr[t];
      cn += (double)cr[t] * (double)cr[t];
    }
    for (int t = kx; t < k; ++t) cn += (double)cr[t] * (double)cr[t];
    double den = sqrt(xn) * sqrt(cn);
    den = den > 1e-8 ? den : 1e-8;
    return 1.0 - dot / den;
  }
  double d = 0.0;
  for (int t = 0; t < kx; ++t) {
    const double df = (double)xrow[t] - (double)cr[t];
    d += df * df;
  }
  for (int t = kx; t < k; ++t) d += (double)cr[t] * (double)cr[t];
  return d;
}

// First minimum over the lanes of a wave.  A row without a single comparable distance (NaN or infinite entries) goes to
// centre 0, where the callers' trainer sends it (examples/my_kmeans.py:92-94 turns such distances into 1 before the
// arg-min); the label must be a valid index whatever the data.
__device__ __forceinline__ int first_minimum(double bestv, int besti) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const double ov = __shfl_xor(bestv, off);
    const int oi = __shfl_xor(besti, off);
    if (ov < bestv || (ov == bestv && oi < besti)) { bestv = ov; besti = oi; }
  }
  return besti == INT_MAX ? 0 : besti;
}

__device__ inline int exact_argmin_row(const float* __restrict__ xrow, const float* __restrict__ centers,
                                       int n, int k, int kx, int metric, int lane) {
  const bool cosine = metric == F2CGT_METRIC_COSINE;
  double bestv = DBL_MAX;
  int besti = INT_MAX;
  double xn = 0.0;
  if (cosine)
    for (int t = 0; t < kx; ++t) xn += (double)xrow[t] * (double)xrow[t];
  for (int c = lane; c < n; c += kWave) {
    const double d = exact_distance(xrow, centers + (int64_t)c * k, k, kx, cosine, xn);
    if (d < bestv) { bestv = d; besti = c; }
  }
  return first_minimum(bestv, besti);
}

}  // namespace f2cgt
