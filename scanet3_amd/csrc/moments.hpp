// Mean and squared deviations of values that come in parts, for the statistics of a batch normalisation.
#pragma once
#include <hip/hip_runtime.h>

namespace sn {

// n values of mean `mean` and squared deviations `m2` joined with k values of mean `m` and squared deviations `q`, for N channels, by the
// pairwise update of Chan, Golub and LeVeque (1983):
//   mean += d w, m2 += q + d^2 n w   with d = m - mean, w = k / (n + k)
// Where d leaves float32's range or an infinity is among the values, the mean is the weighted one, which is what their sum
// over their number would be: a channel that holds an infinity has it for its mean, one that holds both has none (NaN).
// (The weighted form rounds twice as often; d is looked at by one multiply-add a channel.)  CHECK = false: the caller looks at the mean
// when it has joined everything, and finds it not finite in these cases.
template <int N, bool CHECK = true, class V, class W>
__device__ __forceinline__ void join_moments(float n, V& mean, V& m2, float k, const W& m, const W& q) {
  if (k == 0.f) return;
  if (n == 0.f) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      mean[i] = m[i];
      m2[i] = q[i];
    }
    return;
  }
  const float w = k / (n + k), nw = n * w;
  float d[N], finite = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    d[i] = m[i] - mean[i];
    if (CHECK) finite = __builtin_fmaf(d[i], 0.f, finite);  // NaN once a d is not finite
    m2[i] = m2[i] + (q[i] + d[i] * nw * d[i]);
  }
  if (finite == 0.f) {
#pragma unroll
    for (int i = 0; i < N; ++i) mean[i] = mean[i] + d[i] * w;
  } else {
    const float wn = n / (n + k);
#pragma unroll
    for (int i = 0; i < N; ++i) mean[i] = __builtin_isfinite(d[i]) ? mean[i] + d[i] * w : mean[i] * wn + m[i] * w;
  }
}

}  // namespace sn
