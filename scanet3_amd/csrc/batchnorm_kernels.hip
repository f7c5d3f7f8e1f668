// Batch normalisation over the last axis of a channels-last tensor viewed as [rows, C]
// (generic `batchNorm`, math/nn/AllKernels.scala:663-684, as the BatchNorm layer calls it for
// `axes = Seq(-1)`, models/layer/BatchNorm.scala:123-143).
//
//   training:  mean = sum(x)/rows, var = sum((x-mean)^2)/rows   (alg/AllKernels.scala:505-513)
//   frozen:    mean, var = the moving statistics
//   inv = rsqrt(var + eps) * gamma;  y = (x*inv - mean*inv) + beta
//
// All of it is memory bound: every pass reads the activation once with 8 row-loads in flight per
// lane; the per-channel reductions are cut into row slices so the grid covers the chip, and the
// slices are added by 64 threads a channel whose sums meet in a fixed tree (deterministic, no atomics).  So what a pass
// can be spared is what counts: mean and variance come out of one read, and where a 2 x 2 max pooling
// follows, the normalised tensor and its gradient are never in memory (the pooling's windows are normalised as
// they are compared, and their gradients are looked up where they are needed).
#include "batchnorm_rules.hpp"
#include "common.hpp"
#include "moments.hpp"

namespace sn {
namespace {

typedef float bn_f4 __attribute__((ext_vector_type(4)));

enum { BN_SUM = 0, BN_SQDIFF = 1, BN_GRAD = 2 };

// Block = 64 columns x 4 waves; wave w takes rows r0+w, r0+w+4, ... of its slice.
// BN_SUM:    part0 = sum x
// BN_SQDIFF: part0 = sum (x - mean)^2
// BN_GRAD:   part0 = sum dy, part1 = sum dy * (x - mean)
template <int MODE>
__global__ __launch_bounds__(256) void bn_reduce_kernel(const float* __restrict__ x, const float* __restrict__ dy,
                                                         const float* __restrict__ mean, float* __restrict__ part0,
                                                         float* __restrict__ part1, int64_t rows, int cols, int64_t rows_per_slice) {
  __shared__ float smem[2][4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = blockIdx.x * 64 + lane;
  const int64_t r0 = (int64_t)blockIdx.y * rows_per_slice;
  const int64_t r1 = r0 + rows_per_slice < rows ? r0 + rows_per_slice : rows;
  float s0 = 0.f, s1 = 0.f;
  if (c < cols) {
    const float m = MODE == BN_SUM ? 0.f : mean[c];
    int64_t r = r0 + wave;
    for (; r + 28 < r1; r += 32) {
      float a[8], b[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) a[u] = x[(r + 4 * u) * cols + c];
      if (MODE == BN_GRAD) {
#pragma unroll
        for (int u = 0; u < 8; ++u) b[u] = dy[(r + 4 * u) * cols + c];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        if (MODE == BN_SUM) s0 += a[u];
        if (MODE == BN_SQDIFF) { const float d = a[u] - m; s0 += d * d; }
        if (MODE == BN_GRAD) { s0 += b[u]; s1 += b[u] * (a[u] - m); }
      }
    }
    for (; r < r1; r += 4) {
      const float a = x[r * cols + c];
      if (MODE == BN_SUM) s0 += a;
      if (MODE == BN_SQDIFF) { const float d = a - m; s0 += d * d; }
      if (MODE == BN_GRAD) { const float b = dy[r * cols + c]; s0 += b; s1 += b * (a - m); }
    }
  }
  smem[0][wave][lane] = s0;
  if (MODE == BN_GRAD) smem[1][wave][lane] = s1;
  __syncthreads();
  if (wave == 0 && c < cols) {
    part0[(int64_t)blockIdx.y * cols + c] = ((smem[0][0][lane] + smem[0][1][lane]) + smem[0][2][lane]) + smem[0][3][lane];
    if (MODE == BN_GRAD)
      part1[(int64_t)blockIdx.y * cols + c] = ((smem[1][0][lane] + smem[1][1][lane]) + smem[1][2][lane]) + smem[1][3][lane];
  }
}

// Whole vectors of channels (C % 4 == 0, C <= 1024): the tensor is read as one stream of float4.  The `active` threads of a block
// are the largest multiple of C/4 up to 256 and a thread's float4 index moves in steps of them, so it stays on the same four
// channels and a wavefront's load covers 1 KiB of consecutive memory.  A block owns `per4` consecutive float4 (a multiple of
// `active`); threads with equal t % (C/4) meet in LDS.

// Joins the values in LDS of the threads t, t + cg, t + 2 cg, ... of a block pairwise: f(to, from) folds one into the other, thread
// t < cg ends with the whole.  (One thread adding 32 in a row waits for LDS 32 times: 2 us of such a launch.)
template <class F>
__device__ __forceinline__ void over_channel_peers(int t, int cg, int active, F f) {
  const int peers = active / cg, j = t / cg;
  int half = 1;
  while (2 * half < peers) half *= 2;
  for (; half > 0; half >>= 1) {
    __syncthreads();
    if (t < active && j < half && j + half < peers) f(t, t + half * cg);
  }
  __syncthreads();
}

// part0 = sum dy, part1 = sum dy * (x - mean)
__global__ __launch_bounds__(256) void bn_grad_sums_v4_kernel(const bn_f4* __restrict__ x, const bn_f4* __restrict__ dy,
                                                               const float* __restrict__ mean, float* __restrict__ part0,
                                                               float* __restrict__ part1, int64_t n4, int cols, int active, int64_t per4) {
  __shared__ bn_f4 smem[2][256];
  const int t = threadIdx.x, cg = cols / 4, g = t % cg;
  const int64_t begin = (int64_t)blockIdx.x * per4;
  const int64_t end = begin + per4 < n4 ? begin + per4 : n4;
  const bn_f4 m = *(const bn_f4*)(mean + 4 * g);
  bn_f4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
  int64_t i = t < active ? begin + t : end;
  for (; i + 7 * active < end; i += 8 * active) {
    bn_f4 a[8], b[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) a[u] = __builtin_nontemporal_load(x + i + u * active);
#pragma unroll
    for (int u = 0; u < 8; ++u) b[u] = __builtin_nontemporal_load(dy + i + u * active);
#pragma unroll
    for (int u = 0; u < 8; ++u) { s0 = s0 + b[u]; s1 = s1 + b[u] * (a[u] - m); }
  }
  for (; i < end; i += active) {
    const bn_f4 a = x[i], b = dy[i];
    s0 = s0 + b;
    s1 = s1 + b * (a - m);
  }
  smem[0][t] = s0;
  smem[1][t] = s1;
  over_channel_peers(t, cg, active, [&](int to, int from) {
    smem[0][to] = smem[0][to] + smem[0][from];
    smem[1][to] = smem[1][to] + smem[1][from];
  });
  if (t < cg) {
    *(bn_f4*)(part0 + (int64_t)blockIdx.x * cols + 4 * t) = smem[0][t];
    *(bn_f4*)(part1 + (int64_t)blockIdx.x * cols + 4 * t) = smem[1][t];
  }
}

// The same sums where dy is the gradient of a 2 x 2 max pooling right above: it is zero but at the windows' recorded first
// maxima, so the sums run over the pooling's output (n4 = its float4).  A window whose recorded place lies in the padding
// (nothing inside it was above -inf) has no element to hand its gradient to.
// [1000 x 26 x 26 x 32] with stride 2: 19 us for 113 MB; the pooling's backward pass and the sums over its 86 MB result took 29 + 29.
struct PoolWindows {
  int h, w, ho, wo, sh, sw, pt, pl;
  FastDiv by_cg, by_wo, by_ho;
};
__global__ __launch_bounds__(256) void bn_pool_grad_sums_kernel(const float* __restrict__ x, const bn_f4* __restrict__ dy,
                                                                 const uint32_t* __restrict__ arg, const float* __restrict__ mean,
                                                                 float* __restrict__ part0, float* __restrict__ part1, uint32_t n4, int cols,
                                                                 int active, uint32_t per4, PoolWindows p) {
  __shared__ bn_f4 smem[2][256];
  const int t = threadIdx.x, cg = cols / 4, g = t % cg;
  const uint32_t begin = blockIdx.x * per4, end = begin + per4 < n4 ? begin + per4 : n4;
  const bn_f4 m = *(const bn_f4*)(mean + 4 * g);
  bn_f4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
  constexpr int U = 2;  // windows in flight
  for (uint32_t i0 = t < active ? begin + t : end; i0 < end; i0 += U * active) {
    bn_f4 gv[U], xv[U][4];
    uint32_t av[U];
    bool in[U][4];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool on = i0 + u * active < end;
      const uint32_t i = on ? i0 + u * active : i0;
      const uint32_t win = div_by(i, p.by_cg), row = div_by(win, p.by_wo), b = div_by(row, p.by_ho);
      const int ix0 = (int)(win - row * (uint32_t)p.wo) * p.sw - p.pl, iy0 = (int)(row - b * (uint32_t)p.ho) * p.sh - p.pt;
      gv[u] = dy[i];
      av[u] = arg[i];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int iy = iy0 + (k >> 1), ix = ix0 + (k & 1);
        in[u][k] = on && (unsigned)iy < (unsigned)p.h && (unsigned)ix < (unsigned)p.w;
        xv[u][k] = *(const bn_f4*)(x + (in[u][k] ? ((b * p.h + iy) * p.w + ix) * cols + 4 * g : 0u));
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t at = (av[u] >> (8 * e)) & 255u;
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (in[u][k] && at == (uint32_t)k) { s0[e] += gv[u][e]; s1[e] += gv[u][e] * (xv[u][k][e] - m[e]); }
      }
  }
  smem[0][t] = s0;
  smem[1][t] = s1;
  over_channel_peers(t, cg, active, [&](int to, int from) {
    smem[0][to] = smem[0][to] + smem[0][from];
    smem[1][to] = smem[1][to] + smem[1][from];
  });
  if (t < cg) {
    *(bn_f4*)(part0 + (int64_t)blockIdx.x * cols + 4 * t) = smem[0][t];
    *(bn_f4*)(part1 + (int64_t)blockIdx.x * cols + 4 * t) = smem[1][t];
  }
}

// Mean and sum of squared deviations of a block's rows in one read: a thread takes eight values of a channel at a time, forms their own
// mean and deviations in registers and joins them to what it has (join_moments): no large squares are subtracted anywhere, so the
// variance is as good as the two-read form's.
// [676000 x 32]: 17 us, where a read for the mean, its finishing launch and a read for the variance took 15 + 5 + 15.
__global__ __launch_bounds__(256) void bn_stats_v4_kernel(const bn_f4* __restrict__ x, float* __restrict__ part_mean, float* __restrict__ part_m2,
                                                           int64_t n4, int cols, int active, int64_t per4) {
  __shared__ bn_f4 smem[2][256];
  __shared__ float count[256];
  const int t = threadIdx.x, cg = cols / 4;
  const int64_t begin = (int64_t)blockIdx.x * per4;
  const int64_t end = begin + per4 < n4 ? begin + per4 : n4;
  const bn_f4 zero = {0.f, 0.f, 0.f, 0.f};
  bn_f4 mean = zero, m2 = zero;
  float n = 0.f;
  auto join = [&](const bn_f4& m, const bn_f4& q, float k) {  // k values of mean m and squared deviations q
    join_moments<4, false>(n, mean, m2, k, m, q);
    n += k;
  };
  int64_t i = t < active ? begin + t : end;
  for (; i + 7 * active < end; i += 8 * active) {
    bn_f4 a[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) a[u] = __builtin_nontemporal_load(x + i + u * active);
    const bn_f4 m = (((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]))) * 0.125f;
    bn_f4 q = zero;
#pragma unroll
    for (int u = 0; u < 8; ++u) { const bn_f4 d = a[u] - m; q = q + d * d; }
    join(m, q, 8.0f);
  }
  if (i < end) {  // what is left of the block, one to seven values, requested together as well
    const int left = (int)((end - i + active - 1) / active);
    bn_f4 a[7];
#pragma unroll
    for (int u = 0; u < 7; ++u) a[u] = __builtin_nontemporal_load(x + i + (u < left ? u * active : 0));
    bn_f4 m = zero, q = zero;
#pragma unroll
    for (int u = 0; u < 7; ++u) m = u < left ? m + a[u] : m;
    m = m / (float)left;
#pragma unroll
    for (int u = 0; u < 7; ++u) { const bn_f4 d = a[u] - m; q = u < left ? q + d * d : q; }
    join(m, q, (float)left);
  }
  if (n > 0.f && !(__builtin_isfinite(mean[0]) && __builtin_isfinite(mean[1]) && __builtin_isfinite(mean[2]) && __builtin_isfinite(mean[3]))) {
    // an infinity, or values too far apart for their difference: the sum over the number (0.5 us less than looking at every join)
    bn_f4 s = zero;
    for (i = begin + t; i < end; i += active) s = s + x[i];
    mean = s / n;
  }
  smem[0][t] = mean;
  smem[1][t] = m2;
  count[t] = n;
  over_channel_peers(t, cg, active, [&](int to, int from) {
    const float na = count[to], nb = count[from];
    const bn_f4 mb = smem[0][from], qb = smem[1][from];
    bn_f4 ma = smem[0][to], qa = smem[1][to];
    join_moments<4>(na, ma, qa, nb, mb, qb);
    smem[0][to] = ma;
    smem[1][to] = qa;
    count[to] = na + nb;
  });
  if (t < cg) {
    *(bn_f4*)(part_mean + (int64_t)blockIdx.x * cols + 4 * t) = smem[0][t];
    *(bn_f4*)(part_m2 + (int64_t)blockIdx.x * cols + 4 * t) = smem[1][t];
  }
}

// Sums over one channel's slices by 64 threads: a block is 4 channels x 64 slice lanes; lane j takes slices j, j+64, ..., 16 of them
// requested together (nearly always all there are), the lanes' sums meet in a fixed tree.  Every thread of the block must
// call these.  (One thread per channel would walk up to 1024 slices one memory latency after another; 16 threads a channel
// took 8.1 us for 1024 slices of two sums, 64 with all their loads at once take 4.7.)
// Up to 256 slices a lane's share is four, and no more are asked for (200 channels, 4096 rows: all of the layer's launches 35.4 -> 33.6).
constexpr int FINISH_CHANNELS = 4, FINISH_LOADS = 16, FINISH_FEW = 4;
// f(slice, place in the slices' arrays, whether there is such a slice): places that do not exist repeat the last slice
template <int LOADS, class F>
__device__ __forceinline__ void for_slices(int first, int slices, int cols, int c, F f) {
#pragma unroll
  for (int u = 0; u < LOADS; ++u) {
    const int i = first + 64 * u, at = min(i, slices - 1);
    f(u, (int64_t)at * cols + min(c, cols - 1), i < slices);
  }
}
__device__ __forceinline__ float over_slice_lanes(float s, float (*smem)[FINISH_CHANNELS]) {
#pragma unroll
  for (int d = 4; d < 64; d <<= 1) s += __shfl_xor(s, d);
  __syncthreads();  // a previous call's readers are done with smem
  if ((threadIdx.x & 63) < 4) smem[threadIdx.x >> 6][threadIdx.x & 3] = s;
  __syncthreads();
  const int cl = threadIdx.x & 3;
  return (smem[0][cl] + smem[1][cl]) + (smem[2][cl] + smem[3][cl]);
}
template <int LOADS>
__device__ __forceinline__ float lane_total(const float* __restrict__ part, int slices, int cols, int c) {
  float s = 0.f;
  for (int i = threadIdx.x >> 2; i < slices; i += 64 * LOADS) {
    float a[LOADS];
    for_slices<LOADS>(i, slices, cols, c, [&](int u, int64_t at, bool) { a[u] = part[at]; });
    for_slices<LOADS>(i, slices, cols, c, [&](int u, int64_t, bool in) { s += in ? a[u] : 0.f; });
  }
  return s;
}
__device__ __forceinline__ float slices_total(const float* __restrict__ part, int slices, int cols, int c, float (*smem)[FINISH_CHANNELS]) {
  return over_slice_lanes(slices <= 64 * FINISH_FEW ? lane_total<FINISH_FEW>(part, slices, cols, c) : lane_total<FINISH_LOADS>(part, slices, cols, c), smem);
}

// Finishing kernels: grid = ceil(C / FINISH_CHANNELS).
__global__ __launch_bounds__(256) void bn_mean_kernel(const float* __restrict__ part, int slices, int cols, float n, float* __restrict__ mean) {
  __shared__ float smem[4][FINISH_CHANNELS];
  const int c = blockIdx.x * FINISH_CHANNELS + (threadIdx.x & (FINISH_CHANNELS - 1));
  const float total = slices_total(part, slices, cols, c, smem);
  if (threadIdx.x < FINISH_CHANNELS && c < cols) mean[c] = total / n;
}

// What follows from a channel's statistics: r = 1/sqrt(var+eps), inv = r*gamma and, under the fused wiring, the statistics the
// reference hands to the gradient op: "mean" = the unbiased variance, "variance" = the mean.
struct BnScale {
  const float* gamma;
  float* mean;
  float* var;
  float* r;
  float* inv;
  float eps, unbias;
  float* g_mean;  // null: not the fused wiring
  float* g_r;
  float* g_inv;
};
__device__ __forceinline__ void bn_finish_channel(const BnScale& a, int c, float mean, float var) {
  a.mean[c] = mean;
  a.var[c] = var;
  const float rr = 1.0f / sqrtf(var + a.eps);
  a.r[c] = rr;
  a.inv[c] = rr * a.gamma[c];
  if (a.g_mean) {
    a.g_mean[c] = var * a.unbias;
    const float gr = 1.0f / sqrtf(mean + a.eps);   // NaN for a channel whose mean is below -epsilon, as in the reference
    a.g_r[c] = gr;
    a.g_inv[c] = gr * a.gamma[c];
  }
}
BnScale bn_scale_of(const BatchNormArgs& a, int64_t rows, bool wiring) {
  return BnScale{a.gamma, a.mean, a.var, a.r, a.inv, a.epsilon, (float)rows / (float)(rows > 1 ? rows - 1 : 1), wiring ? a.g_mean : nullptr, a.g_r, a.g_inv};
}

// var from the slices' squared deviations (training; the mean is known) or both from the moving statistics (part == null)
__global__ __launch_bounds__(256) void bn_scale_kernel(const float* __restrict__ part, int slices, int cols, float n,
                                                        const float* __restrict__ moving_mean, const float* __restrict__ moving_var, BnScale a) {
  __shared__ float smem[4][FINISH_CHANNELS];
  const int c = blockIdx.x * FINISH_CHANNELS + (threadIdx.x & (FINISH_CHANNELS - 1));
  float total = 0.f;
  if (part) total = slices_total(part, slices, cols, c, smem);  // uniform over the block
  if (threadIdx.x >= FINISH_CHANNELS || c >= cols) return;
  if (part) bn_finish_channel(a, c, a.mean[c], total / n);
  else bn_finish_channel(a, c, moving_mean[c], moving_var[c]);
}

// Joins slices of `whole` rows each (the last one: `last`).  Every thread of the block must call it.
template <int LOADS>
__device__ __forceinline__ void join_slices(const float* __restrict__ part_mean, const float* __restrict__ part_m2, int slices, int cols, int c, float whole,
                                            float last, float n, float (*smem)[FINISH_CHANNELS], float& mean, float& m2) {
  float pm[LOADS], pq[LOADS], s = 0.f, q = 0.f;
  const int first = threadIdx.x >> 2;
  for (int i = first; i < slices; i += 64 * LOADS) {
    for_slices<LOADS>(i, slices, cols, c, [&](int u, int64_t at, bool) { pm[u] = part_mean[at]; pq[u] = part_m2[at]; });
    for_slices<LOADS>(i, slices, cols, c, [&](int u, int64_t, bool in) { s += in ? pm[u] * (i + 64 * u + 1 < slices ? whole : last) : 0.f; });
  }
  mean = over_slice_lanes(s, smem) / n;
  for (int i = first; i < slices; i += 64 * LOADS) {
    if (slices > 64 * LOADS) for_slices<LOADS>(i, slices, cols, c, [&](int u, int64_t at, bool) { pm[u] = part_mean[at]; pq[u] = part_m2[at]; });
    for_slices<LOADS>(i, slices, cols, c, [&](int u, int64_t, bool in) {
      const float d = pm[u] - mean;
      q += in ? pq[u] + d * d * (i + 64 * u + 1 < slices ? whole : last) : 0.f;
    });
  }
  m2 = over_slice_lanes(q, smem);
}
__global__ __launch_bounds__(256) void bn_moments_kernel(const float* __restrict__ part_mean, const float* __restrict__ part_m2, int slices, int cols,
                                                          float whole, float last, float n, BnScale a) {
  __shared__ float smem[4][FINISH_CHANNELS];
  const int c = blockIdx.x * FINISH_CHANNELS + (threadIdx.x & (FINISH_CHANNELS - 1));
  float mean, m2;
  if (slices <= 64 * FINISH_FEW) join_slices<FINISH_FEW>(part_mean, part_m2, slices, cols, c, whole, last, n, smem, mean, m2);
  else join_slices<FINISH_LOADS>(part_mean, part_m2, slices, cols, c, whole, last, n, smem, mean, m2);
  if (threadIdx.x < FINISH_CHANNELS && c < cols) bn_finish_channel(a, c, mean, m2 / n);
}

template <bool V4>
__global__ __launch_bounds__(256) void bn_apply_kernel(const float* __restrict__ x, const float* __restrict__ mean,
                                                        const float* __restrict__ inv, const float* __restrict__ beta,
                                                        float* __restrict__ y, int64_t n, int cols, int centred) {
  // generic form: (x*inv - mean*inv) + beta (math/nn/AllKernels.scala:676-683); the fused op: (x - mean)*inv + beta
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  if (V4) {
    const int64_t n4 = n / 4;
    // the column walks with the index: one division at the start, then an addition and a wrap per trip
    const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int c = (int)((i0 * 4) % cols);
    const int cstep = (int)((stride * 4) % cols);
    for (int64_t i = i0; i < n4; i += stride, c = c + cstep >= cols ? c + cstep - cols : c + cstep) {
      const bn_f4 xv = *(const bn_f4*)(x + i * 4), iv = *(const bn_f4*)(inv + c), mv = *(const bn_f4*)(mean + c), bv = *(const bn_f4*)(beta + c);
      bn_f4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = centred ? (xv[e] - mv[e]) * iv[e] + bv[e] : (xv[e] * iv[e] - mv[e] * iv[e]) + bv[e];
      *(bn_f4*)(y + i * 4) = o;
    }
  } else {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
      const int c = (int)(i % cols);
      y[i] = centred ? (x[i] - mean[c]) * inv[c] + beta[c] : (x[i] * inv[c] - mean[c] * inv[c]) + beta[c];
    }
  }
}

// Normalisation and a 2 x 2 max pooling of the result in one pass: a thread normalises the four cells of a window (four channels)
// as bn_apply_kernel does and compares them as pool2x2_fwd_kernel (elementwise_kernels.hip) does; what lies between is not stored.
// [1000 x 26 x 26 x 32], stride 2: 24 us; the two passes took 28.7 + 23.6.
__global__ __launch_bounds__(256) void bn_pool2x2_fwd_kernel(const float* __restrict__ x, const float* __restrict__ mean,
                                                              const float* __restrict__ inv, const float* __restrict__ beta, float* __restrict__ y,
                                                              uint8_t* __restrict__ arg, uint32_t total, int cols, int centred, PoolWindows p) {
  const uint32_t cg = (uint32_t)cols / 4, stride = gridDim.x * blockDim.x;
  const uint32_t block = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);  // every XCD takes a contiguous run (the grid is a multiple of 8)
  for (uint32_t i = block * blockDim.x + threadIdx.x; i < total; i += stride) {
    const uint32_t win = div_by(i, p.by_cg), ch = (i - win * cg) * 4;
    const uint32_t row = div_by(win, p.by_wo), b = div_by(row, p.by_ho);
    const int ix0 = (int)(win - row * (uint32_t)p.wo) * p.sw - p.pl, iy0 = (int)(row - b * (uint32_t)p.ho) * p.sh - p.pt;
    const bn_f4 mv = *(const bn_f4*)(mean + ch), iv = *(const bn_f4*)(inv + ch), bv = *(const bn_f4*)(beta + ch);
    bn_f4 xv[4];
    bool in[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int iy = iy0 + (k >> 1), ix = ix0 + (k & 1);
      in[k] = (unsigned)iy < (unsigned)p.h && (unsigned)ix < (unsigned)p.w;
      xv[k] = *(const bn_f4*)(x + (in[k] ? ((b * p.h + iy) * p.w + ix) * cols + ch : 0u));
    }
    bn_f4 best = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    uint32_t at = 0u;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t place = 0u;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float v = centred ? (xv[k][e] - mv[e]) * iv[e] + bv[e] : (xv[k][e] * iv[e] - mv[e] * iv[e]) + bv[e];
        if (in[k] && v > best[e]) { best[e] = v; place = (uint32_t)k; }
      }
      at |= place << (8 * e);
    }
    *(bn_f4*)(y + i * 4) = best;
    *(uint32_t*)(arg + i * 4) = at;
  }
}

// d beta = S1, d gamma = S2 * r; k1 = S1/n, k2 = r*r*S2/n for the input gradient
__global__ __launch_bounds__(256) void bn_grad_finish_kernel(const float* __restrict__ part0, const float* __restrict__ part1, int slices,
                                                              int cols, float n, const float* __restrict__ r, float* __restrict__ dbeta,
                                                              float* __restrict__ dgamma, float* __restrict__ k1, float* __restrict__ k2) {
  __shared__ float smem[4][FINISH_CHANNELS];
  const int c = blockIdx.x * FINISH_CHANNELS + (threadIdx.x & (FINISH_CHANNELS - 1));
  const float s1 = slices_total(part0, slices, cols, c, smem);
  const float s2 = slices_total(part1, slices, cols, c, smem);
  if (threadIdx.x >= FINISH_CHANNELS || c >= cols) return;
  const float rr = r[c];
  dbeta[c] = s1;
  dgamma[c] = s2 * rr;
  k1[c] = s1 / n;
  k2[c] = rr * rr * s2 / n;
}

// Gradient of the activation that produced x (the layer below), from its output: models/Activation.scala:32-83.
__device__ __forceinline__ float below_act_grad(int act, float y, float dy, float param) {
  switch (act) {
    case SN_ACT_SIGMOID: return (y * (1.0f - y)) * dy;
    case SN_ACT_TANH: return (1.0f - y * y) * dy;
    case SN_ACT_RELU: return (param < y ? 1.0f : 0.0f) * dy;
    default: return dy;
  }
}

// dx = inv * (dy - k1 - (x - mean) * k2), then (act != identity) through the activation of the layer that wrote x
template <bool V4>
__global__ __launch_bounds__(256) void bn_dx_kernel(const float* __restrict__ x, const float* __restrict__ dy, const float* __restrict__ mean,
                                                     const float* __restrict__ inv, const float* __restrict__ k1,
                                                     const float* __restrict__ k2, float* __restrict__ dx, int64_t n, int cols, int act,
                                                     float act_param) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  if (V4) {
    const int64_t n4 = n / 4;
    const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int c = (int)((i0 * 4) % cols);
    const int cstep = (int)((stride * 4) % cols);
    for (int64_t i = i0; i < n4; i += stride, c = c + cstep >= cols ? c + cstep - cols : c + cstep) {
      const bn_f4 xv = *(const bn_f4*)(x + i * 4), gv = *(const bn_f4*)(dy + i * 4), iv = *(const bn_f4*)(inv + c),
                  mv = *(const bn_f4*)(mean + c), a = *(const bn_f4*)(k1 + c), b = *(const bn_f4*)(k2 + c);
      bn_f4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = below_act_grad(act, xv[e], iv[e] * ((gv[e] - a[e]) - (xv[e] - mv[e]) * b[e]), act_param);
      *(bn_f4*)(dx + i * 4) = o;
    }
  } else {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
      const int c = (int)(i % cols);
      dx[i] = below_act_grad(act, x[i], inv[c] * ((dy[i] - k1[c]) - (x[i] - mean[c]) * k2[c]), act_param);
    }
  }
}

// decayingAvg (alg/AllKernels.scala:541-544): moving = momentum*moving + (1-momentum)*batch
__global__ __launch_bounds__(256) void bn_moving_kernel(float* __restrict__ moving_mean, float* __restrict__ moving_var,
                                                         const float* __restrict__ mean, const float* __restrict__ var, int cols, float momentum) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= cols) return;
  const float keep = 1.0f - momentum;
  moving_mean[c] = momentum * moving_mean[c] + keep * mean[c];
  moving_var[c] = momentum * moving_var[c] + keep * var[c];
}

unsigned grid_for(const sn_ctx* ctx, int64_t n, int per_block) {
  int64_t blocks = ceil_div(n, per_block);
  const int64_t cap = (int64_t)ctx->compute_units * 16;
  if (blocks > cap) blocks = cap;
  return blocks < 1 ? 1u : (unsigned)blocks;
}

bool stream_ok(int cols, const void* x, const void* dy, const void* part0, int64_t part1_offset) {
  return bn_stream_form(cols) && part1_offset % 4 == 0 &&
         ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(dy) | reinterpret_cast<uintptr_t>(part0)) & 15u) == 0;
}

// One row-walking reduction pass; returns the number of slices written to part0 (and part1).
template <int MODE>
int reduce_rows(sn_ctx* ctx, const float* x, const float* dy, const float* mean, float* part0, float* part1, int64_t rows, int cols) {
  const int s = bn_row_slices(ctx->compute_units, rows, cols);
  hipLaunchKernelGGL((bn_reduce_kernel<MODE>), dim3((unsigned)ceil_div((int64_t)cols, (int64_t)64), (unsigned)s), dim3(256), 0, ctx->stream, x, dy,
                     mean, part0, part1, rows, cols, ceil_div(rows, (int64_t)s));
  return s;
}

bool vec4_ok(int cols, std::initializer_list<const void*> ptrs) {
  if (cols % 4 != 0) return false;
  for (const void* p : ptrs)
    if (reinterpret_cast<uintptr_t>(p) & 15u) return false;
  return true;
}

}  // namespace

int64_t batchnorm_workspace_elems(const sn_ctx* ctx, int64_t rows, int cols) { return (int64_t)2 * bn_max_slices(ctx->compute_units, rows, cols) * cols; }

ConvStats batchnorm_conv_stats(const sn_ctx* ctx, int64_t rows, int cols, float* ws, int64_t ws_elems) {
  ConvStats st;
  const int64_t slices = bn_max_slices(ctx->compute_units, rows, cols), half = slices * cols;
  if (ws && 2 * half <= ws_elems) {
    st.part_mean = ws;
    st.part_m2 = ws + half;
    st.max_slices = (int)slices;
  }
  return st;
}

// mean, var and what follows from them (BnScale)
static int batchnorm_statistics(sn_ctx* ctx, const float* x, int64_t rows, int cols, const BatchNormArgs& a, bool training, float* ws,
                                int64_t ws_elems, const ConvStats* stats) {
  SN_REQUIRE(rows * cols <= (int64_t)INT32_MAX * 4, "batch norm over %lld elements exceeds one launch", (long long)(rows * cols));
  const int cb = (int)ceil_div((int64_t)cols, (int64_t)FINISH_CHANNELS);
  if (!training) {
    LaunchScope scope(ctx, "batchnorm_frozen_scale");
    hipLaunchKernelGGL(bn_scale_kernel, dim3(cb), dim3(256), 0, ctx->stream, (const float*)nullptr, 0, cols, 1.0f, a.moving_mean, a.moving_var,
                       bn_scale_of(a, rows, false));
    SN_HIP(hipGetLastError());
    return SN_OK;
  }
  const int64_t half = (int64_t)bn_max_slices(ctx->compute_units, rows, cols) * cols;
  const BnScale scale = bn_scale_of(a, rows, a.fused_wiring);
  SN_REQUIRE(half <= ws_elems, "batch norm needs %lld workspace elements, %lld given", (long long)half, (long long)ws_elems);
  if (stats && stats->slices > 0) {
    LaunchScope scope(ctx, "batchnorm_mean_and_variance_from_convolution");
    hipLaunchKernelGGL(bn_moments_kernel, dim3(cb), dim3(256), 0, ctx->stream, (const float*)stats->part_mean, (const float*)stats->part_m2, stats->slices,
                       cols, stats->whole, stats->last, (float)rows, scale);
  } else if (2 * half <= ws_elems && stream_ok(cols, x, nullptr, ws, half)) {
    const BnStream st = bn_stream_of(ctx->compute_units, rows, cols);
    LaunchScope scope(ctx, "batchnorm_mean_and_variance");
    hipLaunchKernelGGL(bn_stats_v4_kernel, dim3((unsigned)st.slices), dim3(256), 0, ctx->stream, (const bn_f4*)x, ws, ws + half, st.n4, cols, st.active,
                       st.per4);
    hipLaunchKernelGGL(bn_moments_kernel, dim3(cb), dim3(256), 0, ctx->stream, (const float*)ws, (const float*)(ws + half), st.slices, cols,
                       (float)(st.per4 / (cols / 4)), (float)((st.n4 - (st.slices - 1) * st.per4) / (cols / 4)), (float)rows, scale);
  } else {
    {
      LaunchScope scope(ctx, "batchnorm_mean");
      const int s = reduce_rows<BN_SUM>(ctx, x, nullptr, nullptr, ws, nullptr, rows, cols);
      hipLaunchKernelGGL(bn_mean_kernel, dim3(cb), dim3(256), 0, ctx->stream, (const float*)ws, s, cols, (float)rows, a.mean);
    }
    LaunchScope scope(ctx, "batchnorm_variance");
    const int s = reduce_rows<BN_SQDIFF>(ctx, x, nullptr, a.mean, ws, nullptr, rows, cols);
    hipLaunchKernelGGL(bn_scale_kernel, dim3(cb), dim3(256), 0, ctx->stream, (const float*)ws, s, cols, (float)rows, (const float*)nullptr,
                       (const float*)nullptr, scale);
  }
  SN_HIP(hipGetLastError());
  return SN_OK;
}

int launch_batchnorm_fwd(sn_ctx* ctx, const float* x, float* y, int64_t rows, int cols, const BatchNormArgs& a, bool training, float* ws,
                         int64_t ws_elems, const ConvStats* stats) {
  if (rows <= 0 || cols <= 0) return SN_OK;
  SN_TRY(batchnorm_statistics(ctx, x, rows, cols, a, training, ws, ws_elems, stats));
  const int64_t n = rows * cols;
  LaunchScope scope(ctx, "batchnorm_apply");
  if (vec4_ok(cols, {x, y, a.mean, a.inv, a.beta}))
    hipLaunchKernelGGL((bn_apply_kernel<true>), dim3(grid_for(ctx, n / 4, 1024)), dim3(256), 0, ctx->stream, x, (const float*)a.mean,
                       (const float*)a.inv, a.beta, y, n, cols, a.fused_wiring ? 1 : 0);
  else
    hipLaunchKernelGGL((bn_apply_kernel<false>), dim3(grid_for(ctx, n, 1024)), dim3(256), 0, ctx->stream, x, (const float*)a.mean,
                       (const float*)a.inv, a.beta, y, n, cols, a.fused_wiring ? 1 : 0);
  SN_HIP(hipGetLastError());
  return SN_OK;
}

static PoolWindows pool_windows(const PoolGeom& g) {
  return PoolWindows{g.h, g.w, g.ho, g.wo, g.sh, g.sw, g.pt, g.pl, fast_div((uint32_t)(g.c / 4)), fast_div((uint32_t)g.wo), fast_div((uint32_t)g.ho)};
}

// 2 x 2 maxima of whole vectors of channels with 32-bit element indices: what the pooling's own kernel for such windows takes
bool batchnorm_pool_ok(const PoolGeom& g, const BatchNormArgs& a, const float* x, const float* y, const uint8_t* arg) {
  return g.kh == 2 && g.kw == 2 && g.n > 0 && g.c <= 1024 && (int64_t)g.n * g.h * g.w * g.c < (1ll << 31) && (int64_t)g.n * g.ho * g.wo * g.c < (1ll << 31) &&
         (int64_t)g.n * g.ho * g.wo * g.c > 0 && vec4_ok(g.c, {x, y, a.mean, a.inv, a.g_mean, a.g_inv, a.k1, a.k2, a.beta}) &&
         (reinterpret_cast<uintptr_t>(arg) & 15u) == 0;
}

int launch_batchnorm_pool_fwd(sn_ctx* ctx, const float* x, float* y, uint8_t* arg, const PoolGeom& g, const BatchNormArgs& a, bool training, float* ws,
                              int64_t ws_elems, const ConvStats* stats) {
  SN_TRY(batchnorm_statistics(ctx, x, (int64_t)g.n * g.h * g.w, g.c, a, training, ws, ws_elems, stats));
  const int64_t total = (int64_t)g.n * g.ho * g.wo * g.c / 4;
  LaunchScope scope(ctx, "batchnorm_apply_and_maxpool");
  hipLaunchKernelGGL(bn_pool2x2_fwd_kernel, dim3((grid_for(ctx, total, 256) + 7u) & ~7u), dim3(256), 0, ctx->stream, x, (const float*)a.mean,
                     (const float*)a.inv, a.beta, y, arg, (uint32_t)total, g.c, a.fused_wiring ? 1 : 0, pool_windows(g));
  SN_HIP(hipGetLastError());
  return SN_OK;
}

// d beta, d gamma, k1, k2 from the slices of the two gradient sums
static void grad_finish(sn_ctx* ctx, const float* part0, const float* part1, int slices, int64_t rows, int cols, const BatchNormArgs& a, float* dbeta,
                        float* dgamma) {
  hipLaunchKernelGGL(bn_grad_finish_kernel, dim3((unsigned)ceil_div((int64_t)cols, (int64_t)FINISH_CHANNELS)), dim3(256), 0, ctx->stream, part0, part1, slices, cols,
                     (float)rows, a.fused_wiring ? (const float*)a.g_r : (const float*)a.r, dbeta, dgamma, a.k1, a.k2);
}

int launch_batchnorm_pool_bwd(sn_ctx* ctx, const float* x, const float* dy, const uint8_t* arg, const PoolGeom& g, const BatchNormArgs& a, float* dbeta,
                              float* dgamma, float* ws, int64_t ws_elems) {
  const int64_t rows = (int64_t)g.n * g.h * g.w;
  const int64_t half = (int64_t)bn_max_slices(ctx->compute_units, rows, g.c) * g.c;
  SN_REQUIRE(2 * half <= ws_elems, "batch norm gradient needs %lld workspace elements, %lld given", (long long)(2 * half), (long long)ws_elems);
  const int cg = g.c / 4, active = 256 / cg * cg;
  const int64_t n4 = (int64_t)g.n * g.ho * g.wo * cg;
  const int64_t wanted = std::min<int64_t>(ceil_div(n4, (int64_t)4 * active), bn_max_slices(ctx->compute_units, rows, g.c));
  const int64_t per4 = ceil_div(ceil_div(n4, wanted), (int64_t)active) * active;
  const int slices = (int)ceil_div(n4, per4);
  LaunchScope scope(ctx, "batchnorm_gradient_sums_from_maxpool");
  hipLaunchKernelGGL(bn_pool_grad_sums_kernel, dim3((unsigned)slices), dim3(256), 0, ctx->stream, x, (const bn_f4*)dy, (const uint32_t*)arg,
                     a.fused_wiring ? (const float*)a.g_mean : (const float*)a.mean, ws, ws + half, (uint32_t)n4, g.c, active, (uint32_t)per4, pool_windows(g));
  grad_finish(ctx, ws, ws + half, slices, rows, g.c, a, dbeta, dgamma);
  SN_HIP(hipGetLastError());
  return SN_OK;
}

int launch_batchnorm_bwd(sn_ctx* ctx, const float* x, const float* dy, float* dx, int64_t rows, int cols, const BatchNormArgs& a,
                         float* dbeta, float* dgamma, float* ws, int64_t ws_elems, int below_act, float below_act_param) {
  if (rows <= 0 || cols <= 0) return SN_OK;
  const int64_t half = (int64_t)bn_max_slices(ctx->compute_units, rows, cols) * cols;
  SN_REQUIRE(2 * half <= ws_elems, "batch norm gradient needs %lld workspace elements, %lld given", (long long)(2 * half), (long long)ws_elems);
  float* part1 = ws + half;
  const float* mean = a.fused_wiring ? a.g_mean : a.mean;
  const float* inv = a.fused_wiring ? a.g_inv : a.inv;
  {
    LaunchScope scope(ctx, "batchnorm_gradient_sums");
    int s = 0;
    if (stream_ok(cols, x, dy, ws, half)) {
      const BnStream st = bn_stream_of(ctx->compute_units, rows, cols);
      s = st.slices;
      hipLaunchKernelGGL(bn_grad_sums_v4_kernel, dim3((unsigned)s), dim3(256), 0, ctx->stream, (const bn_f4*)x, (const bn_f4*)dy, mean, ws, part1, st.n4,
                         cols, st.active, st.per4);
    } else {
      s = reduce_rows<BN_GRAD>(ctx, x, dy, mean, ws, part1, rows, cols);
    }
    grad_finish(ctx, ws, part1, s, rows, cols, a, dbeta, dgamma);
  }
  if (dx) {
    const int64_t n = rows * cols;
    LaunchScope scope(ctx, "batchnorm_input_gradient");
    if (vec4_ok(cols, {x, dy, dx, mean, inv, a.k1, a.k2}))
      hipLaunchKernelGGL((bn_dx_kernel<true>), dim3(grid_for(ctx, n / 4, 1024)), dim3(256), 0, ctx->stream, x, dy, mean, inv,
                         (const float*)a.k1, (const float*)a.k2, dx, n, cols, below_act, below_act_param);
    else
      hipLaunchKernelGGL((bn_dx_kernel<false>), dim3(grid_for(ctx, n, 1024)), dim3(256), 0, ctx->stream, x, dy, mean, inv,
                         (const float*)a.k1, (const float*)a.k2, dx, n, cols, below_act, below_act_param);
  }
  SN_HIP(hipGetLastError());
  return SN_OK;
}

int launch_batchnorm_moving(sn_ctx* ctx, const BatchNormArgs& a, float* moving_mean, float* moving_var, int cols) {
  if (cols <= 0) return SN_OK;
  LaunchScope scope(ctx, "batchnorm_moving_statistics");
  hipLaunchKernelGGL(bn_moving_kernel, dim3((unsigned)ceil_div((int64_t)cols, (int64_t)256)), dim3(256), 0, ctx->stream, moving_mean,
                     moving_var, (const float*)a.mean, (const float*)(a.fused_wiring ? a.mean : a.var), cols, a.momentum);
  SN_HIP(hipGetLastError());
  return SN_OK;
}

}  // namespace sn
