// First-layer Conv2D (one to four input channels) on the float32 matrix instruction: filter gradient, then forward.
//
//   dW[m, co] = sum over positions p of x(p, m) * d(p, co),   m = (r, q, ci) a few dozen taps, co at most 64 filters
//
// The product is tiny (M x N a few 16 x 16 tiles) and its reduction as long as the batch has output positions, so what it costs is
// getting the operands to the matrix cores.  v_mfma_f32_16x16x4_f32 takes one value of each operand a lane: tap l % 16 at position
// l / 16 of one, filter l % 16 at position l / 16 of the other, and four positions of a row are what 64 lanes
// load in one go (a contiguous run of d; of x a gather that the first-level cache answers).  Nothing is staged, nothing
// waits for a barrier: a wavefront walks its own rows of output positions and keeps all sums.  (The form this replaces kept a filter a
// lane and every tap's sum in registers: 11 LDS reads for 9 multiply-adds.)
//
// POOL: d is not in memory.  A 2 x 2 max pooling sits right above the layer and d is worked out from the pooling's output
// gradient, the recorded first-maximum offsets and the convolution's saved output y (for its activation gradient), exactly as
// pool2x2_bwd_kernel does: an element lies in at most 2 x 2 windows, whose contributions are added in (oh, ow) order, then
// act'(y) multiplies.  With a batch normalisation in between (bn_inv) its input gradient is formed on the way as well.
//
// Measured, with what the launch takes over: 27 taps x 48 filters over 125 x 32 x 32 positions under a pooling of stride 2, 50.4 -> 14.2 us;
// 9 x 32 over 1000 x 26 x 26 under a batch normalisation and a pooling 88 -> 34.9 us (it reads 114 MB); 9 x 32 over 100 x 26 x 26
// under a pooling of stride 1, 11.1 -> 9.3 us.
#include "common.hpp"
#include "conv_first_rules.hpp"
#include "moments.hpp"

#include <algorithm>

namespace sn {
namespace {

typedef float f4v __attribute__((ext_vector_type(4)));

struct FirstWgrad {
  ConvGeom g;
  const float* x;
  const float* dy;      // [n, ho, wo, cout], POOL: not read
  float* partial;       // [block][M][cout]
  int M, items;  // taps; n * ho rows in segments
  FirstWgradCut cut;
  FastDiv by_segments, by_ho, by_cin, by_kw, by_cout;
  PoolGrad pool;
};

__device__ __forceinline__ float first_act_grad(int act, float y, float dy, float param) {  // elementwise_kernels.hip: act_bwd
  switch (act) {
    case SN_ACT_SIGMOID: return (y * (1.0f - y)) * dy;
    case SN_ACT_TANH: return (1.0f - y * y) * dy;
    case SN_ACT_RELU: return (param < y ? 1.0f : 0.0f) * dy;
    default: return dy;
  }
}

// V consecutive values (V * 4 bytes aligned) or bytes
template <int V>
__device__ __forceinline__ void load_values(const float* p, float* v) {
  typedef float vec __attribute__((ext_vector_type(V)));
  if constexpr (V == 1) v[0] = *p;
  else {
    const vec x = *(const vec*)p;
#pragma unroll
    for (int i = 0; i < V; ++i) v[i] = x[i];
  }
}
template <int V>
__device__ __forceinline__ uint32_t load_bytes(const uint8_t* p) {
  if constexpr (V == 1) return *p;
  else if constexpr (V == 2) return *(const uint16_t*)p;
  else return *(const uint32_t*)p;
}

// MT x NT tiles of 16 taps x 16 filters.  VEC: a lane's NT filters are neighbours, loaded as one vector; otherwise they are 16 apart.
// S (POOL only): the pooling's strides if both are 1 or both are 2, else 0; with 2 a position lies in one window.
template <int MT, int NT, bool VEC, bool POOL, int S>
__global__ __launch_bounds__(256) void conv_first_wgrad_kernel(FirstWgrad k) {
  extern __shared__ float lds[];  // [wavefront][MT * 16][NT * 16]
  const ConvGeom& g = k.g;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int l16 = lane & 15, lp = lane >> 4;
  constexpr int G = 4;                  // groups of four positions in flight
  constexpr int V = VEC ? NT : 1, NV = NT / V;
  constexpr int WIN = S == 2 ? 1 : 4;   // windows a position may lie in

  // this lane's taps (those that do not exist repeat the last one: their sums are dropped) and filters
  int tap_y[MT], tap_x[MT], tap_off[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const uint32_t m = (uint32_t)min(16 * i + l16, k.M - 1), rq = div_by(m, k.by_cin), r = div_by(rq, k.by_kw);
    tap_y[i] = (int)r - g.pt;
    tap_x[i] = (int)(rq - r * (uint32_t)g.kw) - g.pl;
    tap_off[i] = (tap_y[i] * g.w + tap_x[i]) * g.cin + (int)(m - rq * (uint32_t)g.cin);
  }
  int ch[NV];
#pragma unroll
  for (int t = 0; t < NV; ++t) ch[t] = VEC ? min(NT * l16, g.cout - NT) : min(16 * t + l16, g.cout - 1);
  float bn_mean[NT], bn_inv[NT], bn_k1[NT], bn_k2[NT];
  const bool bn = POOL && k.pool.bn_inv != nullptr;
  if (bn) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int c = ch[t / V] + t % V;
      bn_mean[t] = k.pool.bn_mean[c];
      bn_inv[t] = k.pool.bn_inv[c];
      bn_k1[t] = k.pool.bn_k1[c];
      bn_k2[t] = k.pool.bn_k2[c];
    }
  }
  f4v acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[i][t] = f4v{0.f, 0.f, 0.f, 0.f};

  // every XCD (workgroup id modulo 8) takes a contiguous run of rows, or of their segments
  const int per_xcd = ((int)gridDim.x + 7) >> 3, extra = (int)gridDim.x - (per_xcd - 1) * 8;  // `extra` XCDs have per_xcd workgroups, the others one less
  const int xcd = (int)blockIdx.x & 7;
  const int block = xcd * (per_xcd - 1) + min(xcd, extra) + ((int)blockIdx.x >> 3);
  const int item0 = (block * 4 + wave) * k.cut.items_per_wave, item1 = min(k.items, item0 + k.cut.items_per_wave);
  const PoolGrad& pg = k.pool;
  for (int item = item0; item < item1; ++item) {
    const int row = (int)div_by((uint32_t)item, k.by_segments);
    const int ow_begin = (item - row * k.cut.segments) * k.cut.segment_length, ow_end = min(g.wo, ow_begin + k.cut.segment_length);
    const int b = (int)div_by((uint32_t)row, k.by_ho), oh = row - b * g.ho;
    const float* const xb = k.x + (int64_t)b * g.h * g.w * g.cin;
    const int iy = oh * g.sh, x_row = iy * g.w * g.cin;
    const float* const d_row = (POOL ? pg.y : k.dy) + (int64_t)row * g.wo * g.cout;
    // the pooling's rows of windows this row of positions lies in: oh_lo, and oh_lo + 1 where that is still <= oh_hi
    int oh_lo = 0, oh_hi = 0;
    const float* pd_row = nullptr;
    const uint8_t* pa_row = nullptr;
    if constexpr (POOL) {
      if constexpr (S == 2) oh_lo = oh_hi = (oh + pg.pt) >> 1;
      else {
        const int lo = oh + pg.pt - 1;
        oh_lo = lo <= 0 ? 0 : (S == 1 ? lo : (lo + pg.sh - 1) / pg.sh);
        oh_hi = S == 1 ? oh + pg.pt : (oh + pg.pt) / pg.sh;
      }
      oh_hi = min(oh_hi, pg.ho - 1);
      const int64_t first = ((int64_t)b * pg.ho + min(oh_lo, pg.ho - 1)) * pg.wo * g.cout;
      pd_row = pg.dy + first;
      pa_row = pg.arg + first;
    }
    for (int ow0 = ow_begin; ow0 < ow_end; ow0 += 4 * G) {
      float a[G][MT], y[G][NT], pd[G][WIN][NT];
      uint32_t pa[G][WIN][NV], want[G][WIN];
#pragma unroll
      for (int u = 0; u < G; ++u) {
        const int at = ow0 + 4 * u + lp, ow = min(at, g.wo - 1);
        const bool on = at < g.wo;
        const int ix = ow * g.sw;
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          const bool in = on && (unsigned)(iy + tap_y[i]) < (unsigned)g.h && (unsigned)(ix + tap_x[i]) < (unsigned)g.w;
          const float v = xb[in ? x_row + ix * g.cin + tap_off[i] : 0];
          a[u][i] = in ? v : 0.f;
        }
#pragma unroll
        for (int t = 0; t < NV; ++t) load_values<V>(d_row + (ow * g.cout + ch[t]), &y[u][t * V]);
        if constexpr (POOL) {
          int ow_lo, ow_hi;
          if constexpr (S == 2) ow_lo = ow_hi = (ow + pg.pl) >> 1;
          else {
            const int lo = ow + pg.pl - 1;
            ow_lo = lo <= 0 ? 0 : (S == 1 ? lo : (lo + pg.sw - 1) / pg.sw);
            ow_hi = S == 1 ? ow + pg.pl : (ow + pg.pl) / pg.sw;
          }
          ow_hi = min(ow_hi, pg.wo - 1);
#pragma unroll
          for (int w = 0; w < WIN; ++w) {  // windows that do not exist re-read the row's first element and match no place
            const int wh = oh_lo + (w >> 1), ww = ow_lo + (w & 1);
            const bool there = on && wh <= oh_hi && ww <= ow_hi;
            want[u][w] = there ? (uint32_t)((oh - (wh * (S ? S : pg.sh) - pg.pt)) * 2 + (ow - (ww * (S ? S : pg.sw) - pg.pl))) : 255u;
            const int o = there ? ((w >> 1) * pg.wo + ww) * g.cout : 0;
#pragma unroll
            for (int t = 0; t < NV; ++t) {
              pa[u][w][t] = load_bytes<V>(pa_row + (o + ch[t]));
              load_values<V>(pd_row + (o + ch[t]), &pd[u][w][t * V]);
            }
          }
        } else {
#pragma unroll
          for (int t = 0; t < NT; ++t) y[u][t] = on ? y[u][t] : 0.f;
        }
      }
#pragma unroll
      for (int u = 0; u < G; ++u) {
        if (ow0 + 4 * u >= ow_end) break;
        float d[NT];
        if constexpr (POOL) {
          const bool on = ow0 + 4 * u + lp < g.wo;
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            float s = 0.f;
#pragma unroll
            for (int w = 0; w < WIN; ++w)
              if (((pa[u][w][t / V] >> (8 * (t % V))) & 255u) == want[u][w]) s += pd[u][w][t];
            if (bn) s = bn_inv[t] * ((s - bn_k1[t]) - (y[u][t] - bn_mean[t]) * bn_k2[t]);
            d[t] = s;
          }
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            d[t] = first_act_grad(pg.act, y[u][t], d[t], pg.act_param);
            d[t] = on ? d[t] : 0.f;
          }
        } else {
#pragma unroll
          for (int t = 0; t < NT; ++t) d[t] = y[u][t];
        }
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int t = 0; t < NT; ++t) acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][i], d[t], acc[i][t], 0, 0, 0);
      }
    }
  }
  // value v of a lane: tap 4 (lane / 16) + v of its tile, the lane's filter
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) lds[(wave * MT * 16 + 16 * i + 4 * lp + v) * (NT * 16) + (VEC ? NT * l16 + t : 16 * t + l16)] = acc[i][t][v];
  __syncthreads();
  const int outs = k.M * g.cout;
  float* const out = k.partial + (int64_t)blockIdx.x * outs;
  for (int o = threadIdx.x; o < outs; o += 256) {
    const int m = (int)div_by((uint32_t)o, k.by_cout), c = o - m * g.cout;
    constexpr int TILE = MT * 16 * NT * 16;
    const float* at = lds + m * (NT * 16) + c;
    out[o] = (at[0] + at[TILE]) + (at[2 * TILE] + at[3 * TILE]);
  }
}

template <int MT, int NT, bool VEC>
int launch_tiles(sn_ctx* ctx, const FirstWgrad& k, int blocks, bool pool) {
  const size_t lds = (size_t)4 * MT * 16 * NT * 16 * sizeof(float);
  const int S = k.pool.sh == k.pool.sw && k.pool.sh <= 2 ? k.pool.sh : 0;
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), lds, ctx->stream, k); };
  if (!pool) launch(conv_first_wgrad_kernel<MT, NT, VEC, false, 0>);
  else if (S == 1) launch(conv_first_wgrad_kernel<MT, NT, VEC, true, 1>);
  else if (S == 2) launch(conv_first_wgrad_kernel<MT, NT, VEC, true, 2>);
  else launch(conv_first_wgrad_kernel<MT, NT, VEC, true, 0>);
  SN_HIP(hipGetLastError());
  return SN_OK;
}
template <int MT>
int launch_taps(sn_ctx* ctx, const FirstWgrad& k, int blocks, bool pool, bool vec) {
  switch (ceil_div(k.g.cout, 16)) {
    case 1: return launch_tiles<MT, 1, false>(ctx, k, blocks, pool);
    case 2: return vec ? launch_tiles<MT, 2, true>(ctx, k, blocks, pool) : launch_tiles<MT, 2, false>(ctx, k, blocks, pool);
    case 3: return launch_tiles<MT, 3, false>(ctx, k, blocks, pool);
    default: return vec ? launch_tiles<MT, 4, true>(ctx, k, blocks, pool) : launch_tiles<MT, 4, false>(ctx, k, blocks, pool);
  }
}

}  // namespace

constexpr int FIRST_MAX_TAPS = 48, FIRST_MAX_FILTERS = 64, FIRST_MIN_POSITIONS = 2048;
static FirstWgradCut first_wgrad_cut(const sn_ctx* ctx, const ConvGeom& g, const float* ws, int64_t ws_elems) {
  const int M = g.kh * g.kw * g.cin, N = g.cout;
  const int64_t rows = (int64_t)g.n * g.ho;
  if (!ws || g.cin > 4 || M > FIRST_MAX_TAPS || N > FIRST_MAX_FILTERS || rows * g.wo < FIRST_MIN_POSITIONS) return {};
  if (rows >= (1ll << 30) || (int64_t)g.h * g.w * g.cin >= (1ll << 30) || (int64_t)(g.wo + 1) * 2 * N >= (1ll << 30)) return {};  // 32-bit offsets inside an image and two rows
  const int64_t room = std::min<int64_t>((int64_t)4 * ctx->compute_units, ws_elems / ((int64_t)M * N));
  if (room < 32) return {};
  return conv_first_wgrad_cut(rows, g.wo, room);  // as many wavefronts as there are rows or segments, up to four on a SIMD
}
int conv_first_wgrad_parts(const sn_ctx* ctx, const ConvGeom& g, const float* ws, int64_t ws_elems) { return first_wgrad_cut(ctx, g, ws, ws_elems).parts; }

int launch_conv_first_wgrad(sn_ctx* ctx, const ConvGeom& g, const float* x, const float* dy, float* ws, int64_t ws_elems, const PoolGrad* pool, int* parts) {
  FirstWgrad k{};
  k.cut = first_wgrad_cut(ctx, g, ws, ws_elems);
  *parts = k.cut.parts;
  SN_REQUIRE(*parts > 0, "conv2d_filter_gradient_first: shape outside the kernel's range");
  k.g = g;
  k.x = x;
  k.dy = dy;
  k.partial = ws;
  k.M = g.kh * g.kw * g.cin;
  k.items = g.n * g.ho * k.cut.segments;
  k.by_segments = fast_div((uint32_t)k.cut.segments);
  k.by_ho = fast_div((uint32_t)g.ho);
  k.by_cin = fast_div((uint32_t)g.cin);
  k.by_kw = fast_div((uint32_t)g.kw);
  k.by_cout = fast_div((uint32_t)g.cout);
  if (pool) k.pool = *pool;
  const int N = g.cout, nt = (int)ceil_div(N, 16);
  auto at16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  const bool vec = N % nt == 0 && N % 2 == 0 && (pool ? at16(pool->dy) && at16(pool->y) && at16(pool->arg) : at16(dy));
  LaunchScope scope(ctx, pool ? "maxpool_backward_and_conv2d_filter_gradient_direct" : "conv2d_filter_gradient_direct", k.M, N, g.n * g.ho * g.wo);
  if (k.M <= 16) return launch_taps<1>(ctx, k, *parts, pool != nullptr, vec);
  if (k.M <= 32) return launch_taps<2>(ctx, k, *parts, pool != nullptr, vec);
  return launch_taps<3>(ctx, k, *parts, pool != nullptr, vec);
}

namespace {

// ============================================================================ forward
// out[p, co] = act(sum over m of x(p, m) * w[m, co] + bias[co]) on the same instruction, 16 consecutive output positions as its rows and
// filters as its columns.  A lane ends with its filters of four positions, and 16 neighbouring lanes with one run of
// filters: every store of 64 lanes writes four whole runs.  (With the filters as rows a lane holds four neighbouring filters
// of one position, and a store scatters 64 pieces of 16 bytes: 30 us instead of 22 for 676000 positions x 32 with STATS.)  The weights
// stay in registers; x is gathered one value a lane and four taps a step, the next tile's values while this one is multiplied.
//
// STATS: a batch normalisation follows.  Every lane keeps mean and squared deviations of its filters over its positions, four at a
// time as bn_stats_v4_kernel does eight; lanes and wavefronts join theirs pairwise, and a workgroup leaves one slice of
// partial statistics: the normalisation need not read the tensor for them.
// Measured against the kernels this replaces (filters in LDS or registers, vector multiply-adds): 27 taps x 48 filters, 128000 positions
// 34.4 -> 17.4 us; 9 x 32, 67600 positions 7.2 -> 6.7; 9 x 32, 676000 positions with STATS 28.0, before 22.4 and 17.1 for the statistics.
struct FirstForward {
  ConvGeom g;
  const float* x;
  const float* w;
  Epilogue e;
  int taps, positions, tiles_per_block;  // a workgroup takes tiles_per_block * 16 consecutive positions
  FastDiv by_wo, by_ho, by_cin, by_kw;
  float* part_mean;  // STATS: [slice][cout]
  float* part_m2;
};

template <int N>
__device__ __forceinline__ void first_act(int act, float (&v)[N], float param) {  // split_gemm.hpp: ep_act_block
  switch (act) {
    case SN_ACT_SIGMOID:
#pragma unroll
      for (int i = 0; i < N; ++i) v[i] = 1.0f / (1.0f + expf(-v[i]));
      break;
    case SN_ACT_TANH:
#pragma unroll
      for (int i = 0; i < N; ++i) v[i] = tanhf(v[i]);
      break;
    case SN_ACT_RELU:
#pragma unroll
      for (int i = 0; i < N; ++i) v[i] = fmaxf(param, v[i]);
      break;
    default: break;
  }
}

// KS steps of four taps, NT tiles of 16 filters (blockIdx.y: which 16 NT of them).  With two or four tiles a lane's NT filters are neighbours
// and leave as one vector (conv_first_fwd_ok: whole vectors of filters, 16-byte aligned), with three they are 16 apart.
template <int KS, int NT, bool STATS>
__global__ __launch_bounds__(256) void conv_first_fwd_kernel(FirstForward k) {
  constexpr bool VEC = NT == 2 || NT == 4;
  __shared__ float moments[STATS ? 4 : 1][2][STATS ? 16 * NT : 1];
  __shared__ float counts[4];
  const ConvGeom& g = k.g;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int l16 = lane & 15, lq = lane >> 4;
  const int co0 = (int)blockIdx.y * (16 * NT);
  int tap_y[KS], tap_x[KS], tap_off[KS];
  float wv[KS][NT], bias[NT];
  int ch[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    ch[t] = co0 + (VEC ? NT * l16 + t : 16 * t + l16);
    bias[t] = k.e.bias && ch[t] < g.cout ? k.e.bias[ch[t]] : 0.f;
  }
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int m = 4 * s + lq;
    const uint32_t mm = (uint32_t)min(m, k.taps - 1), rq = div_by(mm, k.by_cin), r = div_by(rq, k.by_kw);
    tap_y[s] = (int)r - g.pt;
    tap_x[s] = (int)(rq - r * (uint32_t)g.kw) - g.pl;
    tap_off[s] = (tap_y[s] * g.w + tap_x[s]) * g.cin + (int)(mm - rq * (uint32_t)g.cin);
    if (m >= k.taps) tap_y[s] = -(1 << 20);  // outside every image: a tap that does not exist reads a zero
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const float v = k.w[(int64_t)mm * g.cout + min(ch[t], g.cout - 1)];
      wv[s][t] = m < k.taps && ch[t] < g.cout ? v : 0.f;
    }
  }
  const int per_xcd = ((int)gridDim.x + 7) >> 3, extra = (int)gridDim.x - (per_xcd - 1) * 8;  // (as in conv_first_wgrad_kernel)
  const int xcd = (int)blockIdx.x & 7;
  const int block = xcd * (per_xcd - 1) + min(xcd, extra) + ((int)blockIdx.x >> 3);
  const int p_begin = block * k.tiles_per_block * 16, p_end = min(k.positions, p_begin + k.tiles_per_block * 16);
  float n = 0.f, mean[NT], m2[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) mean[t] = m2[t] = 0.f;
  auto gather = [&](int p0, float (&xv)[KS]) {  // positions behind the end repeat the last one
    const uint32_t p = (uint32_t)min(p0 + l16, k.positions - 1), row = div_by(p, k.by_wo), b = div_by(row, k.by_ho);
    const int iy = (int)(row - b * (uint32_t)g.ho) * g.sh, ix = (int)(p - row * (uint32_t)g.wo) * g.sw;
    const float* const xb = k.x + (int64_t)b * (g.h * g.w * g.cin);
    const int at = (iy * g.w + ix) * g.cin;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const bool in = (unsigned)(iy + tap_y[s]) < (unsigned)g.h && (unsigned)(ix + tap_x[s]) < (unsigned)g.w;
      const float v = xb[in ? at + tap_off[s] : 0];
      xv[s] = in ? v : 0.f;
    }
  };
  int p0 = p_begin + 16 * wave;
  float xv[KS], xn[KS];
  if (p0 < p_end) gather(p0, xv);
  for (; p0 < p_end; p0 += 64) {
    if (p0 + 64 < p_end) gather(p0 + 64, xn);
    f4v acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[s], wv[s][t], acc[t], 0, 0, 0);
    float v[4 * NT];  // [position 4 lq + i][filter]
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int t = 0; t < NT; ++t) v[i * NT + t] = acc[t][i];
    if (k.e.bias) {
#pragma unroll
      for (int i = 0; i < 4 * NT; ++i) v[i] = v[i] + bias[i % NT];
    }
    first_act<NT * 4>(k.e.act, v, k.e.act_param);
    const int mine = min(4, p_end - (p0 + 4 * lq));  // positions of this lane that exist (may be negative)
    float* const to = k.e.out + (int64_t)(p0 + 4 * lq) * k.e.ldo;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (i >= mine) continue;
      if constexpr (VEC) {
        typedef float vec __attribute__((ext_vector_type(NT)));
        vec o;
#pragma unroll
        for (int t = 0; t < NT; ++t) o[t] = v[i * NT + t];
        if (ch[0] < g.cout) *(vec*)(to + i * k.e.ldo + ch[0]) = o;
      } else {
#pragma unroll
        for (int t = 0; t < NT; ++t)
          if (ch[t] < g.cout) to[i * k.e.ldo + ch[t]] = v[i * NT + t];
      }
    }
    if constexpr (STATS) {
      if (p0 + 16 <= p_end) {
        float m[NT], q[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          m[t] = ((v[t] + v[NT + t]) + (v[2 * NT + t] + v[3 * NT + t])) * 0.25f;
          q[t] = 0.f;
#pragma unroll
          for (int i = 0; i < 4; ++i) { const float d = v[i * NT + t] - m[t]; q[t] = q[t] + d * d; }
        }
        join_moments<NT>(n, mean, m2, 4.0f, m, q);
        n += 4.0f;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (i >= mine) continue;
          float m[NT], q[NT];
#pragma unroll
          for (int t = 0; t < NT; ++t) { m[t] = v[i * NT + t]; q[t] = 0.f; }
          join_moments<NT>(n, mean, m2, 1.0f, m, q);
          n += 1.0f;
        }
      }
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) xv[s] = xn[s];
  }
  if constexpr (STATS) {
#pragma unroll
    for (int d = 16; d < 64; d <<= 1) {  // (both lanes of a pair join, in opposite order: the lowest ones' sums are kept)
      const float nb = __shfl_xor(n, d);
      float mb[NT], qb[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) { mb[t] = __shfl_xor(mean[t], d); qb[t] = __shfl_xor(m2[t], d); }
      join_moments<NT>(n, mean, m2, nb, mb, qb);
      n += nb;
    }
    if (lq == 0) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        moments[wave][0][ch[t] - co0] = mean[t];
        moments[wave][1][ch[t] - co0] = m2[t];
      }
      if (lane == 0) counts[wave] = n;
    }
    __syncthreads();
    const int c = threadIdx.x;
    if (c < 16 * NT && co0 + c < g.cout) {
      float na = counts[0], ma[1] = {moments[0][0][c]}, qa[1] = {moments[0][1][c]};
#pragma unroll
      for (int w = 1; w < 4; ++w) {
        const float mb[1] = {moments[w][0][c]}, qb[1] = {moments[w][1][c]};
        join_moments<1>(na, ma, qa, counts[w], mb, qb);
        na += counts[w];
      }
      k.part_mean[(int64_t)block * g.cout + co0 + c] = ma[0];
      k.part_m2[(int64_t)block * g.cout + co0 + c] = qa[0];
    }
  }
}

template <int KS, int NT>
void launch_first_fwd_tiles(sn_ctx* ctx, const FirstForward& k, int blocks, bool stats) {
  const dim3 grid((unsigned)blocks, (unsigned)ceil_div(k.g.cout, 16 * NT));
  if (stats) hipLaunchKernelGGL((conv_first_fwd_kernel<KS, NT, true>), grid, dim3(256), 0, ctx->stream, k);
  else hipLaunchKernelGGL((conv_first_fwd_kernel<KS, NT, false>), grid, dim3(256), 0, ctx->stream, k);
}
template <int KS>
void launch_first_fwd_steps(sn_ctx* ctx, const FirstForward& k, int blocks, bool stats) {
  switch (conv_first_fwd_tiles(k.taps, k.g.cout, stats)) {
    case 1: return launch_first_fwd_tiles<KS, 1>(ctx, k, blocks, stats);
    case 2: return launch_first_fwd_tiles<KS, 2>(ctx, k, blocks, stats);
    case 3: return launch_first_fwd_tiles<KS, 3>(ctx, k, blocks, stats);
    default: return launch_first_fwd_tiles<KS, 4>(ctx, k, blocks, stats);
  }
}

}  // namespace

int launch_conv_first_fwd(sn_ctx* ctx, const ConvGeom& g, const float* x, const float* w, const Epilogue& e, ConvStats* stats) {
  SN_REQUIRE(conv_first_fwd_ok(g, e), "conv2d_forward_first: shape outside the kernel's range");
  FirstForward k{};
  k.g = g;
  k.x = x;
  k.w = w;
  k.e = e;
  k.taps = g.kh * g.kw * g.cin;
  k.positions = g.n * g.ho * g.wo;
  k.by_wo = fast_div((uint32_t)g.wo);
  k.by_ho = fast_div((uint32_t)g.ho);
  k.by_cin = fast_div((uint32_t)g.cin);
  k.by_kw = fast_div((uint32_t)g.kw);
  const int64_t tiles = ceil_div(k.positions, 16);
  // a wavefront pays for its weights and tap offsets once: at least two tiles each where that leaves a workgroup for every CU
  int64_t blocks = std::min<int64_t>(std::max<int64_t>(ceil_div(tiles, 8), std::min<int64_t>(ceil_div(tiles, 4), ctx->compute_units)), (int64_t)ctx->compute_units * 4);
  const bool with_stats = stats && stats->max_slices > 0;
  if (with_stats) {
    blocks = std::min<int64_t>(blocks, stats->max_slices);
    k.part_mean = stats->part_mean;
    k.part_m2 = stats->part_m2;
  }
  k.tiles_per_block = (int)ceil_div(tiles, blocks);
  blocks = ceil_div(tiles, (int64_t)k.tiles_per_block);
  if (with_stats) {
    stats->slices = (int)blocks;
    stats->whole = (float)(k.tiles_per_block * 16);
    stats->last = (float)(k.positions - (blocks - 1) * k.tiles_per_block * 16);
  }
  LaunchScope scope(ctx, "conv2d_forward_direct", k.positions, g.cout, k.taps);
  const int steps = (int)ceil_div(k.taps, 4);
  if (steps <= 3) launch_first_fwd_steps<3>(ctx, k, (int)blocks, with_stats);
  else if (steps <= 5) launch_first_fwd_steps<5>(ctx, k, (int)blocks, with_stats);
  else if (steps <= 7) launch_first_fwd_steps<7>(ctx, k, (int)blocks, with_stats);
  else if (steps <= 9) launch_first_fwd_steps<9>(ctx, k, (int)blocks, with_stats);
  else if (steps <= 12) launch_first_fwd_steps<12>(ctx, k, (int)blocks, with_stats);
  else launch_first_fwd_steps<16>(ctx, k, (int)blocks, with_stats);
  SN_HIP(hipGetLastError());
  return SN_OK;
}

}  // namespace sn
