// First-layer Conv2D (one to four input channels): filter gradient on the float32 matrix instruction.
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
// 9 x 32 over 1000 x 26 x 26 under a batch normalisation and a pooling 88 -> 36.5 us (it reads 114 MB); 9 x 32 over 100 x 26 x 26
// under a pooling of stride 1, 11.6 -> 9.7 us.
#include "common.hpp"

#include <algorithm>

namespace sn {
namespace {

typedef float f4v __attribute__((ext_vector_type(4)));

struct FirstWgrad {
  ConvGeom g;
  const float* x;
  const float* dy;      // [n, ho, wo, cout], POOL: not read
  float* partial;       // [block][M][cout]
  int M, rows, rows_per_wave;  // taps; n * ho
  FastDiv by_ho, by_cin, by_kw, by_cout;
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

  // every XCD (workgroup id modulo 8) takes a contiguous run of rows
  const int per_xcd = ((int)gridDim.x + 7) >> 3, extra = (int)gridDim.x - (per_xcd - 1) * 8;  // `extra` XCDs have per_xcd workgroups, the others one less
  const int xcd = (int)blockIdx.x & 7;
  const int block = xcd * (per_xcd - 1) + min(xcd, extra) + ((int)blockIdx.x >> 3);
  const int row0 = (block * 4 + wave) * k.rows_per_wave, row1 = min(k.rows, row0 + k.rows_per_wave);
  const PoolGrad& pg = k.pool;
  for (int row = row0; row < row1; ++row) {
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
    for (int ow0 = 0; ow0 < g.wo; ow0 += 4 * G) {
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
        if (ow0 + 4 * u >= g.wo) break;
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
int conv_first_wgrad_parts(const sn_ctx* ctx, const ConvGeom& g, const float* ws, int64_t ws_elems, int* rows_per_wave) {
  const int M = g.kh * g.kw * g.cin, N = g.cout;
  const int64_t rows = (int64_t)g.n * g.ho;
  if (!ws || g.cin > 4 || M > FIRST_MAX_TAPS || N > FIRST_MAX_FILTERS || rows * g.wo < FIRST_MIN_POSITIONS) return 0;
  if (rows >= (1ll << 30) || (int64_t)g.h * g.w * g.cin >= (1ll << 30) || (int64_t)(g.wo + 1) * 2 * N >= (1ll << 30)) return 0;  // 32-bit offsets inside an image and two rows
  const int64_t room = std::min<int64_t>((int64_t)4 * ctx->compute_units, ws_elems / ((int64_t)M * N));
  if (room < 32) return 0;
  const int per = (int)ceil_div(rows, 4 * room);  // as many wavefronts as there are rows, up to four on a SIMD
  if (rows_per_wave) *rows_per_wave = per;
  return (int)ceil_div(rows, (int64_t)4 * per);
}

int launch_conv_first_wgrad(sn_ctx* ctx, const ConvGeom& g, const float* x, const float* dy, float* ws, int64_t ws_elems, const PoolGrad* pool, int* parts) {
  FirstWgrad k{};
  *parts = conv_first_wgrad_parts(ctx, g, ws, ws_elems, &k.rows_per_wave);
  SN_REQUIRE(*parts > 0, "conv2d_filter_gradient_first: shape outside the kernel's range");
  k.g = g;
  k.x = x;
  k.dy = dy;
  k.partial = ws;
  k.M = g.kh * g.kw * g.cin;
  k.rows = g.n * g.ho;
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

}  // namespace sn
