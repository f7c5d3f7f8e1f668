// A recurrent layer's products that do not depend on the recurrence, each over all time steps at once, on the split kernels
// (split_gemm.hpp): the inputs' share of the pre-activations and the gradient of the inputs.
#include "split_launch.hpp"

namespace sn {
namespace {

// rows of fewer than four values (FlatOp loads four of a row)
struct ShortRowsOp {
  static constexpr bool KC = true, MASKED = true, SIGNED = false;
  const float* p;
  int ld, outer_n, K;
  struct Outer {
    uint32_t off;
  };
  typedef KIndex KState;
  __device__ __forceinline__ int row(int outer) const { return outer; }
  __device__ __forceinline__ void init_outer(Outer& o, int outer) const { o.off = (uint32_t)min(outer, outer_n - 1) * (uint32_t)ld; }
  __device__ __forceinline__ void init_k(KState& s, int k) const { s.k = k; }
  __device__ __forceinline__ void advance(KState& s, int dk) const { s.k += dk; }
  __device__ __forceinline__ uint32_t load(const Outer& o, const KState& s, bool, f4v& v) const {
    uint32_t code = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool in = s.k + i < K;
      v[i] = p[o.off + (in ? (uint32_t)(s.k + i) : 0u)];
      code |= in ? 1u << i : 0u;
    }
    return code;
  }
};

// The gates' weights side by side: tensor q starts at[q] floats behind the first one's
struct GateTensors {
  const float* first;
  int at[4];
  int H;
  FastDiv by_h;
  __device__ __forceinline__ int start(int q) const { return q == 0 ? at[0] : q == 1 ? at[1] : q == 2 ? at[2] : at[3]; }
};

// value(k, n = gate H + u) = Wk_gate[k, u].  WHOLE: H is a multiple of four, a group of four columns has one gate
template <bool WHOLE>
struct GateColumnsOp {
  static constexpr bool KC = false, MASKED = !WHOLE, SIGNED = false;
  GateTensors w;
  int N, K;
  struct Outer {
    int off[WHOLE ? 1 : 4];
    uint32_t code;
  };
  typedef KIndex KState;
  __device__ __forceinline__ int row(int outer) const { return outer; }
  __device__ __forceinline__ void init_outer(Outer& o, int outer) const {
    o.code = 0;
#pragma unroll
    for (int i = 0; i < (WHOLE ? 1 : 4); ++i) {
      const int n = min(outer + i, N - (WHOLE ? 4 : 1)), q = (int)div_by((uint32_t)n, w.by_h);
      o.off[i] = w.start(q) + n - q * w.H;
      o.code |= outer + i < N ? 1u << i : 0u;
    }
  }
  __device__ __forceinline__ void init_k(KState& s, int k) const { s.k = k; }
  __device__ __forceinline__ void advance(KState& s, int dk) const { s.k += dk; }
  __device__ __forceinline__ uint32_t load(const Outer& o, const KState& s, bool tail, f4v& v) const {
    const bool in = !tail || s.k < K;
    const int row = (in ? s.k : 0) * w.H;
    if (WHOLE) {
      v = *(const f4u*)(w.first + o.off[0] + row);
      return in ? 15u : 0u;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = w.first[o.off[i % (WHOLE ? 1 : 4)] + row];
    return in ? o.code : 0u;
  }
};

// value(n = feature, k = gate H + u) = Wk_gate[n, u]
template <bool WHOLE>
struct GateRowsOp {
  static constexpr bool KC = true, MASKED = !WHOLE, SIGNED = false;
  GateTensors w;
  int N, K;
  struct Outer {
    int off;
  };
  typedef KIndex KState;
  __device__ __forceinline__ int row(int outer) const { return outer; }
  __device__ __forceinline__ void init_outer(Outer& o, int outer) const { o.off = min(outer, N - 1) * w.H; }
  __device__ __forceinline__ void init_k(KState& s, int k) const { s.k = k; }
  __device__ __forceinline__ void advance(KState& s, int dk) const { s.k += dk; }
  __device__ __forceinline__ int place(int k) const {
    const int q = (int)div_by((uint32_t)k, w.by_h);
    return w.start(q) + k - q * w.H;
  }
  __device__ __forceinline__ uint32_t load(const Outer& o, const KState& s, bool, f4v& v) const {
    if (WHOLE) {
      const bool in = s.k < K;
      v = *(const f4u*)(w.first + o.off + place(in ? s.k : 0));
      return in ? 15u : 0u;
    }
    uint32_t code = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool in = s.k + i < K;
      v[i] = w.first[o.off + place(in ? s.k + i : 0)];
      code |= in ? 1u << i : 0u;
    }
    return code;
  }
};

// row m = (b, t) of the product goes to row b of slice t
struct SlicesEpilogue {
  float* out;
  const float* bias[4];
  int64_t step;
  int T, H, N;
  FastDiv by_t, by_h;
  __device__ __forceinline__ int map_row(int m) const { return m; }
  __device__ __forceinline__ void store(int m, int n, float acc) const {
    const int b = (int)div_by((uint32_t)m, by_t), q = (int)div_by((uint32_t)n, by_h);
    const float* bq = q == 0 ? bias[0] : q == 1 ? bias[1] : q == 2 ? bias[2] : bias[3];
    out[(int64_t)(m - b * T) * step + (int64_t)b * N + n] = bq ? acc + bq[n - q * H] : acc;
  }
};

// (one division for the column and one for every four rows of a lane's values, not two for each value: 57 -> 45 us at 32000 x
// 512 x 32)
__device__ __forceinline__ void store16(const SlicesEpilogue& ep, int row0, int n, const f16v& acc, int M, int first = 0, int last = 16) {
  const int q = (int)div_by((uint32_t)n, ep.by_h);
  const float* bq = q == 0 ? ep.bias[0] : q == 1 ? ep.bias[1] : q == 2 ? ep.bias[2] : ep.bias[3];
  const float bias = bq ? bq[n - q * ep.H] : 0.f;
#pragma unroll
  for (int v4 = 0; v4 < 16; v4 += 4) {
    const int m = row0 + 2 * v4;
    int b = (int)div_by((uint32_t)m, ep.by_t), t = m - b * ep.T;
    float* to = ep.out + (int64_t)t * ep.step + (int64_t)b * ep.N + n;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      if (m + v < M && v4 + v >= first && v4 + v < last) *to = bq ? acc[v4 + v] + bias : acc[v4 + v];
      to += ep.step;
      if (++t == ep.T) {
        t = 0;
        to += ep.N - (int64_t)ep.T * ep.step;
      }
    }
  }
}

// row m = (t, b) of the product goes to step t of sample b
struct SamplesEpilogue {
  float* dx;
  int T, F, rows;
  FastDiv by_rows;
  __device__ __forceinline__ int map_row(int m) const { return m; }
  __device__ __forceinline__ void store(int m, int n, float acc) const {
    const int t = (int)div_by((uint32_t)m, by_rows), b = m - t * rows;
    dx[((int64_t)b * T + t) * F + n] = acc;
  }
};

// Tens of thousands of rows by a few hundred columns, K of a few dozen to a few hundred: many tiles, no use for a split K
template <class AL, class BL, class EP>
int launch_product(sn_ctx* ctx, const char* name, int M, int N, int K, const AL& al, const BL& bl, const EP& ep) {
  SplitGrid g{};
  g.M = M; g.N = N; g.K = K;
  g.ws_rows = M;
  g.colsum_row = -1;
  LaunchScope scope(ctx, name, M, N, K);
  return launch_split_tile<64, 64, 32, 2, 1, 2, 3>(ctx, g, 1, al, bl, ep);
}

template <class BL, class EP>
int launch_rows(sn_ctx* ctx, const char* name, const float* a, int M, int N, int K, const BL& bl, const EP& ep) {
  if (K >= 4) return launch_product(ctx, name, M, N, K, FlatOp<true>{a, K, M, K}, bl, ep);
  return launch_product(ctx, name, M, N, K, ShortRowsOp{a, K, M, K}, bl, ep);
}

bool gate_tensors(const LstmWeights& w, int gates, int F, int H, GateTensors* out) {
  out->first = w.wk[0];
  out->H = H;
  out->by_h = fast_div((uint32_t)H);
  for (int q = 0; q < 4; ++q) {
    const int64_t d = q < gates ? w.wk[q] - w.wk[0] : 0;
    if (d < 0 || d + (int64_t)F * H >= ((int64_t)1 << 31)) return false;
    out->at[q] = (int)d;
  }
  return true;
}

}  // namespace

// 32-bit byte offsets into x and dz, 32-bit places in the layer's weights
bool recurrent_products_fit(int rows, int T, int F, int H, int gates) {
  return (int64_t)rows * T * std::max<int64_t>(F, (int64_t)gates * H) * 4 < SPLIT_SPAN && (int64_t)gates * H * ((int64_t)F + H + 64) < SPLIT_SPAN / 2;
}

// out, slice t: row b, column gate H + u = x[b, t, :] Wk_gate[:, u] + b_gate[u]
int launch_recurrent_inputs(sn_ctx* ctx, const float* x, int rows, int T, int F, int H, const LstmWeights& w, int gates, float* out, int64_t step) {
  GateTensors g;
  SN_REQUIRE(recurrent_products_fit(rows, T, F, H, gates) && gate_tensors(w, gates, F, H, &g), "recurrent_inputs: operands out of range");
  const int N = gates * H;
  const SlicesEpilogue ep{out, {w.b[0], w.b[1], w.b[2], w.b[3]}, step, T, H, N, fast_div((uint32_t)T), fast_div((uint32_t)H)};
  if (H % 4 == 0) return launch_rows(ctx, "recurrent_inputs", x, rows * T, N, F, GateColumnsOp<true>{g, N, F}, ep);
  return launch_rows(ctx, "recurrent_inputs", x, rows * T, N, F, GateColumnsOp<false>{g, N, F}, ep);
}

// dx[b, t, f] = sum over gates and units of dz (slice t, row b, gate H + u) Wk_gate[f, u]
int launch_recurrent_dx(sn_ctx* ctx, const float* dz, int rows, int T, int F, int H, const LstmWeights& w, int gates, float* dx) {
  GateTensors g;
  SN_REQUIRE(recurrent_products_fit(rows, T, F, H, gates) && gate_tensors(w, gates, F, H, &g), "recurrent_input_gradient: operands out of range");
  const SamplesEpilogue ep{dx, T, F, rows, fast_div((uint32_t)rows)};
  const int K = gates * H;
  if (H % 4 == 0) return launch_rows(ctx, "recurrent_input_gradient", dz, rows * T, F, K, GateRowsOp<true>{g, F, K}, ep);
  return launch_rows(ctx, "recurrent_input_gradient", dz, rows * T, F, K, GateRowsOp<false>{g, F, K}, ep);
}

}  // namespace sn
