// The tiled matrix-core product behind most float32 Dense, Conv2D and recurrent input products (gemm_kernels.hip says what runs
// elsewhere) and, with one plane, the bf16 Dense products whose shapes gemm_bf16.hip does not take.
//
//   C[M, N] = A[M, K] * B[K, N], float32 in, float32 accumulate, float32 out
//
// gfx950 multiplies float32 on its matrix cores at 1/16 of the bf16 rate (64 against 1024 flop per clock and SIMD).  So
// every float32 value is taken apart into three bf16 values on its way into LDS, hi + mid + lo, each the round-to-nearest
// bf16 of what the ones before left over: 3 x 8 significand bits hold all 24 of a float32, the sum is EXACT from 2^-110 on
// (below that the lo part runs out of exponents).  A product is
//   a b = ah bh + (ah bm + am bh) + (ah bl + am bm + al bh) + (am bl + al bm + al bl)
// and the kernel multiplies the first six of these (bf16 x bf16 is exact in float32, the accumulator is float32); what is
// left out is below 2^-24 of |a b| (|am| <= 2^-8 |a|, |al| <= 2^-16 |a|, both halves of that on average), less than the
// rounding of ONE float32 addition.  Six v_mfma_f32_32x32x16_bf16 do the work of eight v_mfma_f32_32x32x2_f32 in 192
// matrix-core cycles instead of 512, and K values meet the accumulator in 6 K / 16 roundings instead of K / 2.
// Measured against float64 (N(0,1) operands, shapes from 5 x 4 x 4 to 32 x 32 x 16384): largest error 0.5-1.7e-7 of sum |a b|
// and root mean square error 0.53-0.88 of what float32 multiply-adds in k order show.  Rate: 8192 x 4096 x 4096 in 1.49 ms
// = 184 TFLOP/s (the float32 matrix peak is 157; the v_mfma_f32_32x32x2_f32 kernel this replaces ran such shapes at 60-80);
// 700 x 770 x 1003 with unaligned rows 59 -> 23 us, 1000 x 1500 x 1000 72 -> 32 us.
//
// The ends of the range.  An Inf taken apart is Inf + NaN + NaN, a finite value within 0.4 % of the largest float32 rounds to
// Inf as bf16, and where a product overflows its part products may do so with either sign.  Every thread keeps the largest
// magnitude it has taken apart (half an instruction per value; NaNs do not count: their parts are NaN), and a workgroup whose
// two largest could make a sum leave the range multiplies its tile once more with v_mfma_f32_32x32x2_f32, on float32 values.
// A value below 2^-110 loses up to 2^-134 in its lo part (a bf16 denormal; the matrix cores keep those), and a sum of k
// products up to k 2^-134 (A + B), A and B being the two largest magnitudes: less than a rounding of every sum of at least
// k 2^-110 (A + B).  Every thread keeps the smallest magnitude that is not zero, too (one and a half instructions per value),
// and a workgroup that has met one below 2^-110 and holds a smaller sum than that takes the same way.
//
// Workgroup = WVM x WVN x WVK wavefronts; block tile BM x BN, K stage BK.  Global loads go to registers (one stage ahead), are
// split there and stored to LDS as PLANES bf16 tiles [BK / 32][row][32 k] of 64 bytes per row, from where a fragment (8
// consecutive k of one row) is one 16-byte read.  The wavefronts divide the tile WVM x WVN ways and every stage's k-values
// WVK ways; the WVK partial sums of a tile meet in LDS at the end, each wavefront finishing its share of the values.
// Dividing K inside the workgroup is what makes a product with few tiles fast: a wavefront alone on its SIMD issues a vector
// instruction every 8 cycles, two to four share the issue slots, and no partial sums go through memory.
#pragma once

#include "common.hpp"

#include <type_traits>

namespace sn {

typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));  // 16-byte load from a 4-byte aligned address
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));

// ============================================================================ operands
// An operand loader describes A as a function of (outer = row m, k), B of (outer = column n, k) and fetches four values
// along its contiguous index: k when KC, the outer index otherwise.  Its state is split by what it depends on:
//   Outer   of a thread's row (KC) or group of four columns: fixed for the whole kernel
//   KState  of a thread's k: walks on by one stage (dk) at a time
//   load(o, k, tail, v) -> code   bits 0-3: element i is valid; bits 4-5: element i sits i + shift places on in v
//           (a vector that would run over the end of its row or tensor is loaded further in front)
//   MASKED  the code has to be looked at in every stage, not only in the last one (tail)
//   SIGNED  bits 4-6 hold the shift + 4 (-3 .. 3: a vector may also be loaded further behind)
//   row(outer)  KC = false: first of the four outer indices the thread really loads (the last group of a ragged row is
//           moved in front; its overlap with its neighbour carries the same values)
struct KIndex {
  int k;
};
// Walking a k that is kept as (row r, place j of Lp): what 32 values are in rows and places is worked out on the host (a loop of
// carries took up to a quarter as many trips as a stage has values: filter gradient of 72 x 48 x 31232, rows of 8 positions, 40 us).
struct RunWalk {
  int rows, places;  // 32 = rows * Lp + places
};
inline RunWalk run_walk(int Lp) { return RunWalk{32 / Lp, 32 % Lp}; }
__device__ __forceinline__ void walk_run(int& r, int& j, int dk, int Lp, const RunWalk& w) {
#pragma unroll
  for (int i = 0; i < dk / 32; ++i) {
    r += w.rows;
    j += w.places;
    const bool carry = j >= Lp;
    r += carry ? 1 : 0;
    j -= carry ? Lp : 0;
  }
}

template <bool KC_>
struct FlatOp {  // value(outer, k) = p[outer * ld + k] (KC) or p[k * ld + outer]
  static constexpr bool KC = KC_, MASKED = false, SIGNED = false;
  const float* p;
  int ld, outer_n, K;
  struct Outer {
    uint32_t off;
  };
  typedef KIndex KState;
  __device__ __forceinline__ int row(int outer) const { return KC ? outer : min(outer, outer_n - 4); }
  __device__ __forceinline__ void init_outer(Outer& o, int outer) const {
    o.off = KC ? (uint32_t)min(outer, outer_n - 1) * (uint32_t)ld * 4u : (uint32_t)row(outer) * 4u;
  }
  __device__ __forceinline__ void init_k(KState& s, int k) const { s.k = k; }
  __device__ __forceinline__ void advance(KState& s, int dk) const { s.k += dk; }
  __device__ __forceinline__ uint32_t load(const Outer& o, const KState& s, bool tail, f4v& v) const {
    int k = s.k;
    uint32_t code = 15u;
    if (tail) {
      if (KC) {
        const int kc = min(k, K - 4), sh = k - kc;
        code = sh > 3 ? 0u : ((15u >> sh) | ((uint32_t)sh << 4));
        k = kc;
      } else if (k >= K) {
        k = K - 1;
        code = 0u;
      }
    }
    v = *(const f4u*)((const char*)p + (o.off + (uint32_t)k * (KC ? 4u : (uint32_t)ld * 4u)));
    return code;
  }
  static bool ok(const float* p, int64_t s_outer, int64_t s_k, int outer_n, int K) {
    const int64_t ld = KC ? s_outer : s_k;
    return p && (KC ? s_k : s_outer) == 1 && ld >= 0 && (KC ? K : outer_n) >= 4 && (int64_t)(KC ? outer_n : K) * ld * 4 < SPLIT_SPAN &&
           (int64_t)(KC ? outer_n : K) * ld < SPLIT_SPAN && (reinterpret_cast<uintptr_t>(p) & 3u) == 0;
  }
};

// Conv2D sees a filter row as one run: for a fixed tap row r the kw taps' channels of a position are kw * C consecutive
// floats of an NHWC image, whatever C is.  The reduction index of the product is therefore k' = r * Lp + j, j < L = kw * C,
// with runs padded to Lp = a multiple of 4 (the other operand reads zeros there), so that a vector of four never leaves
// its run; which j lie inside the image is an interval per position.
//
// Rows m = positions (b, iy, ix) of the iteration space, src[b, iy*sy + oy + r*ty, ix*sx + ox + (j / C), j % C]:
//   forward: src = x, ty = +1, (oy, ox) = -padding;
//   input gradient (unit strides): src = dy, ty = -1, oy = +pt, ox = pl - (kw - 1): the taps of a row in reverse order.
template <bool MASKED_>
struct ConvRunOp {
  static constexpr bool KC = true, MASKED = MASKED_, SIGNED = MASKED_;  // not masked: no padding, and L is a multiple of 4
  const float* src;
  int M, ih, iw, sy, sx, oy, ox, ty;
  int H, W, C, kh, L, Lp;
  int total;  // elements of src
  FastDiv by_iw, by_ih;
  RunWalk walk;
  struct Outer {
    int base, y0;   // element offset of (b, y0, x0, 0), possibly outside the tensor
    int jlo, jhi;   // j inside the image's width
  };
  struct KState {
    int r, j;
  };
  __device__ __forceinline__ int row(int outer) const { return outer; }
  __device__ __forceinline__ void init_outer(Outer& o, int m) const {
    const uint32_t mm = (uint32_t)min(m, M - 1);
    const uint32_t t = div_by(mm, by_iw), b = div_by(t, by_ih);
    const int ix = (int)(mm - t * (uint32_t)iw), iy = (int)(t - b * (uint32_t)ih);
    const int x0 = ix * sx + ox;
    o.y0 = iy * sy + oy;
    o.base = (((int)b * H + o.y0) * W + x0) * C;
    o.jlo = x0 < 0 ? -x0 * C : 0;
    o.jhi = min(L, (W - x0) * C);
  }
  __device__ __forceinline__ void init_k(KState& s, int k) const {
    s.r = k / Lp;
    s.j = k - s.r * Lp;
  }
  __device__ __forceinline__ void advance(KState& s, int dk) const {
    walk_run(s.r, s.j, dk, Lp, walk);
  }
  __device__ __forceinline__ uint32_t load(const Outer& o, const KState& s, bool tail, f4v& v) const {
    int off = o.base + s.r * (ty * W * C) + s.j;
    uint32_t code = 15u;
    if (MASKED) {
      const bool in_rows = s.r < kh && (unsigned)(o.y0 + s.r * ty) < (unsigned)H;
      const int lo = max(o.jlo - s.j, 0), hi = min(o.jhi - s.j, 4);  // valid elements [lo, hi)
      code = in_rows && hi > lo ? (15u >> (4 - hi)) & (15u << lo) & 15u : 0u;
      if (code == 0u) off = 0;
      const int offc = min(max(off, 0), total - 4);
      // an element i sits at v[i + off - offc]: the difference is -3 .. 3, kept + 4 in bits 4-6
      code |= (uint32_t)(off - offc + 4) << 4;
      off = offc;
    } else if (tail && s.r >= kh) {
      code = 0u;
      off = 0;
    }
    v = *(const f4u*)(src + off);
    return code;
  }
};

// The forward filter as the B operand: w[K][N] read by k' (row r * L + j of the tensor, zeros for the padding of a run).
struct ConvRunFilterOp {
  static constexpr bool KC = false, MASKED = true, SIGNED = false;
  const float* w;
  int N, kh, L, Lp;
  RunWalk walk;
  struct Outer {
    int off;
  };
  struct KState {
    int r, j;
  };
  __device__ __forceinline__ int row(int outer) const { return min(outer, N - 4); }
  __device__ __forceinline__ void init_outer(Outer& o, int n) const { o.off = row(n); }
  __device__ __forceinline__ void init_k(KState& s, int k) const {
    s.r = k / Lp;
    s.j = k - s.r * Lp;
  }
  __device__ __forceinline__ void advance(KState& s, int dk) const {
    walk_run(s.r, s.j, dk, Lp, walk);
  }
  __device__ __forceinline__ uint32_t load(const Outer& o, const KState& s, bool, f4v& v) const {
    const bool in = s.r < kh && s.j < L;
    v = *(const f4u*)(w + (in ? (s.r * L + s.j) * N + o.off : o.off));
    return in ? 15u : 0u;
  }
};

// The input gradient's B operand: column n = input channel, k' = r * Lp + j with j = q' * cout + co, q' = kw - 1 - q:
// w[((r * kw + q) * cin + n) * cout + co].  A group of four j may cross from one tap to the next unless cout % 4 == 0.
template <bool WHOLE>
struct ConvDgradFilterOp {
  static constexpr bool KC = true, MASKED = !WHOLE, SIGNED = false;
  const float* w;
  int cin, cout, kh, kw, L, Lp;
  FastDiv by_cout;
  RunWalk walk;
  struct Outer {
    int off;
  };
  struct KState {
    int r, j;
  };
  __device__ __forceinline__ int row(int outer) const { return outer; }
  __device__ __forceinline__ void init_outer(Outer& o, int n) const { o.off = min(n, cin - 1) * cout; }
  __device__ __forceinline__ void init_k(KState& s, int k) const {
    s.r = k / Lp;
    s.j = k - s.r * Lp;
  }
  __device__ __forceinline__ void advance(KState& s, int dk) const {
    walk_run(s.r, s.j, dk, Lp, walk);
  }
  __device__ __forceinline__ int place(int r, int j) const {
    const int qq = (int)div_by((uint32_t)j, by_cout);
    return (r * kw + (kw - 1 - qq)) * cin * cout + (j - qq * cout);
  }
  __device__ __forceinline__ uint32_t load(const Outer& o, const KState& s, bool tail, f4v& v) const {
    if (WHOLE) {
      const bool in = !tail || s.r < kh;
      v = *(const f4u*)(w + o.off + (in ? place(s.r, s.j) : 0));
      return in ? 15u : 0u;
    }
    const bool in = s.r < kh;
    uint32_t code = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool ok = in && s.j + i < L;
      v[i] = w[o.off + (ok ? place(s.r, s.j + i) : 0)];
      code |= ok ? 1u << i : 0u;
    }
    return code;
  }
};

// The filter gradient's A operand: row m' = r * Lp + j (tap row r, j = q * C + ci), k = output position (b, oh, ow):
// x[b, oh*sh - pt + r, ow*sw - pl + j / C, j % C].
template <bool MASKED_>
struct ConvWgradRunOp {
  static constexpr bool KC = false, MASKED = MASKED_, SIGNED = MASKED_;  // not masked: no padding, and L is a multiple of 4
  const float* x;
  ConvGeom g;
  int L, Lp, K, total, rows;  // rows = kh * Lp
  FastDiv by_wo, by_ho;
  int step_ow, step_oh, step_b;  // 32 = (step_b * ho + step_oh) * wo + step_ow
  struct Outer {
    int off, r, j;
  };
  struct KState {
    int k, b, oh, ow;
  };
  __device__ __forceinline__ int row(int outer) const { return min(outer, rows - 4); }
  __device__ __forceinline__ void init_outer(Outer& o, int m) const {
    const int mm = row(m);
    o.r = mm / Lp;
    o.j = mm - o.r * Lp;
    o.off = o.r * g.w * g.cin + o.j;
  }
  __device__ __forceinline__ void init_k(KState& s, int k) const {
    s.k = k;
    const uint32_t t = div_by((uint32_t)k, by_wo), b = div_by(t, by_ho);
    s.ow = k - (int)t * g.wo;
    s.oh = (int)(t - b * (uint32_t)g.ho);
    s.b = (int)b;
  }
  __device__ __forceinline__ void advance(KState& s, int dk) const {
    s.k += dk;
#pragma unroll
    for (int i = 0; i < dk / 32; ++i) {
      s.ow += step_ow;
      const bool next_row = s.ow >= g.wo;
      s.ow -= next_row ? g.wo : 0;
      s.oh += step_oh + (next_row ? 1 : 0);
      const bool next_image = s.oh >= g.ho;  // (step_oh < ho: at most one)
      s.oh -= next_image ? g.ho : 0;
      s.b += step_b + (next_image ? 1 : 0);
    }
  }
  __device__ __forceinline__ uint32_t load(const Outer& o, const KState& s, bool tail, f4v& v) const {
    const int y0 = s.oh * g.sh - g.pt, x0 = s.ow * g.sw - g.pl;
    int off = ((s.b * g.h + y0) * g.w + x0) * g.cin + o.off;
    uint32_t code = 15u;
    if (MASKED) {
      const bool in = (!tail || s.k < K) && (unsigned)(y0 + o.r) < (unsigned)g.h;
      const int lo = max(-x0 * g.cin - o.j, 0), hi = min(min(L, (g.w - x0) * g.cin) - o.j, 4);
      code = in && hi > lo ? (15u >> (4 - hi)) & (15u << lo) & 15u : 0u;
      if (code == 0u) off = 0;
      const int offc = min(max(off, 0), total - 4);
      code |= (uint32_t)(off - offc + 4) << 4;
      off = offc;
    } else if (tail && s.k >= K) {
      code = 0u;
      off = 0;
    }
    v = *(const f4u*)(x + off);
    return code;
  }
};

// ============================================================================ epilogues
// store(m, n, acc) takes one element of the product; map_row(m) is the row it belongs to (-1: dropped), which differs from
// m only where the product's rows carry padding.
__device__ __forceinline__ float ep_act(int act, float v, float param) {
  switch (act) {
    case SN_ACT_SIGMOID: return 1.0f / (1.0f + expf(-v));
    case SN_ACT_TANH: return tanhf(v);
    case SN_ACT_RELU: return fmaxf(param, v);
    default: return v;
  }
}

// The same activation over N values with ONE dispatch on `act`: a switch per value costs a handful of scalar branches
// each, which in a 16-value accumulator tile is more instruction-fetch stalls than arithmetic.
template <int N>
__device__ __forceinline__ void ep_act_block(int act, float (&v)[N], float param) {
  switch (act) {
    case SN_ACT_SIGMOID:
#pragma unroll
      for (int k = 0; k < N; ++k) v[k] = 1.0f / (1.0f + expf(-v[k]));
      break;
    case SN_ACT_TANH:
#pragma unroll
      for (int k = 0; k < N; ++k) v[k] = tanhf(v[k]);
      break;
    case SN_ACT_RELU:
#pragma unroll
      for (int k = 0; k < N; ++k) v[k] = fmaxf(param, v[k]);
      break;
    default: break;
  }
}

struct StdEpilogue {
  Epilogue e;
  __device__ __forceinline__ int map_row(int m) const { return m; }
  __device__ __forceinline__ void store(int m, int n, float acc) const {
    if (m == e.row_index) {
      e.row_out[n] = acc;
      return;
    }
    float v = acc;
    if (e.bias) v = v + e.bias[n];
    e.out[(int64_t)m * e.ldo + n] = ep_act(e.act, v, e.act_param);
  }
};

// An input gradient dX on its way through the activation of the layer below, whose output y [rows, ldo] lies beside it: the
// arithmetic of act_bwd_kernel on the finished sum.
struct ActGradEpilogue {
  float* out;
  const float* y;
  int64_t ldo;
  int act;
  float act_param;
  __device__ __forceinline__ int map_row(int m) const { return m; }
  __device__ __forceinline__ void store(int m, int n, float acc) const {
    const int64_t at = (int64_t)m * ldo + n;
    float g = acc;
    switch (act) {
      case SN_ACT_SIGMOID: { const float s = y[at]; g = (s * (1.0f - s)) * acc; break; }
      case SN_ACT_TANH: { const float s = y[at]; g = (1.0f - s * s) * acc; break; }
      case SN_ACT_RELU: g = (act_param < y[at] ? 1.0f : 0.0f) * acc; break;
      default: break;
    }
    out[at] = g;
  }
};

// the filter gradient's rows m' = r * Lp + j: row r * L + j of the tensor, nothing for the padding
struct RunRowsEpilogue {
  float* out;
  int ldo, L, Lp;
  __device__ __forceinline__ int map_row(int m) const {
    const int r = m / Lp, j = m - r * Lp;
    return j < L ? r * L + j : -1;
  }
  __device__ __forceinline__ void store(int m, int n, float acc) const { out[(int64_t)m * ldo + n] = acc; }
};

// A lane's accumulator values first .. last - 1 of one 32x32 MFMA tile: value v is column n, row row0 + 8*(v/4) + v%4; rows >= M
// are dropped.
template <class EP>
__device__ __forceinline__ void store16(const EP& ep, int row0, int n, const f16v& acc, int M, int first = 0, int last = 16) {
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int row = row0 + (v >> 2) * 8 + (v & 3);
    if (row < M && v >= first && v < last) {
      const int to = ep.map_row(row);
      if (to >= 0) ep.store(to, n, acc[v]);
    }
  }
}
// The plain epilogue reads the column's bias once and dispatches on the activation once for the 16 values: inside an
// instantiation the activation is a compile-time constant, so the 16 stores carry no scalar branches.
template <int ACT>
__device__ __forceinline__ float ep_act_const(float v, float param) {
  if constexpr (ACT == SN_ACT_SIGMOID) return 1.0f / (1.0f + expf(-v));
  else if constexpr (ACT == SN_ACT_TANH) return tanhf(v);
  else if constexpr (ACT == SN_ACT_RELU) return fmaxf(param, v);
  else return v;
}

template <int ACT>
__device__ __forceinline__ void store16_act(const Epilogue& e, int row0, int n, const f16v& acc, int M, int first, int last) {
  const bool has_bias = e.bias != nullptr;
  const float b = has_bias ? e.bias[n] : 0.f;
  float* out = e.out + (int64_t)row0 * e.ldo + n;
  // One value at a time, each behind its own row check: a straight run of 16 stores lets the compiler compute all 16
  // addresses and read all 16 accumulators up front, which doubles the kernel's registers and costs the split-K launches
  // their occupancy (measured: filter gradient 31 -> 37 us).
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const int dr = (k >> 2) * 8 + (k & 3);
    if (row0 + dr >= M || k < first || k >= last) continue;
    if (row0 + dr == e.row_index) {
      e.row_out[n] = acc[k];
    } else {
      const float x = has_bias ? acc[k] + b : acc[k];
      out[(int64_t)dr * e.ldo] = ep_act_const<ACT>(x, e.act_param);
    }
  }
}

__device__ __forceinline__ void store16(const StdEpilogue& ep, int row0, int n, const f16v& acc, int M, int first = 0, int last = 16) {
  switch (ep.e.act) {
    case SN_ACT_SIGMOID: store16_act<SN_ACT_SIGMOID>(ep.e, row0, n, acc, M, first, last); break;
    case SN_ACT_TANH: store16_act<SN_ACT_TANH>(ep.e, row0, n, acc, M, first, last); break;
    case SN_ACT_RELU: store16_act<SN_ACT_RELU>(ep.e, row0, n, acc, M, first, last); break;
    default: store16_act<SN_ACT_IDENTITY>(ep.e, row0, n, acc, M, first, last); break;
  }
}

// All of a lane's values of y are requested before the first is used, and the activation is looked at once.
__device__ __forceinline__ void store16(const ActGradEpilogue& ep, int row0, int n, const f16v& acc, int M, int first = 0, int last = 16) {
  float y[16];
#pragma unroll
  for (int v = 0; v < 16; ++v)
    if (v >= first && v < last) y[v] = ep.y[(int64_t)min(row0 + (v >> 2) * 8 + (v & 3), M - 1) * ep.ldo + n];
  auto store = [&](auto grad) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int row = row0 + (v >> 2) * 8 + (v & 3);
      if (row < M && v >= first && v < last) ep.out[(int64_t)row * ep.ldo + n] = grad(y[v], acc[v]);
    }
  };
  switch (ep.act) {
    case SN_ACT_SIGMOID: store([](float s, float a) { return (s * (1.0f - s)) * a; }); break;
    case SN_ACT_TANH: store([](float s, float a) { return (1.0f - s * s) * a; }); break;
    case SN_ACT_RELU: store([&](float s, float a) { return (ep.act_param < s ? 1.0f : 0.0f) * a; }); break;
    default: store([](float, float a) { return a; }); break;
  }
}

// ============================================================================ the kernel
// two float32 values -> two bf16 values (round to nearest even) in one register
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  uint32_t r;
  asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// hi + mid + lo of a pair, PLANES of them
template <int PLANES>
__device__ __forceinline__ void split_pair(float a, float b, uint32_t (&p)[PLANES]) {
  p[0] = pack_bf16(a, b);
#pragma unroll
  for (int i = 1; i < PLANES; ++i) {
    a = a - __uint_as_float(p[i - 1] << 16);
    b = b - __uint_as_float(p[i - 1] & 0xffff0000u);
    p[i] = pack_bf16(a, b);
  }
}

// Up to these magnitudes of two operands, and k products a sum, no part of a value and no sum of part products leaves float32's
// range (an Inf taken apart is Inf + NaN + NaN, and part products that overflow do so with either sign).
constexpr float LARGEST_BF16 = 3.3895313892515355e38f, LARGEST_SUM = 0x1p126f;
// whatever the other operand and k <= 2^31 are, as long as it holds for both
constexpr float SURELY_IN_RANGE = 0x1p47f;
// sums of k products from k (A + B) times this on
constexpr float LOSSLESS_SUM = 0x1p-110f;
// |a| below 2^-110, but not zero (by its bits: twice the magnitude, minus one, so that a zero is the largest)
constexpr uint32_t LEAST_WHOLE = (17u << 24) - 1u;
__device__ __forceinline__ uint32_t magnitude_key(float a) { return (__float_as_uint(a) << 1) - 1u; }
__device__ __forceinline__ bool parts_in_range(float a, float b, int k) {
  return a <= LARGEST_BF16 && b <= LARGEST_BF16 && a * b * (float)k <= LARGEST_SUM;
}

// max(m, |a|, |b|), NaNs ignored
__device__ __forceinline__ float max_magnitude(float m, float a, float b) {
  float r;
  asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(m), "v"(a), "v"(b));
  return r;
}

// the vector as its code says: elements moved into place, the invalid ones zero
template <bool SIGNED_SHIFT>
__device__ __forceinline__ void apply_code(f4v& v, uint32_t code) {
  if constexpr (SIGNED_SHIFT) {
    const int sh = (int)(code >> 4) - 4;  // element i = v[i + sh]
    if (__any(sh != 0 && (code & 15u) != 0)) {
      f4v w = v;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float x = 0.f;
#pragma unroll
        for (int s = 0; s < 4; ++s) x = i + sh == s ? v[s] : x;
        w[i] = x;
      }
      v = w;
    }
  } else {
    const uint32_t sh = code >> 4;
    if (sh & 1u) v = f4v{v[1], v[2], v[3], v[3]};
    if (sh & 2u) v = f4v{v[2], v[3], v[3], v[3]};
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = (code >> i) & 1u ? v[i] : 0.f;
}

// Byte offset of the 16-byte chunk `chunk` (0-3, 8 k-values) of row `row` inside a 32-k plane of 64-byte rows.  Both the chunk
// and the row's place in its group of four are XOR-ed with the group's number: the 16-byte fragment reads of 16 neighbouring
// rows cover all 64 banks once (as do rows 0-3, 12-15, 20-23, 24-27), and the writes of every fourth row spread over them too.
__device__ __forceinline__ uint32_t plane_at(int row, int chunk) {
  return (uint32_t)(((row & ~3) | ((row ^ (row >> 2)) & 3)) * 64 + ((chunk ^ ((row >> 2) & 3)) << 4));
}

// One operand's share of a workgroup of T threads: which vectors a thread loads, and how they go to LDS.
template <class OP, int BT, int BK, int PLANES, int T>
struct Stager {
  // KC: thread -> (k-group of four, row), E rows RP apart.  Otherwise a thread takes KB consecutive k of four outer indices: the
  // transposition happens in registers, pairs of k are packed into the same word.  16 neighbouring threads read 64
  // consecutive outer indices of one k.
  static constexpr int KB = OP::KC ? 4 : (BT / 4 * (BK / 4) >= T ? 4 : 2);
  static constexpr int KG = BK / KB;                                   // k-groups
  static constexpr int OV = OP::KC ? BT : BT / 4;                      // rows, or groups of four outer indices
  static constexpr int OW = OV < 16 ? OV : 16;
  static constexpr int ACTIVE = OV * KG < T ? OV * KG : T;             // threads that take part
  static constexpr int RP = ACTIVE / KG;                               // KC: rows per pass
  static constexpr int E = OP::KC ? OV / RP : KB;                      // vectors per thread
  static constexpr int ROWS = BT + 4;                                  // (the moved last group of a ragged row may start up to 3 rows in front)
  static constexpr int SUB = ROWS * 64, PLANE = SUB * (BK / 32);
  static_assert(E >= 1 && (OP::KC ? RP % 16 == 0 && OV % RP == 0 : OV * KG == ACTIVE && OV % OW == 0), "tile does not suit the workgroup");
  typename OP::Outer o[OP::KC ? E : 1];
  typename OP::KState k[OP::KC ? 1 : E];
  f4v v[E];
  uint32_t code[E];
  uint32_t at[OP::KC ? 1 : 4];  // KC: byte offset of the thread's 8 bytes of its first row; else of its bytes of each row
  bool on;
  bool tail;
  f4v colsum = {0.f, 0.f, 0.f, 0.f};
  float largest = 0.f;           // magnitude of what this thread has taken apart
  uint32_t least = 0xffffffffu;  // magnitude_key of the same

  static __device__ __forceinline__ int kgroup(int tid) { return OP::KC ? tid % KG : (tid / OW) % KG; }
  static __device__ __forceinline__ int ogroup(int tid) { return OP::KC ? tid / KG : tid % OW + OW * (tid / (OW * KG)); }
  static __device__ __forceinline__ uint32_t place(int row, int k) {  // byte offset of element k of a stage
    return (uint32_t)((k >> 5) * SUB) + plane_at(row, (k >> 3) & 3) + (uint32_t)(k & 7) * 2u;
  }
  static __device__ __forceinline__ uint32_t f32_place(int row, int k) { return (uint32_t)((k * ROWS + row) * 4); }  // ... in float32
  static_assert(BK * ROWS * 4 <= 3 * PLANE, "a stage in float32 fits the three planes");
  template <bool F32>
  __device__ __forceinline__ void init(const OP& op, int tid, int outer0, int k_begin) {
    on = ACTIVE == T || tid < ACTIVE;
    const int kg = kgroup(tid), ov = on ? ogroup(tid) : 0;
    if constexpr (OP::KC) {
#pragma unroll
      for (int e = 0; e < E; ++e) op.init_outer(o[e], outer0 + ov + RP * e);
      op.init_k(k[0], k_begin + kg * 4);
      at[0] = F32 ? f32_place(ov + 4, kg * 4) : place(ov + 4, kg * 4);  // rows RP apart: the same swizzle
    } else {
      op.init_outer(o[0], outer0 + 4 * ov);
#pragma unroll
      for (int e = 0; e < E; ++e) op.init_k(k[e], k_begin + kg * KB + e);
      const int local = op.row(outer0 + 4 * ov) - outer0 + 4;  // >= 1
#pragma unroll
      for (int i = 0; i < 4; ++i) at[i] = F32 ? f32_place(local + i, kg * KB) : place(local + i, kg * KB);
    }
  }
  __device__ __forceinline__ void fetch(const OP& op, bool is_tail) {
    tail = is_tail;
    if (!on) return;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if constexpr (OP::KC) code[e] = op.load(o[e], k[0], is_tail, v[e]);
      else {
        code[e] = op.load(o[0], k[e], is_tail, v[e]);
        op.advance(k[e], BK);
      }
    }
    if constexpr (OP::KC) op.advance(k[0], BK);
  }
  // PL planes of the fetched vectors go to LDS.  sum (KC = false only): adds the thread's KB rows to its four column sums
  template <int PL>
  __device__ __forceinline__ void stage(char* lds, bool sum) {
    if (!on) return;
    if (OP::MASKED || tail) {
#pragma unroll
      for (int e = 0; e < E; ++e) apply_code<OP::SIGNED>(v[e], code[e]);
    }
    if constexpr (PL > 1) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        largest = max_magnitude(max_magnitude(largest, v[e][0], v[e][1]), v[e][2], v[e][3]);
        least = min(min(least, magnitude_key(v[e][0])), magnitude_key(v[e][1]));
        least = min(min(least, magnitude_key(v[e][2])), magnitude_key(v[e][3]));
      }
    }
    if constexpr (OP::KC) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        uint32_t a[PL], b[PL];
        split_pair<PL>(v[e][0], v[e][1], a);
        split_pair<PL>(v[e][2], v[e][3], b);
#pragma unroll
        for (int p = 0; p < PL; ++p) *(u2v*)(lds + p * PLANE + at[0] + e * RP * 64) = u2v{a[p], b[p]};
      }
    } else {
      if (sum) {
#pragma unroll
        for (int e = 0; e < E; ++e) colsum += v[e];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        uint32_t a[PL], b[PL];
        split_pair<PL>(v[0][i], v[1][i], a);
        if constexpr (KB == 4) {
          split_pair<PL>(v[2][i], v[3][i], b);
#pragma unroll
          for (int p = 0; p < PL; ++p) *(u2v*)(lds + p * PLANE + at[i]) = u2v{a[p], b[p]};
        } else {
#pragma unroll
          for (int p = 0; p < PL; ++p) *(uint32_t*)(lds + p * PLANE + at[i]) = a[p];
        }
      }
    }
  }
  // the fetched vectors go to LDS as they are
  __device__ __forceinline__ void stage_f32(char* lds) {
    if (!on) return;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if (OP::MASKED || tail) apply_code<OP::SIGNED>(v[e], code[e]);
#pragma unroll
      for (int i = 0; i < 4; ++i) *(float*)(lds + (OP::KC ? at[0] + i * ROWS * 4 + e * RP * 4 : at[i % (OP::KC ? 1 : 4)] + e * ROWS * 4)) = v[e][i];
    }
  }
};

struct SplitGrid {
  int M, N, K;         // M without the column-sum row
  int k_per_split, splits;
  int tiles_m, tiles_n;
  float* ws;           // partial products [split][rows][N] (rows counts the column-sum row), null: one split, the epilogue stores
  int ws_rows;
  int colsum_row;      // >= 0: output row that receives the column sums of B (a Dense layer's bias gradient)
};

// LDS of a workgroup: the operand planes, or the partial sums that the WVK wavefronts of a tile exchange at the end
template <int BM, int BN, int BK, int WVM, int WVN, int WVK, int PLANES, class AL, class BL>
struct SplitShape {
  static constexpr int T = 64 * WVM * WVN * WVK;
  typedef Stager<AL, BM, BK, PLANES, T> SA;
  typedef Stager<BL, BN, BK, PLANES, T> SB;
  static constexpr int TM = BM / WVM / 32, TN = BN / WVN / 32, VALUES = TM * TN * 16;  // accumulator values per lane
  static constexpr int KEEP = VALUES / WVK;                                            // of which a wavefront finishes these
  static constexpr int STAGE_BYTES = PLANES * (SA::PLANE + SB::PLANE);
  static constexpr int SWAP_BYTES = WVK > 1 ? BM * BN * 4 * (WVK - 1) : 0;
  static constexpr int SUM_BYTES = BL::KC ? 0 : SB::KG * BN * 4;                       // column sums of B
  static constexpr int LDS = STAGE_BYTES > SWAP_BYTES ? (STAGE_BYTES > SUM_BYTES ? STAGE_BYTES : SUM_BYTES)
                                                      : (SWAP_BYTES > SUM_BYTES ? SWAP_BYTES : SUM_BYTES);
  static_assert(BK % 32 == 0 && TM >= 1 && TN >= 1 && BK % (16 * WVK) == 0 && VALUES % WVK == 0 && KEEP % 4 == 0, "tile does not suit the wavefronts");
  static_assert(LDS <= 160 * 1024, "more LDS than a CU has");
};

template <int BM, int BN, int BK, int WVM, int WVN, int WVK, int PLANES, class AL, class BL, class EP>
__global__ __launch_bounds__(64 * WVM * WVN * WVK) void split_gemm_kernel(SplitGrid g, AL al, BL bl, EP ep) {
  typedef SplitShape<BM, BN, BK, WVM, WVN, WVK, PLANES, AL, BL> Shape;
  typedef typename Shape::SA SA;
  typedef typename Shape::SB SB;
  constexpr int TM = Shape::TM, TN = Shape::TN, KEEP = Shape::KEEP;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  char* const la = lds;
  char* const lb = lds + PLANES * SA::PLANE;

  // Consecutive workgroup ids land on different XCDs (8, each with its own L2).  Work items are numbered splits first, then
  // rows of tiles, then columns, and every XCD takes a contiguous run of them: what neighbouring tiles share (a K range, a
  // row of A) is fetched into few L2s.
  const int tiles = g.tiles_m * g.tiles_n, items = tiles * g.splits, per_xcd = (items + 7) >> 3;
  const int item = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_xcd || item >= items) return;
  const int bz = item / tiles, tile = item - bz * tiles;
  const int bm = tile / g.tiles_n, bn = tile - bm * g.tiles_n;
  const int m0 = bm * BM, n0 = bn * BN;
  const int k_begin = bz * g.k_per_split, k_end = min(g.K, k_begin + g.k_per_split);

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l32 = lane & 31, lhi = lane >> 5;
  const int wk = wave % WVK, wmn = wave / WVK;
  const int wm = (wmn / WVN) * (TM * 32), wn = (wmn % WVN) * (TN * 32);

  SA sa;
  SB sb;
  f16v acc[TM][TN];
  const bool sum_columns = !BL::KC && g.colsum_row >= 0 && bm == 0;

  // fragment addresses of this wavefront's 16-long parts of a stage: k = 16 part + 8 (lane / 32) of row (tile row + lane % 32)
  constexpr int PARTS = BK / 16 / WVK;
  uint32_t fa[PARTS], fb[PARTS];
#pragma unroll
  for (int h = 0; h < PARTS; ++h) {
    const int k = 16 * (wk * PARTS + h) + 8 * lhi;
    fa[h] = SA::place(wm + l32 + 4, k);
    fb[h] = SB::place(wn + l32 + 4, k);
  }

  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
  };
  // adds the wavefronts' shares of the stages' k-values: the sums are complete in every wavefront for the values it keeps
  auto exchange = [&]() {
    if constexpr (WVK > 1) {
      // value u (of TM x TN x 16) of a lane belongs to wavefront u / KEEP of its tile; the others hand theirs over:
      // [tile of the workgroup][keeper][sender other than the keeper][value of the keeper's share][lane]
      float* ex = reinterpret_cast<float*>(lds) + wmn * (WVK * (WVK - 1) * KEEP * 64) + lane;
#pragma unroll
      for (int u = 0; u < Shape::VALUES; ++u) {
        const int keeper = u / KEEP;
        if (keeper != wk) ex[((keeper * (WVK - 1) + (wk > keeper ? wk - 1 : wk)) * KEEP + u % KEEP) * 64] = acc[u / 16 / TN][u / 16 % TN][u % 16];
      }
      __syncthreads();
#pragma unroll
      for (int u = 0; u < Shape::VALUES; ++u) {
        if (u / KEEP != wk) continue;
        float s = acc[u / 16 / TN][u / 16 % TN][u % 16];
#pragma unroll
        for (int o = 0; o < WVK - 1; ++o) s += ex[((wk * (WVK - 1) + o) * KEEP + u % KEEP) * 64];
        acc[u / 16 / TN][u / 16 % TN][u % 16] = s;
      }
    }
  };

  sa.template init<false>(al, threadIdx.x, m0, k_begin);
  sb.template init<false>(bl, threadIdx.x, n0, k_begin);
  clear();
  // (Two, three and four stages of loads in flight instead of one were measured: no faster at any size, and the registers
  // cost a wavefront per SIMD.)
  sa.fetch(al, k_begin + BK > k_end);
  sb.fetch(bl, k_begin + BK > k_end);
  for (int k0 = k_begin; k0 < k_end; k0 += BK) {
    sa.template stage<PLANES>(la, false);
    sb.template stage<PLANES>(lb, sum_columns);
    __syncthreads();
    if (k0 + BK < k_end) {  // the next stage's global loads fly while this one is multiplied
      const bool tail = k0 + 2 * BK > k_end;
      sa.fetch(al, tail);
      sb.fetch(bl, tail);
    }
#pragma unroll
    for (int h = 0; h < PARTS; ++h) {
      bf16x8 af[TM][PLANES], bf[TN][PLANES];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int p = 0; p < PLANES; ++p) af[i][p] = *(const bf16x8*)(la + p * SA::PLANE + fa[h] + i * 2048);
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int p = 0; p < PLANES; ++p) bf[j][p] = *(const bf16x8*)(lb + p * SB::PLANE + fb[h] + j * 2048);
      // small terms first; consecutive MFMAs go to different accumulators
#pragma unroll
      for (int s = PLANES - 1; s >= 0; --s)
#pragma unroll
        for (int p = 0; p <= s; ++p)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i][p], bf[j][s - p], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  exchange();

  // f(row0, col, tile's accumulator, first, last) for every 32x32 tile this wavefront keeps values of: value v of lane l sits at
  // row 8*(v/4) + 4*(l/32) + v%4, column l%32 of its tile
  auto kept = [&](auto f) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int t16 = (i * TN + j) * 16;
        const int first = WVK == 1 ? 0 : min(max(wk * KEEP - t16, 0), 16), last = WVK == 1 ? 16 : min(max((wk + 1) * KEEP - t16, 0), 16);
        const int col = n0 + wn + j * 32 + l32;
        if (first < last && col < g.N) f(m0 + wm + i * 32 + lhi * 4, col, acc[i][j], first, last);
      }
  };

  if constexpr (PLANES > 1) {  // (see the head of the file)
    const bool lossy = sa.least < LEAST_WHOLE || sb.least < LEAST_WHOLE;
    if (__syncthreads_or(sa.largest > SURELY_IN_RANGE || sb.largest > SURELY_IN_RANGE || lossy)) {
      int* const top = reinterpret_cast<int*>(lds);  // (magnitudes order as their bits do)
      if (threadIdx.x < 2) top[threadIdx.x] = 0;
      __syncthreads();
      atomicMax(top, __float_as_int(sa.largest));
      atomicMax(top + 1, __float_as_int(sb.largest));
      __syncthreads();
      const float top_a = __int_as_float(top[0]), top_b = __int_as_float(top[1]);
      bool whole = parts_in_range(top_a, top_b, k_end - k_begin);
      if (__syncthreads_or(lossy)) {
        const float limit = (float)(k_end - k_begin) * LOSSLESS_SUM * (top_a + top_b);
        bool small = false;
        kept([&](int row0, int, const f16v& a, int first, int last) {
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int row = row0 + (v >> 2) * 8 + (v & 3);
            if (fabsf(a[v]) < limit && v >= first && v < last && row < g.M && ep.map_row(row) >= 0) small = true;
          }
        });
        whole = !__syncthreads_or(small || !whole);
      }
      if (!whole) {
        // Everything is worked out anew from values the compiler cannot know to be the same: nothing is kept in registers
        // through the loop above for the sake of this one.
        int tid = threadIdx.x, from = k_begin;
        asm volatile("" : "+v"(tid), "+s"(from));
        sa.template init<true>(al, tid, m0, from);
        sb.template init<true>(bl, tid, n0, from);
        clear();
        sa.fetch(al, from + BK > k_end);
        sb.fetch(bl, from + BK > k_end);
        const int khalf = (tid >> 5) & 1, part = ((tid >> 6) % WVK) * (BK / WVK) + khalf;
        const uint32_t fa32 = SA::f32_place(wm + (tid & 31) + 4, part), fb32 = SB::f32_place(wn + (tid & 31) + 4, part);
#pragma unroll 1
        for (int k0 = from; k0 < k_end; k0 += BK) {
          sa.stage_f32(la);
          sb.stage_f32(lb);
          __syncthreads();
          if (k0 + BK < k_end) {
            const bool tail = k0 + 2 * BK > k_end;
            sa.fetch(al, tail);
            sb.fetch(bl, tail);
          }
#pragma unroll 1
          for (int k = 0; k < BK / WVK; k += 2) {
            float af[TM], bf[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) af[i] = *(const float*)(la + fa32 + k * (SA::ROWS * 4) + i * 128);
#pragma unroll
            for (int j = 0; j < TN; ++j) bf[j] = *(const float*)(lb + fb32 + k * (SB::ROWS * 4) + j * 128);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
              for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[i], bf[j], acc[i][j], 0, 0, 0);
          }
          __syncthreads();
        }
        exchange();
      }
    }
  }
  float* const part = g.ws ? g.ws + (int64_t)bz * g.ws_rows * g.N : nullptr;

  kept([&](int row0, int col, const f16v& a, int first, int last) {
    if (part) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int row = row0 + (v >> 2) * 8 + (v & 3);
        const int to = v >= first && v < last && row < g.M ? ep.map_row(row) : -1;
        if (to >= 0) part[(int64_t)to * g.N + col] = a[v];
      }
    } else {
      store16(ep, row0, col, a, g.M, first, last);
    }
  });

  if constexpr (!BL::KC) {
    if (sum_columns) {  // a group of four columns was read by KG threads (one per group of k): their sums meet in LDS
      __syncthreads();
      float* cs = reinterpret_cast<float*>(lds);
      if (sb.on) *(f4v*)(cs + SB::kgroup(threadIdx.x) * BN + SB::ogroup(threadIdx.x) * 4) = sb.colsum;
      __syncthreads();
      if ((int)threadIdx.x < BN) {
        const int c = bl.row(n0 + ((int)threadIdx.x & ~3)) + ((int)threadIdx.x & 3);  // (a moved group repeats its neighbour's columns)
        float s = 0.f;
#pragma unroll
        for (int q = 0; q < SB::KG; ++q) s += cs[q * BN + threadIdx.x];
        if (part) part[(int64_t)g.colsum_row * g.N + c] = s;
        else ep.store(g.colsum_row, c, s);
      }
    }
  }
}

}  // namespace sn
