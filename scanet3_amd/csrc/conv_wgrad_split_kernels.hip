// Conv2D filter gradient on bf16 matrix instructions (the split products of split_gemm.hpp) with the POSITION as the k index and both
// operands loaded straight from the tensors: nothing is staged and no barrier stands in the loop.
//
//   dW[r, j, n] = sum over output positions p of x[run of p in filter row r][j] * dy[p][n],   j = q * cin + channel < L = kw * cin
//   (math/nn/AllKernels.scala:211-261: the filter's side of Conv2D's gradient)
//
// For a fixed filter row the taps' channels of a position are one run of L consecutive floats of x, so a tile of 32 values of j x 32
// filters is one accumulator of v_mfma_f32_32x32x16_bf16: lane l supplies value j = l % 32 (filter n = l % 32) of 8 positions,
// 8 * (l / 32) and on of a chunk of 16, as 8 loads of 4 bytes, of which 32 neighbouring lanes read 128 consecutive bytes.  A wavefront
// keeps TM x TN tiles and walks chunks of positions; every operand tile is taken apart once for the TN (TM) products it is in, during
// the products of the tile before, and the next chunk's values are requested as soon as its registers are free.  Where a
// position's run begins comes from a table in LDS, made for 512 chunks at a time; under padding a second one holds which rows and
// columns of the run lie inside the image.  Positions beyond the last, and values outside the image, are loads from beyond
// the tensor, answered with zeros.  The 8 wavefronts of a workgroup add their tiles in LDS, in wavefront order; every workgroup leaves
// a partial result for its range of positions, and the caller adds these in part order.
//
// What bounds it: instruction issue.  A chunk of the 3 x 2 tiles is 36 matrix instructions of 32 cycles and, for two wavefronts of a
// SIMD each, some 550 others that fetch, take five tiles apart and add; behind them, for few positions, the tiles' sums in LDS and
// the partial results.  A tile of x is read again by every 64 filters and a tile of dy by every filter row, by workgroups of one XCD.
// Microseconds without the sum of the partial results, positions x filters x values (channels), the kernels before -> this one:
//   52900 x 64 x 288 (32) 29.5 -> 25.1   121000 x 64 x 288 (32) 64 -> 42    529000 x 64 x 288 (32) 216 -> 150   28800 x 64 x 800 (32) 47 -> 36
//   32000 x 80 x 432 (48) 57 -> 39       204768 x 40 x 81 (9) 50 -> 35      409948 x 15 x 522 (58) 262 -> 168   193536 x 73 x 288 (32) 170 -> 108
//   7840 x 64 x 342 (38) 15.0 -> 12.5    20736 x 8 x 144 (16) 11.2 -> 9.9   12544 x 128 x 576 (64) 38 -> 25     1031742 x 8 x 216 (24) 246 -> 169
// (3 x 2 tiles under padding spill 16 registers and are still faster than 2 x 2: 313308 x 64 x 207 (23) 98 against 122.)
// Gradients below 2^-110 (a saturated softmax's) multiplied in float32 as well: 111132 x 96 x 324 (36) 271 -> 217.
#include "split_launch.hpp"

#include "conv_wgrad_split_rules.hpp"

namespace sn {
namespace {

typedef uint32_t u4v __attribute__((ext_vector_type(4)));

constexpr uint32_t OOB = 0x80000000u;  // beyond any operand (tensors are checked to be < 2 GiB)
constexpr int SEGMENT = 512;           // chunks of 16 positions whose table LDS holds at a time

struct WgradArgs {
  const float* x;
  const float* dy;
  uint32_t x_bytes, dy_bytes;
  int M, wo;              // positions (b, oh, ow)
  FastDiv by_wo, by_ho, by_c;
  int sh, sw, pt, pl, H, W, C, kh, kw, L, N;
  int groups_m, groups_n, parts, chunks;
  float* ws;              // [part][kh * L][N]
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ float load4(__amdgpu_buffer_rsrc_t rs, uint32_t off) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, (int)off, 0, 0));
}

template <int TM, int TN, bool PADDED>
__global__ __launch_bounds__(512) void conv_wgrad_split_kernel(WgradArgs a) {
  __shared__ __attribute__((aligned(16))) uint32_t begins[SEGMENT * 16];                       // byte offset of a position's run
  __shared__ __attribute__((aligned(16))) uint32_t insides[PADDED ? SEGMENT * 16 : 1];         // bit r: row r, bit 16 + q: column q inside the image
  __shared__ float sums[8][16 * 64];
  const int groups = a.kh * a.groups_m * a.groups_n;
  const int per_xcd = (int)gridDim.x >> 3, index = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
  if (index >= groups * a.parts) return;  // (the grid is rounded up to whole XCDs; what shares a range of positions shares an XCD)
  const int part = index / groups, group = index - part * groups;
  const int r = group / (a.groups_m * a.groups_n), gmn = group - r * a.groups_m * a.groups_n, gm = gmn / a.groups_n, gn = gmn - gm * a.groups_n;
  const int j0 = gm * TM * 32, n0 = gn * TN * 32;
  const int chunk_begin = (int)((int64_t)a.chunks * part / a.parts), chunk_end = (int)((int64_t)a.chunks * (part + 1) / a.parts);

  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, lhi = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(a.x, a.x_bytes), ry = make_rsrc(a.dy, a.dy_bytes);

  // this lane's part of the addresses, and what a position has to have for its value to count
  const uint32_t x_lane = (uint32_t)(r * a.W * a.C + j0 + l32) * 4u;
  uint32_t need[TM], y_lane[TN];
#pragma unroll
  for (int t = 0; t < TM; ++t) {
    const int q = (int)div_by((uint32_t)(j0 + 32 * t + l32), a.by_c);
    need[t] = (1u << r) | (1u << (16 + min(q, 15)));
  }
#pragma unroll
  for (int t = 0; t < TN; ++t) y_lane[t] = (uint32_t)min(n0 + 32 * t + l32, a.N - 1) * 4u;

  f16v acc[TM][TN];
  uint32_t least_x = 0xffffffffu, least_y = 0xffffffffu;
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
  };
  clear();

  // The table of a segment: begins[chunk][half][8].  Positions beyond the last begin beyond the tensor.
  auto make_table = [&](int first, int last) {
    __syncthreads();
    for (int i = tid; i < (last - first) * 16; i += 512) {
      const int m = first * 16 + i;
      const uint32_t mm = (uint32_t)min(m, a.M - 1), t = div_by(mm, a.by_wo), b = div_by(t, a.by_ho);
      const int y0 = (int)(t - b * a.by_ho.d) * a.sh - a.pt, x0 = (int)(mm - t * (uint32_t)a.wo) * a.sw - a.pl;
      begins[i] = m < a.M ? (uint32_t)((((int)b * a.H + y0) * a.W + x0) * a.C) * 4u : OOB;
      if constexpr (PADDED) {
        uint32_t in = 0;
        for (int k = 0; k < a.kh; ++k) in |= (unsigned)(y0 + k) < (unsigned)a.H ? 1u << k : 0u;
        for (int k = 0; k < a.kw; ++k) in |= (unsigned)(x0 + k) < (unsigned)a.W ? 1u << (16 + k) : 0u;
        insides[i] = m < a.M ? in : 0u;
      }
    }
    __syncthreads();
  };
  struct Places {
    u4v begin[2], inside[PADDED ? 2 : 1];
  };
  auto places = [&](int slot, Places& p) {  // of this lane's 8 positions of a chunk of the table
    const uint32_t at = (uint32_t)(slot * 16 + lhi * 8);
    p.begin[0] = *(const u4v*)(begins + at);
    p.begin[1] = *(const u4v*)(begins + at + 4);
    if constexpr (PADDED) {
      p.inside[0] = *(const u4v*)(insides + at);
      p.inside[1] = *(const u4v*)(insides + at + 4);
    }
  };
  auto fetch_x = [&](const Places& p, int t, float (&v)[8]) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      uint32_t off = p.begin[k >> 2][k & 3] + x_lane + 128u * (uint32_t)t;
      if constexpr (PADDED) off = (p.inside[k >> 2][k & 3] & need[t]) == need[t] ? off : OOB;
      v[k] = load4(rx, off);
    }
  };
  auto fetch_y = [&](int chunk, int t, float (&v)[8]) {
    const uint32_t at = (uint32_t)(chunk * 16 + lhi * 8) * (uint32_t)a.N * 4u + y_lane[t];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = load4(ry, at + (uint32_t)(k * a.N) * 4u);
  };
  auto take_apart = [&](const float (&v)[8], uint32_t& least, bf16x8 (&out)[3]) {
    u4v q[3];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      least = min(min(least, magnitude_key(v[2 * k])), magnitude_key(v[2 * k + 1]));
      uint32_t p[3];
      split_pair<3>(v[2 * k], v[2 * k + 1], p);
#pragma unroll
      for (int i = 0; i < 3; ++i) q[i][k] = p[i];
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) out[i] = __builtin_bit_cast(bf16x8, q[i]);
  };

  for (int first = chunk_begin; first < chunk_end; first += SEGMENT) {
    const int last = min(first + SEGMENT, chunk_end);
    make_table(first, last);
    // (chunks beyond the segment's last are requested too, for the sake of one order of loads, from the last one's places)
    const int mine = first + wave;
    if (mine >= last) continue;
    Places p;
    float x[TM][8], y[TN][8];
    bf16x8 xa[3], ya[TN][3];
    places(mine - first, p);
#pragma unroll
    for (int t = 0; t < TN; ++t) fetch_y(mine, t, y[t]);
#pragma unroll
    for (int t = 0; t < TM; ++t) fetch_x(p, t, x[t]);
    int next = min(mine + 8, last - 1);
    places(next - first, p);
#pragma unroll
    for (int t = 0; t < TN; ++t) {
      take_apart(y[t], least_y, ya[t]);
      fetch_y(next, t, y[t]);
    }
    take_apart(x[0], least_x, xa);
    fetch_x(p, 0, x[0]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
    for (int chunk = mine; chunk < last; chunk += 8) {
      // tile t of x against every tile of dy, while the next tile is taken apart and requested anew; behind the last one those of
      // the next chunk
#pragma unroll
      for (int t = 0; t < TM; ++t) {
        bf16x8 xn[3], yn[TN][3];
        if (t + 1 < TM) {
          take_apart(x[t + 1], least_x, xn);
          fetch_x(p, t + 1, x[t + 1]);
        } else {
          next = min(next + 8, last - 1);
          places(next - first, p);
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            take_apart(y[j], least_y, yn[j]);
            fetch_y(next, j, y[j]);
          }
          take_apart(x[0], least_x, xn);
          fetch_x(p, 0, x[0]);
        }
        // A chunk's five small products have a sum of their own, small terms first, and are added to what hi x hi leaves: two roundings at
        // the result's magnitude in 16 positions, one of them the matrix unit's.  Relative error against float64 at the sizes below:
        // 1.2e-7 to 2.7e-7, where the float32 kernels leave 1.9e-7 to 2.1e-6 (all six onto one sum: 1.9e-7 to 1.9e-6).
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          f16v sum;
#pragma unroll
          for (int v = 0; v < 16; ++v) sum[v] = 0.f;
#pragma unroll
          for (int s = 2; s >= 1; --s)
#pragma unroll
            for (int i = 0; i <= s; ++i) sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa[i], ya[j][s - i], sum, 0, 0, 0);
          acc[t][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa[0], ya[j][0], acc[t][j], 0, 0, 0);
          acc[t][j] += sum;
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) xa[i] = xn[i];
        if (t + 1 == TM) {
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int i = 0; i < 3; ++i) ya[j][i] = yn[j][i];
        }
        // the order of issue: a matrix instruction at a time with what hides behind it
        if (t + 1 < TM) {
#pragma unroll
          for (int i = 0; i < 6 * TN; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, (72 + 16 * TN + 6 * TN - 1) / (6 * TN), 0);
            __builtin_amdgcn_sched_group_barrier(0x020, (8 + 6 * TN - 1) / (6 * TN), 0);
          }
        } else {
#pragma unroll
          for (int i = 0; i < 6 * TN; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 12 * (TN + 1) / TN + 3, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, 3, 0);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  // The ends of the range (split_gemm.hpp): a part or a part product beyond it leaves an Inf or a NaN behind, for good; values below
  // 2^-110 lose bits that a small sum would show.  Either way this wavefront's share is multiplied in float32.
  const bool lossy = __any(least_x < LEAST_WHOLE || least_y < LEAST_WHOLE);
  auto counts = [&](int i, int v) { return j0 + 32 * i + (v >> 2) * 8 + 4 * lhi + (v & 3) < a.L; };
  bool again = false;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) again |= !(fabsf(acc[i][j][v]) <= 3.4028234663852886e38f) && counts(i, v);
  again = __any(again);
  // this lane's 8 positions of a chunk, requested together; from one position to the next it is one step, unless a row or an image ends
  int column[TM];  // the run's column of this lane's value; none inside the image for a value behind the run
#pragma unroll
  for (int t = 0; t < TM; ++t) {
    const int j = j0 + 32 * t + l32;
    column[t] = j < a.L ? (int)div_by((uint32_t)j, a.by_c) : 1 << 30;
  }
  const uint32_t step = (uint32_t)(a.sw * a.C) * 4u, row_step = (uint32_t)((a.sh * a.W - a.wo * a.sw) * a.C) * 4u;
  const uint32_t image_step = (uint32_t)((a.H - (int)a.by_ho.d * a.sh) * a.W * a.C) * 4u;
  auto fetch_all = [&](int chunk, float (&fx)[TM][8], float (&fy)[TN][8]) {
    const int m = chunk * 16 + lhi * 8;
    const uint32_t mm = (uint32_t)min(m, a.M - 1), row = div_by(mm, a.by_wo), b = div_by(row, a.by_ho);
    int ow = (int)(mm - row * (uint32_t)a.wo), oh = (int)(row - b * a.by_ho.d), x0 = ow * a.sw - a.pl, y = oh * a.sh - a.pt + r;
    uint32_t begin = (uint32_t)((((int)b * a.H + y) * a.W + x0) * a.C) * 4u;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const bool row_in = m + k < a.M && (unsigned)y < (unsigned)a.H;
#pragma unroll
      for (int t = 0; t < TM; ++t)
        fx[t][k] = load4(rx, row_in && (unsigned)(x0 + column[t]) < (unsigned)a.W ? begin + (uint32_t)(j0 + 32 * t + l32) * 4u : OOB);
      const bool row_ends = ++ow == a.wo;
      ow = row_ends ? 0 : ow;
      x0 = row_ends ? -a.pl : x0 + a.sw;
      oh += row_ends ? 1 : 0;
      begin += step + (row_ends ? row_step : 0u);
      const bool image_ends = oh == (int)a.by_ho.d;
      oh = image_ends ? 0 : oh;
      y = image_ends ? r - a.pt : y + (row_ends ? a.sh : 0);
      begin += image_ends ? image_step : 0u;
    }
#pragma unroll
    for (int t = 0; t < TN; ++t) fetch_y(chunk, t, fy[t]);
  };
  if (lossy && !again) {
    float top_x = 0.f, top_y = 0.f;
    for (int c = chunk_begin + wave; c < chunk_end; c += 8) {
      float fx[TM][8], fy[TN][8];
      fetch_all(c, fx, fy);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
#pragma unroll
        for (int t = 0; t < TM; ++t) top_x = max_magnitude(top_x, fx[t][k], 0.f);
#pragma unroll
        for (int t = 0; t < TN; ++t) top_y = max_magnitude(top_y, fy[t][k], 0.f);
      }
    }
    for (int o = 32; o > 0; o >>= 1) {
      top_x = fmaxf(top_x, __shfl_xor(top_x, o));
      top_y = fmaxf(top_y, __shfl_xor(top_y, o));
    }
    const float limit = (float)((chunk_end - chunk_begin) * 16) * LOSSLESS_SUM * (top_x + top_y);
    bool small = false;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) small |= fabsf(acc[i][j][v]) < limit && counts(i, v) && n0 + 32 * j + l32 < a.N;
    again = __any(small);
  }
  if (again) {
    clear();
    for (int c = chunk_begin + wave; c < chunk_end; c += 8) {
      float fx[TM][8], fy[TN][8];
      fetch_all(c, fx, fy);
#pragma unroll
      for (int k = 0; k < 8; ++k)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fx[i][k], fy[j][k], acc[i][j], 0, 0, 0);
    }
  }

  float* const out = a.ws + ((int64_t)part * a.kh + r) * a.L * a.N;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      __syncthreads();
#pragma unroll
      for (int v = 0; v < 16; ++v) sums[wave][v * 64 + lane] = acc[i][j][v];
      __syncthreads();
#pragma unroll
      for (int e = tid; e < 1024; e += 512) {
        float s = 0.f;
#pragma unroll
        for (int w = 0; w < 8; ++w) s += sums[w][e];
        const int v = e >> 6, l = e & 63, row = j0 + 32 * i + (v >> 2) * 8 + 4 * (l >> 5) + (v & 3), col = n0 + 32 * j + (l & 31);
        if (row < a.L && col < a.N) out[(int64_t)row * a.N + col] = s;
      }
    }
}

template <int TM, int TN, bool PADDED>
int launch_tiles(sn_ctx* ctx, const WgradArgs& a) {
  LaunchScope scope(ctx, "conv2d_filter_gradient_split", a.kh * a.L, a.N, a.M);
  hipLaunchKernelGGL((conv_wgrad_split_kernel<TM, TN, PADDED>), dim3((unsigned)(8 * ceil_div((int64_t)a.kh * a.groups_m * a.groups_n * a.parts, 8))),
                     dim3(512), 0, ctx->stream, a);
  SN_HIP(hipGetLastError());
  return SN_OK;
}
template <bool PADDED>
int launch_shape(sn_ctx* ctx, const WgradArgs& a, int tm, int tn) {
  switch (tm * 4 + tn) {
    case 5: return launch_tiles<1, 1, PADDED>(ctx, a);
    case 6: return launch_tiles<1, 2, PADDED>(ctx, a);
    case 7: return launch_tiles<1, 3, PADDED>(ctx, a);
    case 9: return launch_tiles<2, 1, PADDED>(ctx, a);
    case 10: return launch_tiles<2, 2, PADDED>(ctx, a);
    case 13: return launch_tiles<3, 1, PADDED>(ctx, a);
    default: return launch_tiles<3, 2, PADDED>(ctx, a);
  }
}

}  // namespace

int launch_conv_wgrad_split(sn_ctx* ctx, const ConvGeom& g, const float* x, const float* dy, float* dw, float* ws, int64_t ws_elems) {
  const WgradSplitPlan p = conv_wgrad_split_plan(g, ctx->compute_units, ws_elems);
  SN_REQUIRE(ws && p.parts >= 1, "conv2d_filter_gradient_split: workspace too small");
  WgradArgs a{};
  a.x = x;
  a.dy = dy;
  a.x_bytes = (uint32_t)((int64_t)g.n * g.h * g.w * g.cin * 4);
  a.dy_bytes = (uint32_t)((int64_t)g.n * g.ho * g.wo * g.cout * 4);
  a.M = g.n * g.ho * g.wo;
  a.wo = g.wo;
  a.by_wo = fast_div((uint32_t)g.wo);
  a.by_ho = fast_div((uint32_t)g.ho);
  a.by_c = fast_div((uint32_t)g.cin);
  a.sh = g.sh; a.sw = g.sw; a.pt = g.pt; a.pl = g.pl; a.H = g.h; a.W = g.w; a.C = g.cin; a.kh = g.kh; a.kw = g.kw;
  a.L = g.kw * g.cin;
  a.N = g.cout;
  a.groups_m = p.groups_m; a.groups_n = p.groups_n; a.parts = p.parts; a.chunks = p.chunks;
  a.ws = ws;
  if (p.padded) SN_TRY(launch_shape<true>(ctx, a, p.tm, p.tn));
  else SN_TRY(launch_shape<false>(ctx, a, p.tm, p.tn));
  Epilogue e;
  e.out = dw;
  e.ldo = g.cout;
  return launch_split_reduce(ctx, ws, p.parts, g.kh * a.L, g.cout, StdEpilogue{e});
}

}  // namespace sn
