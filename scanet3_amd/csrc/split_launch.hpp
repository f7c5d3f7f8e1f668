// Host side of the split products (split_gemm.hpp): tile and split-K choice, launch, and the kernels that add partial sums.
#pragma once

#include "split_gemm.hpp"

#include <algorithm>

namespace sn {

// Adds the split-K partial tiles.  Eight lanes share one output: lane g adds splits g, g+8, ... in order, then the
// eight partial sums are combined pairwise (a fixed tree), so the result does not depend on the launch shape.
template <class EP>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ ws, int splits, int M, int N, EP ep) {
  const int64_t total = (int64_t)M * N;
  const int g = threadIdx.x >> 5, j = threadIdx.x & 31;  // 8 groups of 32 consecutive outputs
  for (int64_t base = (int64_t)blockIdx.x * 32; base < total; base += (int64_t)gridDim.x * 32) {
    const int64_t i = base + j;
    float s = 0.f;
    if (i < total) {
      int z = g;
      for (; z + 120 < splits; z += 128) {  // 16 loads in flight, added in split order
        float a[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) a[u] = ws[(int64_t)(z + 8 * u) * total + i];
#pragma unroll
        for (int u = 0; u < 16; ++u) s += a[u];
      }
      for (; z + 24 < splits; z += 32) {  // 4 loads in flight
        float a[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) a[u] = ws[(int64_t)(z + 8 * u) * total + i];
#pragma unroll
        for (int u = 0; u < 4; ++u) s += a[u];
      }
      for (; z < splits; z += 8) s += ws[(int64_t)z * total + i];
    }
    __shared__ float part[8][32];
    part[g][j] = s;
    __syncthreads();
    if (g == 0 && i < total) {
      const float t = ((part[0][j] + part[1][j]) + (part[2][j] + part[3][j])) + ((part[4][j] + part[5][j]) + (part[6][j] + part[7][j]));
      ep.store((int)(i / N), (int)(i % N), t);
    }
    __syncthreads();
  }
}

// The same reduction when M*N is a multiple of 4 (every partial tile then starts on a 16-byte boundary): a lane owns 4
// consecutive outputs and reads them as one 16-byte load per split; every output sees the same additions in the same order.
template <class EP>
__global__ __launch_bounds__(256) void splitk_reduce4_kernel(const float* __restrict__ ws, int splits, int M, int N, EP ep) {
  const int64_t total4 = (int64_t)M * N / 4;
  const int g = threadIdx.x >> 5, j = threadIdx.x & 31;  // 8 groups of 32 lanes x 4 consecutive outputs
  for (int64_t base = (int64_t)blockIdx.x * 32; base < total4; base += (int64_t)gridDim.x * 32) {
    const int64_t i = base + j;
    f4v s = {0.f, 0.f, 0.f, 0.f};
    if (i < total4) {
      const f4v* w4 = reinterpret_cast<const f4v*>(ws) + i;
      int z = g;
      for (; z + 56 < splits; z += 64) {  // 8 loads of 16 bytes in flight, added in split order
        f4v a[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) a[u] = w4[(int64_t)(z + 8 * u) * total4];
#pragma unroll
        for (int u = 0; u < 8; ++u) s += a[u];
      }
      for (; z < splits; z += 8) s += w4[(int64_t)z * total4];
    }
    __shared__ f4v part4[8][32];
    part4[g][j] = s;
    __syncthreads();
    if (g == 0 && i < total4) {
      const f4v t = ((part4[0][j] + part4[1][j]) + (part4[2][j] + part4[3][j])) + ((part4[4][j] + part4[5][j]) + (part4[6][j] + part4[7][j]));
      // row and column of the first of the four outputs by one division (32-bit where the index allows: a 64-bit division
      // is some hundred instructions on this device), the others by stepping
      const int64_t o0 = i * 4;
      int m, n;
      if (o0 < ((int64_t)1 << 31)) {
        const uint32_t q = (uint32_t)o0 / (uint32_t)N;
        m = (int)q;
        n = (int)((uint32_t)o0 - q * (uint32_t)N);
      } else {
        m = (int)(o0 / N);
        n = (int)(o0 % N);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        ep.store(m, n, t[e]);
        if (++n == N) { n = 0; ++m; }
      }
    }
    __syncthreads();
  }
}

// Whether a caller that applies the optimizer next (ctx->defer) can add the partial results: every sum goes straight to one
// contiguous tensor, `plain`, in vectors of four, and there are enough of them to be worth a section of that launch.
template <class EP>
inline float* split_plain_destination(const EP& ep, int N) {
  if constexpr (std::is_same<EP, StdEpilogue>::value) {
    if (!ep.e.bias && ep.e.act == SN_ACT_IDENTITY && ep.e.row_index < 0 && ep.e.ldo == N) return ep.e.out;
  } else if constexpr (std::is_same<EP, RunRowsEpilogue>::value) {
    if (ep.ldo == N) return ep.out;
  }
  return nullptr;
}
inline bool split_defers(const float* plain, const float* ws, int M, int N) {
  const int64_t total = (int64_t)M * N;
  return plain && total % 4 == 0 && total >= 4096 && total < ((int64_t)1 << 30) && (reinterpret_cast<uintptr_t>(ws) & 15u) == 0;
}

// Adds `splits` partial results [split][M][N] and hands every sum to the epilogue, or leaves that to a caller that applies
// the optimizer next.
template <class EP>
static int launch_split_reduce(sn_ctx* ctx, const float* ws, int splits, int M, int N, const EP& ep) {
  const int64_t total = (int64_t)M * N;
  const bool aligned = (reinterpret_cast<uintptr_t>(ws) & 15u) == 0;
  float* const plain = split_plain_destination(ep, N);
  if (ctx->defer && split_defers(plain, ws, M, N)) {
    *ctx->defer = DeferredReduce{1, ws, splits, (int)total, plain};
    ctx->defer = nullptr;
    return SN_OK;
  }
  LaunchScope scope(ctx, "splitk_reduce");
  if (total % 4 == 0 && total >= 4096 && aligned) {
    const int64_t blocks = std::min<int64_t>(ceil_div(total / 4, 32), (int64_t)ctx->compute_units * 16);
    hipLaunchKernelGGL((splitk_reduce4_kernel<EP>), dim3((unsigned)blocks), dim3(256), 0, ctx->stream, ws, splits, M, N, ep);
  } else {
    const int64_t blocks = std::min<int64_t>(ceil_div(total, 32), (int64_t)ctx->compute_units * 16);
    hipLaunchKernelGGL((splitk_reduce_kernel<EP>), dim3((unsigned)blocks), dim3(256), 0, ctx->stream, ws, splits, M, N, ep);
  }
  SN_HIP(hipGetLastError());
  return SN_OK;
}

// Tile and split count for a product of M x N x K: the cheapest by a model of what a launch costs.  Per tile shape: the time
// per 32 k-values of a workgroup that has its CU to itself (a chain of load, split, store, read, multiply), and of a CU that
// is full of workgroups, per workgroup (measured on MI355X: 288 x 64 x 52900 in one split, 8192 x 4096 x 4096; the bf16 column, one plane
// instead of three, by the tiles and splits of 655 products of 16 to 8192 rows, 17 to 4096 columns and as long sums, forward, input and weight
// gradient: the chosen ones take 1.026 times the fastest on the mean).  A launch lasts as long as its fullest CU; splitting K costs
// the partial sums' way through memory and the launch that adds them.
// One plane has nothing to take apart; where a CU holds several workgroups, what it can fetch bounds them, and larger tiles fetch
// less: 2124 x 2820 x 220 19.4 us in tiles of 128 x 128, 1869 x 1496 x 1312 (weight gradient) 35.4 in 64 x 64 and 43.5 in 128 x 128, 1000 x 1500 x
// 1000 22.8 in 64 x 64 x 64 and 25.3 in 64 x 32.  Tiles of 128 x 64 were the fastest of one product in those 655 (two wavefronts of 64 x 64 each a
// half of K: three and more of them on a CU take as long each as tiles of 128 x 128, 2124 x 2820 x 220 31.1 us), and are not built for one plane.
// (Three stages of loads in flight instead of one, with every wait counting on the loads behind it, were measured over all tiles: 20 to
// 60 % slower where a CU holds several workgroups, whose registers they take, and within 5 % of the same where it holds one.)
struct SplitTile {
  int bm, bn, bk;
  float lone[2], full[2];  // microseconds; [0] three planes (float32), [1] one plane (bf16)
};
enum { TILE_128x128, TILE_128x64, TILE_64x64, TILE_64x64_DEEP, TILE_64x32_DEEP, TILE_32x64_DEEP, SPLIT_TILES };
constexpr SplitTile SPLIT_TILE[SPLIT_TILES] = {
    {128, 128, 32, {1.45f, 1.00f}, {1.45f, 0.68f}}, {128, 64, 32, {1.14f, 0.f}, {0.85f, 0.f}},  {64, 64, 32, {0.83f, 0.68f}, {0.47f, 0.29f}},
    {64, 64, 64, {0.60f, 0.46f}, {0.52f, 0.30f}},   {64, 32, 64, {0.44f, 0.31f}, {0.31f, 0.21f}}, {32, 64, 64, {0.46f, 0.29f}, {0.34f, 0.23f}}};
struct SplitChoice {
  int tile = 0, splits = 1;
};
inline SplitChoice split_choose(int M, int N, int K, int cu, int64_t max_parts, bool deferred, int planes) {
  static const int counts[] = {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32, 48, 64, 96, 128, 192, 256};
  SplitChoice best;
  float best_us = 1e30f;
  const int p = planes == 1 ? 1 : 0;
  for (int t = 0; t < SPLIT_TILES; ++t) {
    const SplitTile& c = SPLIT_TILE[t];
    if (c.full[p] == 0.f) continue;  // no such tile
    const int64_t tiles = ceil_div(M, c.bm) * ceil_div(N, c.bn);
    const int stages = (int)ceil_div(K, c.bk);
    for (int wanted : counts) {
      if (wanted > max_parts && wanted > 1) break;
      const int per = (int)ceil_div(stages, wanted), s = (int)ceil_div(stages, per);  // (the same s gives the same `per` again)
      if (s > 1 && per * c.bk < 64) continue;
      const float wgs = (float)ceil_div(tiles * s, cu);
      float us = 3.0f + (float)(per * c.bk / 32) * std::max(c.lone[p], wgs * c.full[p]);
      if (s > 1) us += (deferred ? 1.0f : 4.5f) + 8.0e-6f * (float)s * (float)M * (float)N / 3.5f;
      if (us < best_us) {
        best_us = us;
        best.tile = t;
        best.splits = s;
      }
    }
  }
  return best;
}
inline int64_t split_workspace_elems(int m, int n, int k, int cu) {
  int splits = 1;
  for (int planes : {1, 3})
    for (bool deferred : {false, true}) splits = std::max(splits, split_choose(m, n, k, cu, 256, deferred, planes).splits);
  return splits > 1 ? (int64_t)splits * (m + 1) * n : 0;
}

template <int BM, int BN, int BK, int WVM, int WVN, int WVK, int PLANES, class AL, class BL, class EP>
static int launch_split_tile(sn_ctx* ctx, SplitGrid g, int splits, const AL& al, const BL& bl, const EP& ep) {
  typedef SplitShape<BM, BN, BK, WVM, WVN, WVK, PLANES, AL, BL> Shape;
  auto kernel = split_gemm_kernel<BM, BN, BK, WVM, WVN, WVK, PLANES, AL, BL, EP>;
  g.k_per_split = (int)(ceil_div(ceil_div(g.K, BK), splits) * BK);
  g.splits = (int)ceil_div(g.K, g.k_per_split);
  if (g.splits == 1) g.ws = nullptr;
  g.tiles_m = (int)ceil_div(g.M, BM);
  g.tiles_n = (int)ceil_div(g.N, BN);
  if (Shape::LDS > 64 * 1024) SN_TRY(allow_dynamic_lds(ctx, reinterpret_cast<const void*>(kernel), Shape::LDS));
  const int64_t items = (int64_t)g.tiles_m * g.tiles_n * g.splits;
  SN_REQUIRE(items < ((int64_t)1 << 30), "product of %d x %d x %d: too many tiles", g.M, g.N, g.K);
  hipLaunchKernelGGL(kernel, dim3((unsigned)(8 * ceil_div(items, 8))), dim3(Shape::T), Shape::LDS, ctx->stream, g, al, bl, ep);
  SN_HIP(hipGetLastError());
  return SN_OK;
}

// M rows of the product (without the column-sum row; colsum_row >= 0: B's column sums become that output row), `rows` of the
// tensor it goes to
template <int PLANES, class AL, class BL, class EP>
static int launch_split(sn_ctx* ctx, const char* name, int M, int N, int K, int rows, int colsum_row, const AL& al, const BL& bl, const EP& ep,
                        float* ws, int64_t ws_elems) {
  SplitGrid g{};
  g.M = M; g.N = N; g.K = K;
  g.ws_rows = rows;
  g.colsum_row = colsum_row;
  const SplitChoice c = split_choose(M, N, K, ctx->compute_units, ws ? ws_elems / ((int64_t)rows * N) : 1,
                                     ctx->defer && split_defers(split_plain_destination(ep, N), ws, rows, N), PLANES);
  g.ws = c.splits > 1 ? ws : nullptr;
  {
    LaunchScope scope(ctx, name, rows, N, K);
    int rc = SN_OK;
    switch (c.tile) {
      case TILE_128x128: rc = launch_split_tile<128, 128, 32, 4, 2, 1, PLANES>(ctx, g, c.splits, al, bl, ep); break;
      case TILE_128x64:
        if constexpr (PLANES != 1) rc = launch_split_tile<128, 64, 32, 2, 1, 2, PLANES>(ctx, g, c.splits, al, bl, ep);
        break;
      case TILE_64x64_DEEP: rc = launch_split_tile<64, 64, 64, 2, 1, 4, PLANES>(ctx, g, c.splits, al, bl, ep); break;
      case TILE_64x32_DEEP: rc = launch_split_tile<64, 32, 64, 2, 1, 4, PLANES>(ctx, g, c.splits, al, bl, ep); break;
      case TILE_32x64_DEEP: rc = launch_split_tile<32, 64, 64, 1, 2, 4, PLANES>(ctx, g, c.splits, al, bl, ep); break;
      default: rc = launch_split_tile<64, 64, 32, 2, 1, 2, PLANES>(ctx, g, c.splits, al, bl, ep); break;
    }
    SN_TRY(rc);
  }
  return c.splits > 1 ? launch_split_reduce(ctx, ws, c.splits, rows, N, ep) : SN_OK;
}

}  // namespace sn
