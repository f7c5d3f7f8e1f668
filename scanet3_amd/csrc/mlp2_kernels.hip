// Training pass of a small two-layer perceptron in two launches (gfx950):
//
//   Dense(H, act) >> Dense(C, Softmax) under CategoricalCrossentropy, H <= 64 hidden units, C <= 16 classes
//   (layer/Dense.scala:30-71, Activation.scala:46-83, Loss.scala:44-57; the reference's first benchmark configuration
//   784 -> 50 -> 10 at batch 1000).
//
// As a chain of general kernels this step is a dozen dependent launches of 3-9 us each.  Here
//   kernel 1 (one workgroup per 4 batch rows): z1 = x W1 on the matrix cores, h = act(z1 + b1), z2 = h W2 + b2, softmax, the
//     loss terms, dz2, dh = dz2 W2^T, dz1 = act'(h) dh, and these rows' terms of dW2, db1 and db2; dz1 leaves in the order
//     kernel 2's matrix-core fragments want it;
//   kernel 2: dW1 = x^T dz1 on the matrix cores, one workgroup per 16 input features x 16 hidden units, the sums of the row
//     blocks' partial dW2 / db1 / db2, 32 of them a workgroup, and the optimizer.
// Both are chains of latencies, not of bytes: every load of a wavefront is requested before the first is used, the length of the
// products is divided over eight wavefronts that meet in LDS, and the chip is filled (1000 rows are 250 workgroups).  With
// v_mfma_f32_4x4x1_16b_f32 four rows meet 64 hidden units in one instruction of 8 cycles, its second operand one coalesced row
// of W1; 16 rows a workgroup on v_mfma_f32_16x16x4_f32 left 63 workgroups with 196 instructions of 32 cycles one after the
// other.  784 -> 50 -> 10 at batch 1000, by the profiler: 18.4 -> 10.8 us and 15.2 -> 7.2 (4.4 of each are what an empty launch takes).
// Every sum has a fixed order, so results do not depend on the launch.
#include "common.hpp"
#include "optim_update.hpp"

namespace sn {
namespace {

typedef float f4v __attribute__((ext_vector_type(4)));
constexpr int RB = 4;             // batch rows per workgroup of kernel 1
constexpr int MR = 16;            // batch rows of a k-block of kernel 2
constexpr int WAVES = 8;          // of a workgroup, either kernel
constexpr int T = 64 * WAVES;
constexpr int MH = 64;            // hidden units, padded
constexpr int MC = 16;            // classes, padded
constexpr int STEPS = 14;         // k-blocks of kernel 2 per wavefront: 8 * 14 of 16 rows
constexpr int MAX_ROWS = WAVES * STEPS * MR;
constexpr int PARTS = 32;         // partial sums a workgroup of kernel 2 adds up, by T / 32 threads each

struct Mlp2Args {
  const float* x;    // [rows, K]
  const float* y;    // [rows, C]
  const float* w1;   // [K, H]
  const float* b1;   // [H] or null
  const float* w2;   // [H, C]
  const float* b2;   // [C] or null
  float* h;          // [rows, H]
  float* z2;         // [rows, C]
  float* p;          // [rows, C]
  float* dz1f;       // [blocks of 16 rows][4 column blocks][64 lanes][4]: dz1[16 kb + 4 (lane / 16) + j][16 cb + lane % 16]
  float* row_loss;   // [rows]
  float* part;       // [blocks of 4 rows][H * C + H + C]: partial dW2, db1, db2
  float* g_w1; float* g_b1; float* g_w2; float* g_b2;   // gradients (b may be null)
  int rows, K, H, C, act1, stable;
  float act1_param, neg_inv_rows;
  Mlp2Update upd;    // kind >= 0: kernel 2 applies every gradient value it finishes to its parameter
};

// A parameter and its optimizer state, requested ahead of the gradient value that will move it.
struct Parameter {
  float w, s0, s1, s2;
  int64_t off;
  __device__ __forceinline__ void load(const Mlp2Update& u, const float* g_at) {
    off = g_at - u.g;
    w = u.w[off];
    s0 = u.s0[off];
    s1 = u.n_states > 1 ? u.s1[off] : 0.f;
    s2 = u.n_states > 2 ? u.s2[off] : 0.f;
  }
  __device__ __forceinline__ void update(const Mlp2Update& u, float grad) {
    update_any(u.kind, w, grad, s0, s1, s2, u.p);
    u.w[off] = w;
    u.s0[off] = s0;
    if (u.n_states > 1) u.s1[off] = s1;
    if (u.n_states > 2) u.s2[off] = s2;
  }
};

__device__ __forceinline__ float act_fwd1(int act, float v, float param) {
  switch (act) {
    case SN_ACT_SIGMOID: return 1.0f / (1.0f + expf(-v));   // TF Sigmoid
    case SN_ACT_TANH: return tanhf(v);
    case SN_ACT_RELU: return fmaxf(param, v);               // Maximum(threshold, x), Activation.scala:79-82
    default: return v;
  }
}
__device__ __forceinline__ float act_bwd1(int act, float y, float dy, float param) {
  switch (act) {
    case SN_ACT_SIGMOID: return (y * (1.0f - y)) * dy;
    case SN_ACT_TANH: return (1.0f - y * y) * dy;
    case SN_ACT_RELU: return (param < y ? 1.0f : 0.0f) * dy;
    default: return dy;
  }
}

// N: sixteenths of a wavefront's share of the K input features, rounded up (N = 7 for 784)
template <int N>
__global__ __launch_bounds__(T) void mlp2_rows_kernel(Mlp2Args a) {
  constexpr int KW = 16 * N, XP = WAVES * KW + 4;  // x rows as they are divided: wavefront w reads KW values from w * share on
  __shared__ __attribute__((aligned(16))) float Xs[RB][XP];
  __shared__ float sums[WAVES][RB][MH];
  __shared__ float Hs[RB][MH + 1], Ds[RB][MH + 1], Z2[RB][MC + 1], W2s[MH * MC];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int blk = blockIdx.x, r0 = blk * RB;
  const int share = (((a.K + WAVES - 1) / WAVES) + 3) & ~3;  // <= KW
  const int k0 = wave * share, mine = min(share, a.K - k0);  // (mine <= 0: nothing left for this wavefront)

  // ---- every load in flight: the wavefront's rows of W1 (lane = hidden unit; clamped ones are not multiplied or not kept), the x tile
  const float* const wcol = a.w1 + min(lane, a.H - 1);
  float b[KW];
#pragma unroll
  for (int i = 0; i < KW; ++i) b[i] = wcol[(int64_t)min(k0 + i, a.K - 1) * a.H];
  {
    constexpr int QUADS = 256 * RB / T;  // of up to 256 a row
    f4v v[QUADS];
#pragma unroll
    for (int i = 0; i < QUADS; ++i) {
      const int e = tid + i * T, row = e >> 8, q = e & 255;
      v[i] = *(const f4v*)(a.x + (int64_t)min(r0 + row, a.rows - 1) * a.K + 4 * min(q, a.K / 4 - 1));
    }
#pragma unroll
    for (int i = 0; i < QUADS; ++i) {
      const int e = tid + i * T, row = e >> 8, q = e & 255;
      if (4 * q < a.K) *(f4v*)(&Xs[row][4 * q]) = r0 + row < a.rows ? v[i] : f4v{0.f, 0.f, 0.f, 0.f};
    }
  }
  for (int e = tid; e < a.H * a.C; e += T) W2s[e] = a.w2[e];
  __syncthreads();
  // ---- z1: lane l holds x of row l % 4 and hidden unit l of W1; accumulator element v is row v of unit l
  {
    f4v acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    const float* const xr = &Xs[lane & 3][k0];
#pragma unroll
    for (int c = 0; c < N; ++c) {
      f4v x[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = *(const f4v*)(xr + min(16 * c + 4 * i, max(mine - 4, 0)));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (16 * c + 4 * i < mine) {
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[j & 1] = __builtin_amdgcn_mfma_f32_4x4x1f32(x[i][j], b[16 * c + 4 * i + j], acc[j & 1], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int v = 0; v < RB; ++v) sums[wave][v][lane] = acc[0][v] + acc[1][v];
  }
  __syncthreads();
  // ---- h = act(z1 + b1): a wavefront per row, a lane per hidden unit
  if (wave < RB) {
    const int row = wave, col = lane;
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) s += sums[w][row][col];
    float hv = 0.f;
    if (col < a.H && r0 + row < a.rows) {
      hv = act_fwd1(a.act1, a.b1 ? s + a.b1[col] : s, a.act1_param);
      a.h[(int64_t)(r0 + row) * a.H + col] = hv;
    }
    Hs[row][col] = hv;
  }
  __syncthreads();
  // ---- z2 = h W2 + b2 (Dense.scala:57-61, Bias.scala:32-33): eight lanes per row and class, every eighth hidden unit each
  {
    const int row = tid >> 7, c = (tid >> 3) & 15, q = tid & 7;
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < MH / 8; ++i) {
      const int j = q + 8 * i;
      if (j < a.H && c < a.C) s += Hs[row][j] * W2s[j * a.C + c];
    }
#pragma unroll
    for (int off = 4; off > 0; off >>= 1) s += __shfl_xor(s, off, 8);
    if (q == 0 && c < a.C) {
      if (a.b2) s = s + a.b2[c];
      Z2[row][c] = s;
      if (r0 + row < a.rows) a.z2[(int64_t)(r0 + row) * a.C + c] = s;
    }
  }
  __syncthreads();
  // ---- softmax, loss term and d loss / d z2 per row (Activation.scala:63-69, Loss.scala:44-57, general form with epsilon):
  // 16 lanes per row, one class each; the row sums are butterflies over the 16 lanes (a fixed order)
  if (wave == 0) {
    const int row = tid >> 4, c = tid & 15;
    const bool on = c < a.C && r0 + row < a.rows;
    const float eps = 1e-8f;
    auto sum16 = [](float v) {
#pragma unroll
      for (int off = 8; off > 0; off >>= 1) v += __shfl_xor(v, off, 16);
      return v;
    };
    const float z = on ? Z2[row][c] : 0.f;
    const float yi = on ? a.y[(int64_t)(r0 + row) * a.C + c] : 0.f;
    float mx = 0.f;
    if (a.stable) {
      mx = on ? z : -INFINITY;
#pragma unroll
      for (int off = 8; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 16));
    }
    const float e = on ? expf(z - mx) : 0.f;
    const float total = sum16(e);
    const float pi = on ? e / total : 0.f;
    const float dpi = on ? (yi * a.neg_inv_rows) / (pi + eps) : 0.f;
    const float term = sum16(on ? yi * logf(pi + eps) : 0.f);
    const float dot = sum16(pi * dpi);
    if (on) a.p[(int64_t)(r0 + row) * a.C + c] = pi;
    if (c < a.C) Z2[row][c] = on ? pi * dpi - pi * dot : 0.f;   // dz2 (zeros for rows past the batch)
    if (c == 0 && r0 + row < a.rows) a.row_loss[r0 + row] = term;
  }
  __syncthreads();
  // ---- dh = dz2 W2^T, dz1 = act'(h) dh; dz1 leaves in fragment order (zeros outside the matrix)
  if (tid < RB * MH) {
    const int row = tid & 3, j = tid >> 2;
    float d = 0.f;
    if (j < a.H && r0 + row < a.rows) {
      float s = 0.f;
#pragma unroll 4
      for (int c = 0; c < a.C; ++c) s += Z2[row][c] * W2s[j * a.C + c];
      d = act_bwd1(a.act1, Hs[row][j], s, a.act1_param);
    }
    Ds[row][j] = d;
    a.dz1f[(((int64_t)(blk >> 2) * 4 + (j >> 4)) * 64 + (blk & 3) * 16 + (j & 15)) * 4 + row] = d;
  }
  __syncthreads();
  // ---- these rows' terms of dW2 = h^T dz2, db1 = column sums of dz1, db2 = column sums of dz2
  float* part = a.part + (int64_t)blk * (a.H * a.C + a.H + a.C);
  for (int e = tid; e < a.H * a.C + a.H + a.C; e += T) {
    float s = 0.f;
    if (e < a.H * a.C) {
      const int j = e / a.C, c = e - j * a.C;
#pragma unroll
      for (int row = 0; row < RB; ++row) s += Hs[row][j] * Z2[row][c];
    } else if (e < a.H * a.C + a.H) {
      const int j = e - a.H * a.C;
#pragma unroll
      for (int row = 0; row < RB; ++row) s += Ds[row][j];
    } else {
      const int c = e - a.H * a.C - a.H;
#pragma unroll
      for (int row = 0; row < RB; ++row) s += Z2[row][c];
    }
    part[e] = s;
  }
}

// STEPS_: k-blocks per wavefront, at least the row count's eighth
template <int STEPS_>
__global__ __launch_bounds__(T) void mlp2_weights_kernel(Mlp2Args a, int nblk, int nslab, int ncol) {
  __shared__ __attribute__((aligned(16))) float sums[WAVES * 64 * 4];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  Parameter par;
  if ((int)blockIdx.x >= nslab * ncol) {
    // sums of the row blocks' partial dW2 / db1 / db2: thread q of an output adds row blocks q, q + 16, ..., all requested at once
    constexpr int Q = T / PARTS, PER = MAX_ROWS / RB / Q;
    const int np = a.H * a.C + a.H + a.C, e = ((int)blockIdx.x - nslab * ncol) * PARTS + (tid & (PARTS - 1)), q = tid / PARTS;
    const int n = nblk * (MR / RB);
    float* at = nullptr;
    if (e < a.H * a.C) at = a.g_w2 + e;
    else if (e < a.H * a.C + a.H) at = a.g_b1 ? a.g_b1 + (e - a.H * a.C) : nullptr;
    else if (e < np) at = a.g_b2 ? a.g_b2 + (e - a.H * a.C - a.H) : nullptr;
    if (q == 0 && at && a.upd.kind >= 0) par.load(a.upd, at);
    float v[PER], s = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) v[i] = a.part[(int64_t)min(q + Q * i, n - 1) * np + min(e, np - 1)];
#pragma unroll
    for (int i = 0; i < PER; ++i) s += q + Q * i < n ? v[i] : 0.f;
    sums[tid] = s;
    __syncthreads();
    if (q == 0 && at) {
      s = 0.f;
#pragma unroll
      for (int i = 0; i < Q; ++i) s += sums[i * PARTS + tid];
      *at = s;
      if (a.upd.kind >= 0) par.update(a.upd, s);
    }
    return;
  }
  // ---- dW1[f0 .. f0 + 15, 16 cb .. 16 cb + 15] = x[:, f0 ..]^T dz1[:, 16 cb ..]: wavefront w takes k-blocks w, w + 8, ...
  const int slab = (int)blockIdx.x / ncol, cb = (int)blockIdx.x - slab * ncol, f0 = slab * 16;
  const int n16 = lane & 15, g = lane >> 4;
  const int f = f0 + (tid >> 4), col = cb * 16 + (tid & 15);  // the value that this thread finishes
  float* const at = tid < 256 && f < a.K && col < a.H ? a.g_w1 + (int64_t)f * a.H + col : nullptr;
  if (at && a.upd.kind >= 0) par.load(a.upd, at);
  const float* const xf = a.x + min(f0 + n16, a.K - 1);
  const f4v* const bsrc = (const f4v*)a.dz1f + cb * 64 + lane;
  float x[STEPS_][4];
  f4v d[STEPS_];
#pragma unroll
  for (int i = 0; i < STEPS_; ++i) {
    const int kb = min(wave + WAVES * i, nblk - 1);
#pragma unroll
    for (int j = 0; j < 4; ++j) x[i][j] = xf[(int64_t)min(16 * kb + 4 * g + j, a.rows - 1) * a.K];
    d[i] = bsrc[(int64_t)kb * 256];
  }
  f4v acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < STEPS_; ++i) {
    const int kb = wave + WAVES * i;
    if (kb < nblk) {
      if (kb == nblk - 1) {  // rows behind the batch
#pragma unroll
        for (int j = 0; j < 4; ++j) x[i][j] = 16 * kb + 4 * g + j < a.rows ? x[i][j] : 0.f;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i][j], d[i][j], acc, 0, 0, 0);
    }
  }
  *(f4v*)(sums + (wave * 64 + lane) * 4) = acc;  // element v of lane (n, g): feature f0 + 4 g + v, hidden unit 16 cb + n
  __syncthreads();
  if (at) {
    const int place = (((tid >> 6) & 3) * 16 + (tid & 15)) * 4 + ((tid >> 4) & 3);
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) s += sums[w * 256 + place];
    *at = s;
    if (a.upd.kind >= 0) par.update(a.upd, s);
  }
}

__global__ __launch_bounds__(256) void mlp2_loss_kernel(const float* __restrict__ row_loss, int rows, float* __restrict__ loss) {
  __shared__ float sm[4];
  float s = 0.f;
  for (int i = threadIdx.x; i < rows; i += 256) s += row_loss[i];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) *loss = (-(((sm[0] + sm[1]) + sm[2]) + sm[3])) / (float)rows;   // -Sum(y log(p + eps)) / B, Loss.scala:44-57
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

template <int N>
void launch_rows(sn_ctx* ctx, const Mlp2Args& a, int blocks, int n) {
  if constexpr (N > 1) {
    if (n < N) return launch_rows<N - 1>(ctx, a, blocks, n);
  }
  hipLaunchKernelGGL(mlp2_rows_kernel<N>, dim3((unsigned)blocks), dim3(T), 0, ctx->stream, a);
}

}  // namespace

// Shapes the fused pass takes: K a multiple of 4 up to 1024, H <= 64, C <= 16, up to 1792 rows; x in whole vectors.
// A training step here and by the general kernels: 8 -> 5 -> 1 at 16 rows 7.6 and 28.6 us, 36 -> 37 -> 16 at 33 rows 9.5 and 32.5,
// 32 -> 32 -> 10 at 1000 rows 11.0 and 41.8, 68 -> 64 -> 16 at 1000 rows 12.1 and 40.1.
bool mlp2_fused_ok(int rows_max, int K, int H, int C) {
  return K % 4 == 0 && K >= 4 && K <= 1024 && H >= 1 && H <= MH && C >= 1 && C <= MC && rows_max <= MAX_ROWS;
}
bool mlp2_input_ok(const float* x) { return aligned16(x); }
static int64_t fragment_elems(int rows) { return ceil_div(rows, MR) * 4 * 64 * 4; }
int64_t mlp2_scratch_elems(int rows_max, int H, int C) { return fragment_elems(rows_max) + ceil_div(rows_max, MR) * (MR / RB) * ((int64_t)H * C + H + C); }

int launch_mlp2_grad(sn_ctx* ctx, const float* x, const float* y, const float* w1, const float* b1, const float* w2, const float* b2, int rows,
                     int K, int H, int C, int act1, float act1_param, bool stable, float* h, float* z2, float* p, float* scratch,
                     float* row_loss, float* loss_dev, float* g_w1, float* g_b1, float* g_w2, float* g_b2,
                     const Mlp2Update* update) {
  SN_REQUIRE(rows > 0, "loss over an empty batch");
  SN_REQUIRE(mlp2_input_ok(x) && aligned16(scratch), "mlp2: x and the scratch buffer must be 16-byte aligned");
  Mlp2Args a{x, y, w1, b1, w2, b2, h, z2, p, scratch, row_loss, scratch + fragment_elems(rows), g_w1, g_b1, g_w2, g_b2,
             rows, K, H, C, act1, stable ? 1 : 0, act1_param, -(1.0f / (float)rows), update ? *update : Mlp2Update{}};
  const int nblk = (int)ceil_div(rows, MR), nslab = (int)ceil_div(K, 16);
  {
    LaunchScope scope(ctx, "mlp2_rows_forward_backward", rows, H, K);
    launch_rows<8>(ctx, a, nblk * (MR / RB), (int)ceil_div((ceil_div(K, WAVES) + 3) / 4 * 4, 16));
  }
  {
    LaunchScope scope(ctx, update ? "mlp2_weight_gradients_and_optimizer" : "mlp2_weight_gradients", K, H, rows);
    const int ncol = (int)ceil_div(H, 16);
    const dim3 grid((unsigned)(nslab * ncol + ceil_div((int64_t)H * C + H + C, PARTS)));
    if (nblk <= 4 * WAVES) hipLaunchKernelGGL(mlp2_weights_kernel<4>, grid, dim3(T), 0, ctx->stream, a, nblk, nslab, ncol);
    else if (nblk <= 8 * WAVES) hipLaunchKernelGGL(mlp2_weights_kernel<8>, grid, dim3(T), 0, ctx->stream, a, nblk, nslab, ncol);
    else hipLaunchKernelGGL(mlp2_weights_kernel<STEPS>, grid, dim3(T), 0, ctx->stream, a, nblk, nslab, ncol);
  }
  if (loss_dev) {
    LaunchScope scope(ctx, "loss_stage2");
    hipLaunchKernelGGL(mlp2_loss_kernel, dim3(1), dim3(256), 0, ctx->stream, (const float*)row_loss, rows, loss_dev);
  }
  SN_HIP(hipGetLastError());
  return SN_OK;
}

}  // namespace sn
