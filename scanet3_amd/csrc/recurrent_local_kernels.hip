// Recurrent layers whose whole recurrence fits one CU: all time steps of a few batch rows in one workgroup.
//
// The input's share of every step, x_t Wk + b, is one product over all steps beforehand (split_recurrent.hip), and so is the
// gradient of the inputs afterwards.  What is left is serial: h_{t-1} Wr (backward: dz_{t+1} Wr^T) and the cell.  Here a
// workgroup owns 4 batch rows and ALL units, one wavefront per 16 of them, and keeps Wr in registers for the whole
// sequence; the state goes from step to step through LDS behind one barrier.  Nothing is handed from workgroup to workgroup,
// so no row waits for another, and any unit count, batch and alignment will do.
//
// Products are those of split_gemm.hpp: a float32 value is the exact sum of three bf16 parts, hi + mid + lo, and accumulation
// is float32.  A workgroup owns 4 batch rows (a CU's vector unit is busy with the cells of no more: five exp or tanh each; and a
// batch of 512 is still only 128 workgroups), which leaves 12 of a tile's 16 rows free: tile row 4 g + p holds part p of batch
// row g.  So v_mfma_f32_16x16x32_bf16 with one part of the weights multiplies it with all parts of the state, three of them
// give all nine part products (six would need six with a part per instruction, and three times the LDS reads), and the three
// sums of a cell (row g, unit c) lie in values 0 .. 2 of lane (c, g).  128 units x 512 weights take 384 KiB of the CU's
// 512 KiB of registers.
#include "split_gemm.hpp"

namespace sn {
namespace {

typedef uint32_t u4v __attribute__((ext_vector_type(4)));

constexpr int ROWS = 4;  // batch rows of a workgroup

__device__ __forceinline__ float sigmoidf_(float x) { return 1.0f / (1.0f + expf(-x)); }

// The ends of the range (split_gemm.hpp).  Up to LARGEST_USUAL no sum of 256 products nor any part of one overflows, and a nonzero
// value below 2^-110 is not the sum of three bf16 parts.  A workgroup that has met a value outside (in the weights, or in any
// state so far) multiplies in float32 from then on.  Its wavefronts have to agree on that at every step: values of the state a
// step reads raise the flag of that step's parity, which is written next two barriers later.
constexpr float LARGEST_USUAL = 0x1p47f;
struct Seen {
  float largest = 0.f;
  uint32_t least = LEAST_WHOLE;
  __device__ __forceinline__ void add(float a) {
    largest = fmaxf(largest, fabsf(a));
    least = min(least, magnitude_key(a));
  }
  __device__ __forceinline__ bool outside() const { return (int)(largest > LARGEST_USUAL) | (int)(least < LEAST_WHOLE); }
};

// Column u of [H, H] weights (TRANSPOSED: row u) in operand order: lane (column, g) holds k = 32 kb + 8 g .. + 7 of every kb,
// in three parts, zeros from H on.  Every load is made, from inside the tensor, and what lies outside is dropped after: loads
// under a condition come one at a time (128 of them were 90 us before the first step).
template <int KB, bool TRANSPOSED>
__device__ __forceinline__ void load_column(bf16x8 (&b)[KB][3], int g, const float* __restrict__ w, int u, int H, Seen& seen) {
  const uint32_t uc = (uint32_t)min(u, H - 1);
  float all[KB][8];
#pragma unroll
  for (int kb = 0; kb < KB; ++kb)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t k = (uint32_t)min(32 * kb + 8 * g + j, H - 1);
      all[kb][j] = w[TRANSPOSED ? uc * (uint32_t)H + k : k * (uint32_t)H + uc];
    }
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = 32 * kb + 8 * g + j < H && u < H ? all[kb][j] : 0.f;
    u4v q[3];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float l = x[2 * j], r = x[2 * j + 1];
      seen.add(l);
      seen.add(r);
      const uint32_t hi = pack_bf16(l, r);
      l -= __uint_as_float(hi << 16);
      r -= __uint_as_float(hi & 0xffff0000u);
      const uint32_t mid = pack_bf16(l, r);
      l -= __uint_as_float(mid << 16);
      r -= __uint_as_float(mid & 0xffff0000u);
      q[0][j] = hi;
      q[1][j] = mid;
      q[2][j] = pack_bf16(l, r);
    }
#pragma unroll
    for (int p = 0; p < 3; ++p) b[kb][p] = __builtin_bit_cast(bf16x8, q[p]);
  }
  __builtin_amdgcn_sched_barrier(0);  // (the next column's raw values do not join these in the registers)
}

// The state in LDS: row 4 r + p holds part p of batch row r (p = 3: zeros), 32 KB bf16 values; rows are an odd number of 16
// bytes apart, so the 16-byte reads of 16 rows meet all banks once.
template <int KB>
struct State {
  static constexpr int PITCH = 64 * KB + 16, BYTES = 16 * PITCH;
  // value k of batch row r
  static __device__ __forceinline__ void put(char* lds, int r, int k, float a) {
    char* at = lds + 4 * r * PITCH + 2 * k;
    const uint32_t hi = pack_bf16(a, 0.f);
    a -= __uint_as_float(hi << 16);
    const uint32_t mid = pack_bf16(a, 0.f);
    a -= __uint_as_float(mid << 16);
    *(uint16_t*)at = (uint16_t)hi;
    *(uint16_t*)(at + PITCH) = (uint16_t)mid;
    *(uint16_t*)(at + 2 * PITCH) = (uint16_t)pack_bf16(a, 0.f);
  }
};

// out[n] = this lane's cell of state x column block n, for N blocks that share the state (at: the lane's first chunk)
template <int KB, int N>
__device__ __forceinline__ void multiply_state(const char* at, const bf16x8 (&w)[N][KB][3], float (&out)[N]) {
  constexpr int CHAINS = N == 1 ? 3 : 1;  // (consecutive instructions go to different accumulators)
  f4v acc[N][CHAINS];
#pragma unroll
  for (int n = 0; n < N; ++n)
#pragma unroll
    for (int p = 0; p < CHAINS; ++p) acc[n][p] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const bf16x8 a = *(const bf16x8*)(at + 64 * kb);
#pragma unroll
    for (int p = 2; p >= 0; --p)
#pragma unroll
      for (int n = 0; n < N; ++n) acc[n][p % CHAINS] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w[n][kb][p], acc[n][p % CHAINS], 0, 0, 0);
  }
#pragma unroll
  for (int n = 0; n < N; ++n) {
    f4v s = acc[n][CHAINS - 1];
#pragma unroll
    for (int p = CHAINS - 2; p >= 0; --p) s += acc[n][p];
    out[n] = (s[2] + s[1]) + s[0];
  }
}

// LDS writes are visible, reads done; stores to memory stay in flight (no other lane reads them in this launch)
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// The same cell in float32: a row of the state x column u (TRANSPOSED: row u) of the weights in memory, k ascending.
template <bool TRANSPOSED>
__device__ __forceinline__ float multiply_float32(const float* state, const float* __restrict__ w, int u, int H) {
  const uint32_t uc = (uint32_t)min(u, H - 1);
  float s = 0.f;
#pragma unroll 4
  for (int k = 0; k < H; ++k) s = fmaf(state[k], w[TRANSPOSED ? uc * (uint32_t)H + (uint32_t)k : (uint32_t)k * (uint32_t)H + uc], s);
  return s;
}

// uniform base + a lane's byte offset of 32 bits: one register of address, not two per tensor
__device__ __forceinline__ const float& at_bytes(const float* base, uint32_t off) { return *(const float*)((const char*)base + off); }
__device__ __forceinline__ float& at_bytes(float* base, uint32_t off) { return *(float*)((char*)base + off); }

__device__ __forceinline__ void clear_lds(char* lds, int bytes) {
  for (int i = (int)threadIdx.x * 16; i < bytes; i += (int)blockDim.x * 16) *(u4v*)(lds + i) = u4v{0u, 0u, 0u, 0u};
}

// ---------------------------------------------------------------------------- LSTM forward
struct LocalFwdArgs {
  const float* c0;     // [rows, H] or null: zeros
  const float* h0;     // [rows, H] or null: zeros
  const float* wr[4];  // [H, H] forget, input, gate, output
  float* gates;        // T slices of 4 * slice floats: in x_t Wk + b of [rows, 4H], out the activated gates
  float* c;            // T slices
  float* h;            // T slices: h_t
  float* y_seq;        // [rows, T, H] or null: h_t once more
  int64_t slice;
  int rows, T, H;
};

template <int KB>
__global__ __launch_bounds__(512) void lstm_local_fwd_kernel(LocalFwdArgs a) {
  typedef State<KB> P;
  __shared__ __attribute__((aligned(16))) char lds[2 * P::BYTES];
  __shared__ float whole[ROWS][32 * KB];  // the state in float32, where it is needed
  __shared__ int outside[2];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c16 = lane & 15, g = lane >> 4;
  const int u = wave * 16 + c16, r = blockIdx.x * ROWS + g;
  const int H = a.H;
  clear_lds(lds, 2 * P::BYTES);
  if (threadIdx.x < 2) outside[threadIdx.x] = 0;
  Seen seen;
  bf16x8 w[4][KB][3];
#pragma unroll
  for (int q = 0; q < 4; ++q) load_column<KB, false>(w[q], g, a.wr[q], u, H, seen);
  __syncthreads();

  // this lane's cell; lanes without one read cell 0 and write nothing
  const bool live = u < H && r < a.rows;
  const uint32_t ci = live ? 4u * (uint32_t)(r * H + u) : 0u, zi = live ? 4u * (uint32_t)(r * 4 * H + u) : 0u;
  const uint32_t yi = live ? 4u * (uint32_t)(r * a.T * H + u) : 0u;
  float c = a.c0 ? at_bytes(a.c0, ci) : 0.f, z[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) z[q] = at_bytes(a.gates + q * H, zi);
  float h = a.h0 && live ? at_bytes(a.h0, ci) : 0.f;
  if (a.h0 && live) P::put(lds, g, u, h);
  seen.add(h);
  if (seen.outside()) outside[0] = outside[1] = 1;
  __syncthreads();
  const int at = c16 * P::PITCH + 16 * g;
  int float32 = 0;
  for (int t = 0; t < a.T; ++t) {
    const char* now = lds + (t & 1) * P::BYTES + at;
    char* next = lds + ((t + 1) & 1) * P::BYTES;
    float zn[4], s[4] = {0.f, 0.f, 0.f, 0.f};
    const float* zt = a.gates + (int64_t)min(t + 1, a.T - 1) * 4 * a.slice;  // the next step's inputs fly while this one is multiplied
#pragma unroll
    for (int q = 0; q < 4; ++q) zn[q] = at_bytes(zt + q * H, zi);
    if (t > 0 || a.h0) {
      const int met = outside[t & 1];
      multiply_state<KB, 4>(now, w, s);
      float32 |= __builtin_amdgcn_readfirstlane(met);
      if (float32) {
        if (live) whole[g][u] = h;
        lds_barrier();
#pragma unroll
        for (int q = 0; q < 4; ++q) s[q] = multiply_float32<false>(whole[g], a.wr[q], u, H);
      }
    }
    // c = c_prev * f + i * g ; h = o * tanh(c)   (layer/RNN.scala:336-337)
    const float f = sigmoidf_(s[0] + z[0]);
    const float in = sigmoidf_(s[1] + z[1]);
    const float gg = tanhf(s[2] + z[2]);
    const float o = sigmoidf_(s[3] + z[3]);
    c = c * f + in * gg;
    h = o * tanhf(c);
    if (live) {
      P::put(next, g, u, h);
      seen.add(h);
      float* gt = a.gates + (int64_t)t * 4 * a.slice;
      at_bytes(gt, zi) = f;
      at_bytes(gt + H, zi) = in;
      at_bytes(gt + 2 * H, zi) = gg;
      at_bytes(gt + 3 * H, zi) = o;
      at_bytes(a.c + (int64_t)t * a.slice, ci) = c;
      at_bytes(a.h + (int64_t)t * a.slice, ci) = h;
      if (a.y_seq) at_bytes(a.y_seq + (int64_t)t * H, yi) = h;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) z[q] = zn[q];
    if (seen.outside()) outside[(t + 1) & 1] = 1;
    lds_barrier();
  }
}

// ---------------------------------------------------------------------------- LSTM backward
struct LocalBwdArgs {
  const float* gates;    // T slices of 4 * slice floats, activated
  const float* c;        // T slices
  const float* c0;       // [rows, H] or null
  const float* dh_last;  // [rows, H] or null: gradient of the last step's output
  const float* dy_seq;   // [rows, T, H] or null: gradient of every step's output
  const float* wr[4];
  float* dz;             // T slices of 4 * slice floats
  int64_t slice;
  int rows, T, H;
};

// The state handed on is dz of the four gates, side by side; a wavefront's 16 columns are 16 units of dh.
template <int KB>
__global__ __launch_bounds__(512) void lstm_local_bwd_kernel(LocalBwdArgs a) {
  typedef State<KB> P;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  __shared__ float whole[4][ROWS][32 * KB];  // the state in float32, where it is needed
  __shared__ int outside[2];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c16 = lane & 15, g = lane >> 4;
  const int u = wave * 16 + c16, r = blockIdx.x * ROWS + g;
  const int H = a.H;
  clear_lds(lds, 2 * 4 * P::BYTES);
  if (threadIdx.x < 2) outside[threadIdx.x] = 0;
  Seen seen;
  bf16x8 w[4][1][KB][3];
#pragma unroll
  for (int q = 0; q < 4; ++q) load_column<KB, true>(w[q][0], g, a.wr[q], u, H, seen);

  const bool live = u < H && r < a.rows;
  const uint32_t ci = live ? 4u * (uint32_t)(r * H + u) : 0u, zi = live ? 4u * (uint32_t)(r * 4 * H + u) : 0u;
  const uint32_t yi = live ? 4u * (uint32_t)(r * a.T * H + u) : 0u;
  auto fetch = [&](int t, float (&gate)[4], float& c_prev, float& dy) {
#pragma unroll
    for (int q = 0; q < 4; ++q) gate[q] = at_bytes(a.gates + (int64_t)t * 4 * a.slice + q * H, zi);
    c_prev = t > 0 ? at_bytes(a.c + (int64_t)(t - 1) * a.slice, ci) : (a.c0 ? at_bytes(a.c0, ci) : 0.f);
    dy = a.dy_seq ? at_bytes(a.dy_seq + (int64_t)t * H, yi) : 0.f;
  };
  float c = at_bytes(a.c + (int64_t)(a.T - 1) * a.slice, ci), dc = 0.f, dh = a.dh_last ? at_bytes(a.dh_last, ci) : 0.f, gate[4], cp, dy;
  fetch(a.T - 1, gate, cp, dy);
  __syncthreads();
  if (seen.outside()) outside[0] = outside[1] = 1;  // (read after the next barrier)
  const int at = c16 * P::PITCH + 16 * g;
  int float32 = 0;
  for (int t = a.T - 1; t >= 0; --t) {
    char* buf = lds + (t & 1) * 4 * P::BYTES;
    float gn[4], cpn, dyn;
    fetch(max(t - 1, 0), gn, cpn, dyn);  // flies until the next step
    const float f = gate[0], in = gate[1], gg = gate[2], o = gate[3];
    const float tc = tanhf(c), d = a.dy_seq ? dh + dy : dh;
    dc = dc + (1.0f - tc * tc) * (d * o);
    const float dz[4] = {(f * (1.0f - f)) * (dc * cp), (in * (1.0f - in)) * (dc * gg), (1.0f - gg * gg) * (dc * in), (o * (1.0f - o)) * (d * tc)};
    dc = dc * f;
    if (live) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        at_bytes(a.dz + (int64_t)t * 4 * a.slice + q * H, zi) = dz[q];
        P::put(buf + q * P::BYTES, g, u, dz[q]);
        seen.add(dz[q]);
      }
    }
    if (seen.outside()) outside[t & 1] = 1;
    if (t == 0) break;
    lds_barrier();
    const int met = outside[t & 1];
    float s[4][1];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      multiply_state<KB, 1>(buf + q * P::BYTES + at, w[q], s[q]);
      if constexpr (KB > 3) __builtin_amdgcn_sched_barrier(0);  // (four gates' sums and state reads at once are more than the registers hold)
    }
    float32 |= __builtin_amdgcn_readfirstlane(met);
    if (float32) {
      if (live) {
#pragma unroll
        for (int q = 0; q < 4; ++q) whole[q][g][u] = dz[q];
      }
      lds_barrier();
#pragma unroll
      for (int q = 0; q < 4; ++q) s[q][0] = multiply_float32<true>(whole[q][g], a.wr[q], u, H);
    }
    dh = (s[0][0] + s[1][0]) + (s[2][0] + s[3][0]);
    c = cp;
    cp = cpn;
    dy = dyn;
#pragma unroll
    for (int q = 0; q < 4; ++q) gate[q] = gn[q];
  }
}

// ---------------------------------------------------------------------------- simple cell, both directions
// out_s = add_s + out_{s-1} W, out_{-1} = seed: forward r_t = x_t Wk + r_{t-1} Wr (layer/RNN.scala:189-196), backward
// dr_{t-1} = dout_{t-1} + dr_t Wr^T.
struct LocalMulArgs {
  const float* seed;          // [rows, H] or null: zeros
  const float* wr;            // [H, H]
  const float* add;           // or null; element (row, u) of step s at add + s * add_step + row * add_ld + u (may be `out` itself)
  int add_ld;
  int64_t add_step;
  float* out;                 // element (row, u) of step s at out + s * out_step + row * H + u
  int64_t out_step;
  int rows, steps, H;
};

// a wavefront owns UBW blocks of 16 units: one up to 128 units, two up to 256
template <int KB, int UBW, bool BACKWARD>
__global__ __launch_bounds__(512) void rnn_local_kernel(LocalMulArgs a) {
  typedef State<KB> P;
  __shared__ __attribute__((aligned(16))) char lds[2 * P::BYTES];
  __shared__ float whole[ROWS][32 * KB];  // the state in float32, where it is needed
  __shared__ int outside[2];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c16 = lane & 15, g = lane >> 4;
  const int u0 = wave * 16 * UBW + c16, r = blockIdx.x * ROWS + g;
  const int H = a.H;
  clear_lds(lds, 2 * P::BYTES);
  if (threadIdx.x < 2) outside[threadIdx.x] = 0;
  Seen seen;
  bf16x8 w[UBW][KB][3];
#pragma unroll
  for (int b = 0; b < UBW; ++b) load_column<KB, BACKWARD>(w[b], g, a.wr, u0 + 16 * b, H, seen);
  __syncthreads();

  bool live[UBW];
  uint32_t ai[UBW], oi[UBW];
  float add[UBW], state[UBW];
#pragma unroll
  for (int b = 0; b < UBW; ++b) {
    const int u = u0 + 16 * b;
    live[b] = u < H && r < a.rows;
    ai[b] = live[b] ? 4u * (uint32_t)(r * a.add_ld + u) : 0u;
    oi[b] = live[b] ? 4u * (uint32_t)(r * H + u) : 0u;
    add[b] = a.add ? at_bytes(a.add, ai[b]) : 0.f;
    state[b] = a.seed && live[b] ? at_bytes(a.seed, oi[b]) : 0.f;
    if (a.seed && live[b]) P::put(lds, g, u, state[b]);
    seen.add(state[b]);
  }
  if (seen.outside()) outside[0] = outside[1] = 1;
  __syncthreads();
  const int at = c16 * P::PITCH + 16 * g;
  int float32 = 0;
  for (int s = 0; s < a.steps; ++s) {
    const char* now = lds + (s & 1) * P::BYTES + at;
    char* next = lds + ((s + 1) & 1) * P::BYTES;
    float add_next[UBW], x[UBW] = {};
#pragma unroll
    for (int b = 0; b < UBW; ++b) add_next[b] = a.add ? at_bytes(a.add + (int64_t)min(s + 1, a.steps - 1) * a.add_step, ai[b]) : 0.f;
    if (s > 0 || a.seed) {
      const int met = outside[s & 1];
      multiply_state<KB, UBW>(now, w, x);
      float32 |= __builtin_amdgcn_readfirstlane(met);
      if (float32) {
#pragma unroll
        for (int b = 0; b < UBW; ++b)
          if (live[b]) whole[g][u0 + 16 * b] = state[b];
        lds_barrier();
#pragma unroll
        for (int b = 0; b < UBW; ++b) x[b] = multiply_float32<BACKWARD>(whole[g], a.wr, u0 + 16 * b, H);
      }
    }
#pragma unroll
    for (int b = 0; b < UBW; ++b) {
      if (a.add) x[b] += add[b];
      if (live[b]) {
        P::put(next, g, u0 + 16 * b, x[b]);
        seen.add(x[b]);
        at_bytes(a.out + (int64_t)s * a.out_step, oi[b]) = x[b];
      }
      add[b] = add_next[b];
      state[b] = x[b];
    }
    if (seen.outside()) outside[(s + 1) & 1] = 1;
    lds_barrier();
  }
}

template <int KB>
int launch_fwd(sn_ctx* ctx, const LocalFwdArgs& a) {
  hipLaunchKernelGGL((lstm_local_fwd_kernel<KB>), dim3((unsigned)ceil_div(a.rows, ROWS)), dim3((unsigned)ceil_div(a.H, 16) * 64), 0, ctx->stream, a);
  SN_HIP(hipGetLastError());
  return SN_OK;
}
template <int KB>
int launch_bwd(sn_ctx* ctx, const LocalBwdArgs& a) {
  constexpr int LDS = 2 * 4 * State<KB>::BYTES;
  static_assert(LDS <= 64 * 1024, "needs a raised limit");
  hipLaunchKernelGGL((lstm_local_bwd_kernel<KB>), dim3((unsigned)ceil_div(a.rows, ROWS)), dim3((unsigned)ceil_div(a.H, 16) * 64), LDS, ctx->stream, a);
  SN_HIP(hipGetLastError());
  return SN_OK;
}
template <int KB, int UBW, bool BACKWARD>
int launch_rnn(sn_ctx* ctx, const LocalMulArgs& a) {
  hipLaunchKernelGGL((rnn_local_kernel<KB, UBW, BACKWARD>), dim3((unsigned)ceil_div(a.rows, ROWS)), dim3((unsigned)ceil_div(a.H, 16 * UBW) * 64), 0,
                     ctx->stream, a);
  SN_HIP(hipGetLastError());
  return SN_OK;
}
template <bool BACKWARD>
int launch_rnn_blocks(sn_ctx* ctx, const LocalMulArgs& a) {
  switch (ceil_div(a.H, 32)) {
    case 1: return launch_rnn<1, 1, BACKWARD>(ctx, a);
    case 2: return launch_rnn<2, 1, BACKWARD>(ctx, a);
    case 3: return launch_rnn<3, 1, BACKWARD>(ctx, a);
    case 4: return launch_rnn<4, 1, BACKWARD>(ctx, a);
    case 5:
    case 6: return launch_rnn<6, 2, BACKWARD>(ctx, a);
    default: return launch_rnn<8, 2, BACKWARD>(ctx, a);
  }
}

}  // namespace

// 8 wavefronts x 16 units with 192 registers of weights each: an LSTM of 128 units, a simple cell of 256
bool recurrent_local_fits(int rows, int T, int F, int H, int gates) {
  return rows > 0 && T > 0 && H >= 1 && H <= (gates == 4 ? 128 : 256) && recurrent_products_fit(rows, T, F, H, gates);
}

int launch_lstm_local_fwd(sn_ctx* ctx, const float* x, int T, int F, const float* h0, const float* c0, int rows, int H, const LstmWeights& w,
                          float* gates, float* c, float* h, int64_t slice, float* y_seq) {
  SN_REQUIRE(recurrent_local_fits(rows, T, F, H, 4), "lstm_local_forward: rows=%d T=%d F=%d H=%d out of range", rows, T, F, H);
  SN_TRY(launch_recurrent_inputs(ctx, x, rows, T, F, H, w, 4, gates, 4 * slice));
  LocalFwdArgs a{c0, h0, {w.wr[0], w.wr[1], w.wr[2], w.wr[3]}, gates, c, h, y_seq, slice, rows, T, H};
  LaunchScope scope(ctx, "lstm_local_forward", rows * T, 4 * H, H);
  switch (ceil_div(H, 32)) {
    case 1: return launch_fwd<1>(ctx, a);
    case 2: return launch_fwd<2>(ctx, a);
    case 3: return launch_fwd<3>(ctx, a);
    default: return launch_fwd<4>(ctx, a);
  }
}

int launch_lstm_local_bwd(sn_ctx* ctx, const float* gates, const float* c, const float* c0, const float* dh_last, const float* dy_seq, int T,
                          int rows, int H, const LstmWeights& w, float* dz, int64_t slice) {
  SN_REQUIRE(rows > 0 && T > 0 && H >= 1 && H <= 128, "lstm_local_backward: rows=%d T=%d H=%d out of range", rows, T, H);
  LocalBwdArgs a{gates, c, c0, dh_last, dy_seq, {w.wr[0], w.wr[1], w.wr[2], w.wr[3]}, dz, slice, rows, T, H};
  LaunchScope scope(ctx, "lstm_local_backward", rows * (T - 1), H, 4 * H);
  switch (ceil_div(H, 32)) {
    case 1: return launch_bwd<1>(ctx, a);
    case 2: return launch_bwd<2>(ctx, a);
    case 3: return launch_bwd<3>(ctx, a);
    default: return launch_bwd<4>(ctx, a);
  }
}

int launch_rnn_local_fwd(sn_ctx* ctx, const float* x, int T, int F, bool first_valid, int rows, int H, const LstmWeights& w, float* r_slices,
                         int64_t slice) {
  SN_REQUIRE(recurrent_local_fits(rows, T, F, H, 1), "rnn_local_forward: rows=%d T=%d F=%d H=%d out of range", rows, T, F, H);
  SN_TRY(launch_recurrent_inputs(ctx, x, rows, T, F, H, w, 1, r_slices + slice, slice));
  LocalMulArgs a{first_valid ? r_slices : nullptr, w.wr[0], r_slices + slice, H, slice, r_slices + slice, slice, rows, T, H};
  LaunchScope scope(ctx, "rnn_local_forward", rows * T, H, H);
  return launch_rnn_blocks<false>(ctx, a);
}

int launch_rnn_local_bwd(sn_ctx* ctx, float* dr_slices, const float* dy_seq, int T, int rows, int H, const float* wr, int64_t slice) {
  SN_REQUIRE(rows > 0 && H >= 1 && H <= 256, "rnn_local_backward: rows=%d H=%d out of range", rows, H);
  if (T <= 1) return SN_OK;
  LocalMulArgs a{dr_slices + (T - 1) * slice, wr, dy_seq ? dy_seq + (int64_t)(T - 2) * H : nullptr, T * H, -(int64_t)H,
                 dr_slices + (T - 2) * slice, -slice, rows, T - 1, H};
  LaunchScope scope(ctx, "rnn_local_backward", rows * (T - 1), H, H);
  return launch_rnn_blocks<true>(ctx, a);
}

}  // namespace sn
