// Conv2D forward and input gradient with unit strides on bf16 matrix instructions (the split products of split_gemm.hpp: a float32
// value is the exact sum of three bf16 parts, six part products, float32 accumulate), with the FILTER resident in LDS and each
// wavefront taking the image's values apart for itself, once for all taps of a filter row.
//
//   C[M, N] = A[M, K] * B[K, N],  row m = a position (b, iy, ix) of the iteration space, k = (filter row r, tap q, channel):
//     A(m, k) = src[b, iy + oy + r*ty, ix + ox + q, channel]   (0 outside the source image)
//   forward:        src = x,  (oy, ox) = -padding, ty = +1,                      B(k, n) = w[r, q, channel, n]
//   input gradient: src = dy, oy = +pt, ox = pl - (kw - 1), ty = -1,             B(k, n) = w[r, kw - 1 - q, n, channel]
//
// K runs in units of 8 channels of one filter row, two to a step of v_mfma_f32_32x32x16_bf16 (half a wavefront each).  Channel
// counts that are no multiple of 8 end in a unit moved back to the last 8 channels, whose repeated channels meet zeros of the filter.
// A wavefront owns 32 consecutive positions x TN x 32 columns.  For a pair of units it loads the run of elements that its positions
// read in that filter row (32 and kw - 1 more for every row of positions it touches, at most 48; the next runs are in flight),
// takes them apart and puts them into LDS of its own as three planes; the operand of tap q is then one 16-byte read per lane
// and part at the position's element + q.  What lies outside the image is loaded from beyond the buffer's range and comes back as
// zeros; a table in LDS holds every unit's offset and its filter row's bit.  The filter is taken apart once per workgroup and lies
// in LDS in operand order, [step][32 columns][part][lane] 16 bytes.  8 wavefronts of a workgroup share it and walk their tiles
// without a barrier, a tile's first run being loaded, taken apart and read during the last products of the tile before.  A filter too
// large for LDS is walked in chunks, with barriers.  hi x hi products have accumulators of their own, so that the others'
// five times as many roundings happen at 2^-8 of the sum's size: root mean square error against float64 0.5e-7 to 1.5e-7 of the
// result where the float32 tiles have 2.9e-7 to 4.2e-7 and split_gemm.hpp 0.8e-7 to 2.8e-7 (8 to 64 channels, 8 to 128 filters).
//
// What bounds it (529000 positions x 64 x 288, 113 us = 173 TFLOP/s; 211 by conv_ring_kernels.hip): the matrix cores are busy 73 % of
// a tile's time at the clock that their power leaves (1.75 GHz), the rest is the issue of some 50 other instructions a step, 12
// of them LDS reads; taking every tap's values apart anew, straight from memory, it was 131, with the loads left to the compiler's
// order 170.  52900 x 64 x 288: 24.6 us (32.8), of which 5 are the filter's way into LDS.  121000 x 64 x 288 38 (58), 169000 x 32 x
// 576 59 (73), 409948 x 15 x 522 171 (327), 458643 x 8 x 252 62 (144).  An input gradient reads the filter's channels as vectors of four:
// value by value, every lane in a cache line of its own, taking the filter apart was as long as the products where it is walked in
// two chunks (204800 x 64 x 576 175 us, 120 now; 137 to 157 by conv_ring_kernels.hip.  102400 x 64 x 360 69, 47; 63 by split_conv.hip).
// Tiles beyond the ends of the range wait for memory: 32 channels are requested at a time.  One image in twenty of gradients below
// 2^-110 (a saturated softmax's) takes 40000 x 64 x 576 from 36 to 98 us (241 eight channels at a time, value by value; the ring kernel's
// float32 products 42 at any values), 64800 x 13 x 360 from 21 to 47 (81), all images 169000 x 32 x 576 from 55 to 189 (401); a single such
// weight, for which every tile's values are looked at again, 169000 x 64 x 288 from 49 to 65.
#include "split_launch.hpp"

#include "conv_resident_rules.hpp"

namespace sn {
namespace {

typedef uint32_t u4v __attribute__((ext_vector_type(4)));

constexpr uint32_t OOB = 0x80000000u;  // beyond any operand (tensors are checked to be < 2 GiB)

struct ResidentArgs {
  const float* src;
  uint32_t src_bytes, out_bytes;
  int M, ih, iw;           // iteration space: rows m = (b, iy, ix)
  FastDiv by_iw, by_ih, by_run;  // by_run: iw + KW - 1
  int oy, ty;              // image row of filter row r: iy + oy + r * ty
  int ox;                  // image column of the first value of a run
  int H, W, C;             // source image
  int kh;
  const float* w;
  uint32_t w_bytes;
  int w_tap, w_c, w_n;     // element (tap, channel, n) of the filter at tap * w_tap + channel * w_c + n * w_n
  int N;
  int units_per_row, units, pairs, chunk;  // pairs of units; of which LDS holds `chunk` at a time
  FastDiv by_units;        // units_per_row
  int tiles;               // of 32 positions
  int blocks_n, per_block; // column blocks, and workgroups of each
  Epilogue ep;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ f4v load16(__amdgpu_buffer_rsrc_t rs, uint32_t off) {
  return __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off, 0, 0));
}

// WVK = 2: two wavefronts share 32 positions and walk half of K each (few positions, long reductions: twice the workgroups, and still two
// wavefronts a SIMD); the second hands its sums over through LDS at the end.  (32512 x 32 x 864 24.1 us for 29.4.)
// DX: the input gradient, whose runs meet a filter row's taps from the last to the first.
template <int TN, int KW, int WVK, bool DX>
__global__ __launch_bounds__(512) void conv_resident_kernel(ResidentArgs a) {
  constexpr int T = 512, TILES = 8 / WVK, STEP = TN * 3 * 1024;  // tiles of a workgroup; bytes of a step of the filter
  constexpr int LOADS = RESIDENT_ELEMENTS / 16, PLANE = RESIDENT_ELEMENTS * 32;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  __shared__ int filter_top, filter_lossy;
  // [unit]: byte offset from an element's first value, bit of the filter row (0: no unit); more pairs are fetched than walked
  uint2* const table = reinterpret_cast<uint2*>(lds);
  char* const runs = lds + resident_table_bytes(a.pairs);
  char* const filter = runs + 8 * RESIDENT_RUN_BYTES;

  const int per_xcd = (int)gridDim.x >> 3, index = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
  if (index >= a.blocks_n * a.per_block) return;  // (the grid is rounded up to whole XCDs)
  const int block_n = index / a.per_block, share = index - block_n * a.per_block;
  const int n0 = block_n * TN * 32;
  // a contiguous run of tiles is this workgroup's, and every TILES-th of them a wavefront's
  const int tile_begin = (int)((int64_t)a.tiles * share / a.per_block), tile_end = (int)((int64_t)a.tiles * (share + 1) / a.per_block);

  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, lhi = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wk = wave % WVK, wtile = wave / WVK;
  const __amdgpu_buffer_rsrc_t rs = make_rsrc(a.src, a.src_bytes), rw = make_rsrc(a.w, a.w_bytes);

  if (tid == 0) filter_top = filter_lossy = 0;
  auto place_of = [&](int u, int& r, int& c8) {
    r = (int)div_by((uint32_t)u, a.by_units);
    c8 = u - r * a.units_per_row;
  };
  for (int u = tid; u < resident_table_bytes(a.pairs) / 8; u += T) {
    int r, c8;
    place_of(u, r, c8);
    const int c = min(8 * c8, a.C - 8);
    table[u] = u < a.units ? make_uint2((uint32_t)(r * a.ty * a.W * a.C + c) * 4u, 1u << r) : make_uint2(0u, 0u);
  }
  __syncthreads();

  float top = 0.f;               // the filter's largest magnitude, its smallest magnitude_key
  uint32_t least_b = 0xffffffffu;
  auto stage = [&](int pair0, int pair_n) {  // pairs [pair0, pair0 + pair_n) of the filter go to LDS
    // a wavefront takes 64 operands of eight values at a time: 64 columns of a unit (TN = 2), 32 of both units of a pair
    const int blocks = pair_n * KW * TN, n = n0 + (TN == 1 ? l32 : lane);
    constexpr int AHEAD = 5;  // blocks in flight
    for (int b0 = wave; b0 < blocks; b0 += 8 * AHEAD) {
      float v[AHEAD][8];
      int skip[AHEAD];
#pragma unroll
      for (int e = 0; e < AHEAD; ++e) {
        const int block = min(b0 + 8 * e, blocks - 1), step = block / TN, pair = step / KW, q = step - pair * KW;
        const int u = 2 * (pair0 + pair) + (TN == 1 ? lhi : block % TN);
        int r, c8;
        place_of(u, r, c8);
        const int tap = r * KW + (DX ? KW - 1 - q : q), c = min(8 * c8, a.C - 8);
        const bool in = u < a.units;
        skip[e] = in && n < a.N ? 8 * c8 - c : 8;  // channels that the unit before has
        const int column = min(n, a.N - 1) * a.w_n;
        if constexpr (DX) {  // (a column's channels lie side by side, the columns themselves a row of filters apart)
          const uint32_t from = (uint32_t)((in ? tap * a.w_tap + c : 0) + column) * 4u;
          const f4v first = load16(rw, from), second = load16(rw, from + 16u);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            v[e][j] = first[j];
            v[e][4 + j] = second[j];
          }
        } else {
          const float* from = a.w + (in ? tap * a.w_tap + c * a.w_c : 0) + column;
#pragma unroll
          for (int j = 0; j < 8; ++j) v[e][j] = from[j * a.w_c];
        }
      }
#pragma unroll
      for (int e = 0; e < AHEAD; ++e) {
        const int block = b0 + 8 * e;
        if (block >= blocks) break;
        u4v q[3];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float l = 2 * j >= skip[e] ? v[e][2 * j] : 0.f, r = 2 * j + 1 >= skip[e] ? v[e][2 * j + 1] : 0.f;
          top = max_magnitude(top, l, r);
          least_b = min(min(least_b, magnitude_key(l)), magnitude_key(r));
          uint32_t p[3];
          split_pair<3>(l, r, p);
#pragma unroll
          for (int k = 0; k < 3; ++k) q[k][j] = p[k];
        }
        char* to = filter + block / TN * STEP + (TN == 1 ? lane * 16 : lhi * 3072 + (l32 + 32 * (block % TN)) * 16);
#pragma unroll
        for (int k = 0; k < 3; ++k) *(u4v*)(to + k * 1024) = q[k];
      }
    }
  };
  auto note_filter = [&]() {  // (once a wavefront: LDS takes atomics on one word lane by lane, 512 of them were 3 us)
    float most = top;
    for (int o = 32; o > 0; o >>= 1) most = fmaxf(most, __shfl_xor(most, o));
    if (lane == 0) atomicMax(&filter_top, __float_as_int(most));
    if (__any(least_b < LEAST_WHOLE) && lane == 0) filter_lossy = 1;
  };
  const bool resident = a.chunk == a.pairs;

  // A tile's 32 positions lie in `segments` rows; KW - 1 elements follow the last position of each.  Element j's four neighbouring lanes
  // load the 64 bytes of a pair of units (or 32 of each of two places): where they begin, and which filter rows lie inside the image.
  uint32_t base[LOADS], inside[LOADS];
  auto locate = [&](int tile) {
    const uint32_t m0 = (uint32_t)min(tile * 32, a.M - 1), row0 = div_by(m0, a.by_iw);
    const int ix0 = (int)(m0 - row0 * (uint32_t)a.iw), first = a.iw - ix0 + KW - 1;  // elements of the first row
    const int elements = tile < tile_end ? 32 + (KW - 1) * ((int)div_by((uint32_t)(ix0 + 31), a.by_iw) + 1) : 0;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int j = 16 * i + (lane >> 2);
      uint32_t s = 0;
      int x = ix0 + j;
      if (j >= first) {
        s = 1u + div_by((uint32_t)(j - first), a.by_run);
        x = j - first - (int)(s - 1u) * (a.iw + KW - 1);
      }
      const uint32_t row = row0 + s, b = div_by(row, a.by_ih);
      const int y0 = (int)(row - b * (uint32_t)a.ih) + a.oy;
      x += a.ox;
      base[i] = (uint32_t)((((int)b * a.H + y0) * a.W + x) * a.C) * 4u + (uint32_t)(lane & 1) * 16u;
      uint32_t in = 0;
      for (int r = 0; r < a.kh; ++r) in |= (unsigned)(y0 + r * a.ty) < (unsigned)a.H ? 1u << r : 0u;
      inside[i] = j < elements && (unsigned)x < (unsigned)a.W && (int)row * a.iw < a.M ? in : 0u;
    }
  };
  auto entry = [&](int pair) { return table[2 * pair + ((lane >> 1) & 1)]; };
  auto fetch = [&](const uint2& e, f4v (&v)[LOADS]) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const uint32_t off = base[i] + e.x;
      v[i] = load16(rs, (inside[i] & e.y) ? off : OOB);
    }
  };
  f4v image[2][LOADS];  // the image, two pairs in flight
  // this wavefront's share of a chunk's pairs
  auto first_of = [&](int c0, int chunk) { return c0 + chunk * wk / WVK; };
  auto last_of = [&](int c0, int chunk) { return c0 + chunk * (wk + 1) / WVK; };
  // The pair requested next: they follow each other through the chunks, and on into the next tile.
  int next_tile = tile_begin + wtile, next_c0 = 0, next_pair = first_of(0, min(a.chunk, a.pairs)), next_last = last_of(0, min(a.chunk, a.pairs));
  auto advance = [&]() {
    if (++next_pair < next_last) return;
    next_c0 += a.chunk;
    if (next_c0 >= a.pairs) {
      next_c0 = 0;
      next_tile += TILES;
      locate(next_tile);
    }
    const int chunk = min(a.chunk, a.pairs - next_c0);
    next_pair = first_of(next_c0, chunk);
    next_last = last_of(next_c0, chunk);
  };
  // The elements go through LDS, this wavefront's own, as three planes [element][2 units][8 channels]: the operand of 32 positions and
  // tap q is 1 KiB in a row but for the gaps between segments.  LDS serves a wavefront in order: a pair's elements are written
  // behind the last read of the pair before.
  char* const run = runs + wave * RESIDENT_RUN_BYTES;
  uint32_t run_at = 0;  // this lane's part of the operand of tap 0
  auto find_run = [&](int tile) {
    const uint32_t m0 = (uint32_t)min(tile * 32, a.M - 1), ix = m0 - div_by(m0, a.by_iw) * (uint32_t)a.iw + (uint32_t)l32;
    run_at = ((uint32_t)l32 + (KW - 1) * div_by(ix, a.by_iw)) * 32u + (uint32_t)lhi * 16u;
  };
  uint32_t least = 0xffffffffu;
  auto take_apart = [&](const f4v& v, u2v (&planes)[3]) {
    least = min(min(least, magnitude_key(v[0])), magnitude_key(v[1]));
    least = min(min(least, magnitude_key(v[2])), magnitude_key(v[3]));
    uint32_t l[3], r[3];
    split_pair<3>(v[0], v[1], l);
    split_pair<3>(v[2], v[3], r);
#pragma unroll
    for (int p = 0; p < 3; ++p) planes[p] = u2v{l[p], r[p]};
  };
  auto write_run = [&](const u2v (&planes)[LOADS][3]) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
#pragma unroll
      for (int p = 0; p < 3; ++p) *(u2v*)(run + p * PLANE + i * 512 + lane * 8) = planes[i][p];
  };
  auto read_run = [&](int q, uint32_t run_at, bf16x8 (&af)[3]) {
#pragma unroll
    for (int p = 0; p < 3; ++p) af[p] = *(const bf16x8*)(run + p * PLANE + q * 32 + run_at);
  };
  auto read_filter = [&](const char* at, bf16x8 (&bf)[TN][3]) {  // at: this lane's 16 bytes of the step's first operand
#pragma unroll
    for (int n = 0; n < TN; ++n)
#pragma unroll
      for (int p = 0; p < 3; ++p) bf[n][p] = *(const bf16x8*)(at + n * 3072 + p * 1024);
  };
  // byte offset of a position's first channel at row r and value q of its run, OOB outside the image
  auto value_at = [&](int m, int r, int q) {
    const uint32_t mm = (uint32_t)min(m, a.M - 1), row = div_by(mm, a.by_iw), b = div_by(row, a.by_ih);
    const int y = (int)(row - b * (uint32_t)a.ih) + a.oy + r * a.ty, x = (int)(mm - row * (uint32_t)a.iw) + a.ox + q;
    return (unsigned)y < (unsigned)a.H && (unsigned)x < (unsigned)a.W ? (uint32_t)((((int)b * a.H + y) * a.W + x) * a.C) * 4u : OOB;
  };

  // value v of lane l of a tile: column l % 32, row 8 * (v / 4) + 4 * (l / 32) + v % 4.  Rows and columns beyond the result are
  // stores with an offset beyond its range, which are dropped.
  const __amdgpu_buffer_rsrc_t out = make_rsrc(a.ep.out, a.out_bytes);
  float bias[TN];
  uint32_t column[TN];
#pragma unroll
  for (int n = 0; n < TN; ++n) {
    const int col = n0 + n * 32 + l32;
    bias[n] = a.ep.bias ? a.ep.bias[min(col, a.N - 1)] : 0.f;
    column[n] = col < a.N ? (uint32_t)col * 4u : OOB;
  }
  auto store = [&](f16v (&acc)[TN], int m0) {
    const uint32_t row = (uint32_t)(m0 + 4 * lhi) * (uint32_t)a.N * 4u;
#pragma unroll
    for (int n = 0; n < TN; ++n) {
      if (a.ep.bias) {
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[n][v] += bias[n];
      }
      const uint32_t at = column[n] == OOB ? OOB : row + column[n];
      float x[16];
#pragma unroll
      for (int v = 0; v < 16; ++v) x[v] = acc[n][v];
      ep_act_block<16>(a.ep.act, x, a.ep.act_param);
#pragma unroll
      for (int v = 0; v < 16; ++v)
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x[v]), out, (int)(at + (uint32_t)(((v >> 2) * 8 + (v & 3)) * a.N * 4)), 0, 0);
    }
  };

  locate(next_tile);
  fetch(entry(next_pair), image[0]);
  advance();
  fetch(entry(next_pair), image[1]);
  advance();
  if (resident) {
    stage(0, a.pairs);
    note_filter();
    __syncthreads();
  }
  bf16x8 af[3], bf[TN][3];
  u2v planes[LOADS][3];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) take_apart(image[0][i], planes[i]);
  write_run(planes);
  fetch(entry(next_pair), image[0]);
  advance();
  find_run(tile_begin + wtile);
  read_run(0, run_at, af);
  if (resident) read_filter(filter + first_of(0, a.pairs) * KW * STEP + lane * 16, bf);
  // (all wavefronts go through the same chunks and hand-overs: a tile beyond the workgroup's last is one of zeros, whose stores are dropped)
  const int rounds_end = resident && WVK == 1 ? tile_end : tile_begin + (tile_end - tile_begin + TILES - 1) / TILES * TILES;
  for (int tile = tile_begin + wtile; tile < rounds_end; tile += TILES) {
    const int m0 = tile < tile_end ? tile * 32 : a.tiles * 32;
    f16v acc[TN], low[TN];  // sums of the hi x hi products, and of the others
#pragma unroll
    for (int n = 0; n < TN; ++n)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[n][v] = low[n][v] = 0.f;
    uint32_t least_now = 0xffffffffu;
    auto multiply = [&](const bf16x8 (&af)[3], const bf16x8 (&bf)[TN][3]) {
      // small terms first; consecutive instructions go to different accumulators
#pragma unroll
      for (int s = 2; s >= 0; --s)
#pragma unroll
        for (int p = 0; p <= s; ++p)
#pragma unroll
          for (int n = 0; n < TN; ++n) {
            f16v& to = s ? low[n] : acc[n];
            to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[p], bf[n][s - p], to, 0, 0, 0);
          }
    };
    for (int c0 = 0; c0 < a.pairs; c0 += a.chunk) {
      const int chunk = min(a.chunk, a.pairs - c0);
      if (!resident) {
        __syncthreads();  // (the chunk before has been read)
        stage(c0, chunk);
        if (tile == tile_begin + wtile) note_filter();
        __syncthreads();
      }
      const int from = first_of(c0, chunk), to = last_of(c0, chunk);
      const char* const first_step = filter + (from - c0) * KW * STEP + lane * 16;
      const char* at = first_step;
      if (!resident) read_filter(at, bf);
      // A pair: its KW taps multiply what the tap before has read.  Meanwhile the next pair's elements are taken apart, written behind
      // the last tap's reads, and those of the pair three further on requested; a tile's last pair does so for the next tile.
      auto turn = [&](int pair, f4v (&next)[LOADS]) {
        const bool last = pair == to - 1 && c0 + chunk == a.pairs;
        const uint2 e = entry(next_pair);
        const uint32_t run_at_now = run_at;
        if (last) {
          least_now = least;
          least = 0xffffffffu;
          find_run(tile + TILES);
        }
#pragma unroll
        for (int q = 0; q < KW; ++q) {
          bf16x8 an[3], bn[TN][3];
          at += STEP;
          if (q == KW - 1 && last && resident) at = first_step;
          if (q < KW - 1) {
            read_run(q + 1, run_at_now, an);
            read_filter(at, bn);
#pragma unroll
            for (int i = 0; i < LOADS; ++i)
              if (i * (KW - 1) / LOADS == q) take_apart(next[i], planes[i]);
          } else {
            write_run(planes);
            read_filter(at, bn);
            read_run(0, run_at, an);
            fetch(e, next);
          }
          multiply(af, bf);
#pragma unroll
          for (int p = 0; p < 3; ++p) af[p] = an[p];
#pragma unroll
          for (int n = 0; n < TN; ++n)
#pragma unroll
            for (int p = 0; p < 3; ++p) bf[n][p] = bn[n][p];
          // the order of issue: a matrix instruction at a time with what hides behind it
          if (q == KW - 1) __builtin_amdgcn_sched_group_barrier(0x200, 3 * LOADS, 0);
#pragma unroll
          for (int i = 0; i < 6 * TN; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, TN == 1 ? 2 : 1, 0);
            if (q == KW - 1 && i < LOADS) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, TN == 1 ? 10 : 5, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        advance();
      };
      int pair = from;
      __builtin_amdgcn_s_setprio(1);
#pragma unroll 1
      for (; pair + 1 < to; pair += 2) {
        turn(pair, image[1]);
        turn(pair + 1, image[0]);
      }
      if (pair < to) {
        turn(pair, image[1]);
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
          const f4v other = image[0][i];
          image[0][i] = image[1][i];
          image[1][i] = other;
        }
      }
      __builtin_amdgcn_s_setprio(0);
    }
#pragma unroll
    for (int n = 0; n < TN; ++n) acc[n] += low[n];
    bool lossy = (WVK == 1 ? least_now : min(least_now, least)) < LEAST_WHOLE;  // (half of a small last chunk may be empty)
    if constexpr (WVK == 2) {  // (one tile a pair of wavefronts: the filter is not read again)
      __syncthreads();
      float* ex = reinterpret_cast<float*>(filter) + wtile * (TN * 16 * 64 + 64) + lane;
      if (wk == 1) {
#pragma unroll
        for (int n = 0; n < TN; ++n)
#pragma unroll
          for (int v = 0; v < 16; ++v) ex[(n * 16 + v) * 64] = acc[n][v];
        ex[TN * 16 * 64] = lossy ? 1.f : 0.f;
      }
      __syncthreads();
      if (wk == 1) continue;
#pragma unroll
      for (int n = 0; n < TN; ++n)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[n][v] += ex[(n * 16 + v) * 64];
      lossy = lossy || ex[TN * 16 * 64] != 0.f;
    }

    // The ends of the range (split_gemm.hpp): a part or a part product beyond it leaves an Inf or a NaN behind, for good; values
    // below 2^-110 lose bits that a small sum would show.  Either way the tile is multiplied in float32.
    float rest = 0.f;
#pragma unroll
    for (int n = 0; n < TN; ++n)
#pragma unroll
      for (int v = 0; v < 16; ++v) rest = fmaf(acc[n][v], 0.f, rest);
    if (__any(rest != 0.f || lossy || filter_lossy)) {
      bool again = __any(rest != 0.f);
      if (!again) {
        // (of every value that the rows of the tile's positions can meet)
        float largest = 0.f;
        for (int r = 0; r < a.kh; ++r)
          for (int q = 0; q < KW; ++q) {
            const uint32_t from = value_at(m0 + l32, r, q);
#pragma unroll 1
            for (int c0 = 4 * lhi; c0 < a.C; c0 += 32) {
              f4v v[4];
#pragma unroll
              for (int i = 0; i < 4; ++i) v[i] = load16(rs, from == OOB ? OOB : from + 4u * (uint32_t)min(c0 + 8 * i, a.C - 4));
#pragma unroll
              for (int i = 0; i < 4; ++i) largest = max_magnitude(max_magnitude(largest, v[i][0], v[i][1]), v[i][2], v[i][3]);
            }
          }
        for (int o = 32; o > 0; o >>= 1) largest = fmaxf(largest, __shfl_xor(largest, o));
        const float limit = (float)(a.units * 8 * KW) * LOSSLESS_SUM * (largest + __int_as_float(filter_top));
        bool small = false;
#pragma unroll
        for (int n = 0; n < TN; ++n)
#pragma unroll
          for (int v = 0; v < 16; ++v)
            if (fabsf(acc[n][v]) < limit && m0 + lhi * 4 + (v >> 2) * 8 + (v & 3) < a.M && n0 + n * 32 + l32 < a.N) small = true;
        again = __any(small);
      }
      if (again) {
#pragma unroll
        for (int n = 0; n < TN; ++n)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[n][v] = 0.f;
        for (int r = 0; r < a.kh; ++r)
          for (int q = 0; q < KW; ++q) {
            const int tap = r * KW + (DX ? KW - 1 - q : q);
            const uint32_t at = value_at(m0 + l32, r, q);
            // 32 channels requested together, as vectors where they lie side by side: four of a vector are one k of four instructions
#pragma unroll 1
            for (int c0 = 0; c0 < a.C; c0 += 32) {
              f4v v[4], f[4][TN];
              int skip[4];  // channels that the other half of the wavefront, or the vector before, has
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const int c = c0 + 8 * i + 4 * lhi, first = min(c, a.C - 4);
                skip[i] = c - first;
                v[i] = load16(rs, at == OOB ? OOB : at + 4u * (uint32_t)first);
#pragma unroll
                for (int n = 0; n < TN; ++n) {
                  const int from = tap * a.w_tap + first * a.w_c + min(n0 + n * 32 + l32, a.N - 1) * a.w_n;
                  if constexpr (DX) {
                    f[i][n] = load16(rw, (uint32_t)from * 4u);
                  } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) f[i][n][j] = a.w[from + j * a.w_c];
                  }
                }
              }
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                if (c0 + 8 * i >= a.C) break;
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                  for (int n = 0; n < TN; ++n)
                    acc[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(j < skip[i] ? 0.f : v[i][j], j < skip[i] ? 0.f : f[i][n][j], acc[n], 0, 0, 0);
              }
            }
          }
      }
    }
    store(acc, m0);
  }
}

template <int TN, int KW, int WVK, bool DX>
int launch_resident(sn_ctx* ctx, const char* name, ResidentArgs& a, const ResidentPlan& p) {
  auto kernel = conv_resident_kernel<TN, KW, WVK, DX>;
  SN_TRY(allow_dynamic_lds(ctx, reinterpret_cast<const void*>(kernel), RESIDENT_LDS));
  LaunchScope scope(ctx, name, a.M, a.N, a.kh * KW * a.C);
  hipLaunchKernelGGL(kernel, dim3((unsigned)(8 * ceil_div((int64_t)p.blocks_n * p.per_block, 8))), dim3(512), (size_t)p.lds, ctx->stream, a);
  SN_HIP(hipGetLastError());
  return SN_OK;
}

template <int KW, bool DX>
int launch_planned(sn_ctx* ctx, const char* name, ResidentArgs& a) {
  const ResidentPlan p = resident_plan(a.M, a.N, a.C, a.kh, KW, ctx->compute_units);
  a.units_per_row = p.units_per_row;
  a.units = p.units;
  a.pairs = p.pairs;
  a.chunk = p.chunk;
  a.tiles = p.tiles;
  a.blocks_n = p.blocks_n;
  a.per_block = p.per_block;
  a.by_iw = fast_div((uint32_t)a.iw);
  a.by_ih = fast_div((uint32_t)a.ih);
  a.by_run = fast_div((uint32_t)(a.iw + KW - 1));
  a.by_units = fast_div((uint32_t)a.units_per_row);
  a.out_bytes = (uint32_t)((int64_t)a.M * a.N * 4);
  if (p.wvk == 2) return p.tn == 1 ? launch_resident<1, KW, 2, DX>(ctx, name, a, p) : launch_resident<2, KW, 2, DX>(ctx, name, a, p);
  return p.tn == 1 ? launch_resident<1, KW, 1, DX>(ctx, name, a, p) : launch_resident<2, KW, 1, DX>(ctx, name, a, p);
}

}  // namespace

int launch_conv_resident_fwd(sn_ctx* ctx, const ConvGeom& g, const float* x, const float* w, const Epilogue& e) {
  ResidentArgs a{};
  a.src = x;
  a.src_bytes = (uint32_t)((int64_t)g.n * g.h * g.w * g.cin * 4);
  a.M = g.n * g.ho * g.wo; a.ih = g.ho; a.iw = g.wo;
  a.oy = -g.pt; a.ty = 1; a.ox = -g.pl;
  a.H = g.h; a.W = g.w; a.C = g.cin; a.kh = g.kh;
  a.w = w; a.w_bytes = (uint32_t)((int64_t)g.kh * g.kw * g.cin * g.cout * 4); a.w_tap = g.cin * g.cout; a.w_c = g.cout; a.w_n = 1;
  a.N = g.cout;
  a.ep = e;
  return g.kw == 3 ? launch_planned<3, false>(ctx, "conv2d_forward_resident", a) : launch_planned<5, false>(ctx, "conv2d_forward_resident", a);
}

int launch_conv_resident_dgrad(sn_ctx* ctx, const ConvGeom& g, const float* dy, const float* w, float* dx) {
  ResidentArgs a{};
  a.src = dy;
  a.src_bytes = (uint32_t)((int64_t)g.n * g.ho * g.wo * g.cout * 4);
  a.M = g.n * g.h * g.w; a.ih = g.h; a.iw = g.w;
  a.oy = g.pt; a.ty = -1; a.ox = g.pl - (g.kw - 1);
  a.H = g.ho; a.W = g.wo; a.C = g.cout; a.kh = g.kh;
  a.w = w; a.w_bytes = (uint32_t)((int64_t)g.kh * g.kw * g.cin * g.cout * 4); a.w_tap = g.cin * g.cout; a.w_c = 1; a.w_n = g.cout;
  a.N = g.cin;
  a.ep.out = dx;
  a.ep.ldo = g.cin;
  return g.kw == 3 ? launch_planned<3, true>(ctx, "conv2d_input_gradient_resident", a) : launch_planned<5, true>(ctx, "conv2d_input_gradient_resident", a);
}

}  // namespace sn
