// Which convolutions conv_resident_kernels.hip takes, and how it divides them over workgroups (host only).
#pragma once
#include "common.hpp"

#include <algorithm>

namespace sn {

constexpr int RESIDENT_LDS = 160 * 1024 - 64;          // of a CU's 160 KiB (a few words are the kernel's own)
constexpr int RESIDENT_ELEMENTS = 48;                  // of an image row that the 32 positions of a tile read
constexpr int RESIDENT_RUN_BYTES = RESIDENT_ELEMENTS * 96;  // ... of a pair of units, as three planes

// 8 bytes for every unit, and for those that are requested but not multiplied
__host__ __device__ inline constexpr int resident_table_bytes(int pairs) { return (pairs + 4) * 16; }

struct ResidentPlan {
  int units_per_row = 0, units = 0;  // of 8 channels, of a filter row and of all
  int pairs = 0, chunk = 0;          // pairs of units, of which LDS holds `chunk` at a time
  int tn = 0, blocks_n = 0;          // tiles of 32 columns of a workgroup, column blocks
  int tiles = 0, wvk = 0;            // tiles of 32 positions, wavefronts that share one
  int per_block = 0, lds = 0;        // workgroups of a column block, bytes of LDS
};
inline ResidentPlan resident_plan(int64_t positions, int columns, int channels, int kh, int kw, int cu) {
  ResidentPlan p;
  p.units_per_row = (int)ceil_div(channels, 8);
  p.units = kh * p.units_per_row;
  p.pairs = (int)ceil_div(p.units, 2);
  const int column_tiles = (int)ceil_div(columns, 32);
  p.tn = column_tiles % 2 == 0 ? 2 : 1;
  p.blocks_n = column_tiles / p.tn;
  p.tiles = (int)ceil_div(positions, 32);
  // Two wavefronts on a tile where the chip takes all of them at once and the reduction is long enough to pay for handing the sums
  // over.  Microseconds of one / two at 30208 positions, columns x reduction: 8 x 72 11.4 / 13.0, 32 x 144 14.1 / 14.4, 32 x 216 13.9 / 14.4,
  // 64 x 192 17.1 / 16.4, 64 x 288 20.7 / 18.8, 32 x 288 17.3 / 15.9, 24 x 360 17.2 / 14.7, 64 x 576 31.4 / 26.4, 32 x 864 29.3 / 24.1;
  // five wide: 16 x 80 11.6 / 12.1, 32 x 160 13.4 / 14.9, 32 x 400 18.5 / 18.1, 10 x 500 20.7 / 16.4, 12 x 1000 28.9 / 23.8.
  p.wvk = ceil_div(p.tiles, 4) * p.blocks_n <= cu && p.pairs * kw * p.tn >= 18 ? 2 : 1;
  const int fixed = resident_table_bytes(p.pairs) + 8 * RESIDENT_RUN_BYTES, step = p.tn * 3072;
  const int most = ((RESIDENT_LDS - fixed) / step - 1) / kw;  // (a step more is read than multiplied)
  if (most < 1) return ResidentPlan{};  // the table and the runs leave no room for one pair of units: nothing to divide
  p.chunk = (int)ceil_div(p.pairs, ceil_div(p.pairs, most));
  const int groups = (int)ceil_div(p.tiles, 8 / p.wvk);  // as many workgroups as leave every wavefront a tile (two of them: one tile)
  p.per_block = p.wvk == 2 ? groups : std::min(groups, std::max(1, cu / p.blocks_n));
  p.lds = fixed + std::max((p.chunk * kw + 1) * step, p.wvk == 2 ? 4 * (p.tn * 1024 + 64) * 4 : 0);
  return p;
}

// 32-bit byte offsets, a bit per filter row, at least one whole unit of channels, and the rows that 32 positions lie in together
// with what the filter row reaches beyond their ends fit the elements.
inline bool resident_tensor_ok(const float* p, int64_t elems) { return (reinterpret_cast<uintptr_t>(p) & 3u) == 0 && elems * 4 < ((int64_t)1 << 31); }
inline bool resident_shape_ok(const ConvGeom& g, int64_t positions, int row, int columns, int channels, int cu) {
  if (!(positions >= 30000 && g.sh == 1 && g.sw == 1 && (g.kw == 3 || g.kw == 5) && g.kh <= 31 && channels >= 8 && channels <= 4096 && row >= 1 &&
        32 + (g.kw - 1) * ((row + 30) / row + 1) <= RESIDENT_ELEMENTS))
    return false;
  // A workgroup spends up to 5 us on taking the filter apart before the first product, so there have to be positions enough to
  // share it, and a filter of three or more chunks is taken apart again for every eight tiles.  The tiled kernels cover 128 positions a CU
  // in one round, 32768, and begin a second one behind that; up to there only reductions of nine steps and more come out ahead.
  // Microseconds, the split, ring or float32 kernels' and here, positions x columns x reduction: 12100 x 64 x 288 15.7 / 17.8, 25600 x 16 x
  // 72 12.1 / 14.8, 25600 x 32 x 576 20.2 / 24.0; 30208 x 16 x 48 9.4 / 10.2, 30208 x 32 x 96 12.2 / 13.2, 30208 x 16 x 144 13.6 / 12.6, 30208 x
  // 32 x 288 19.5 / 15.9, 30208 x 64 x 576 29.9 / 26.4, 32000 x 80 x 432 40.8 / 30.0; 33280 x 16 x 48 12.5 / 10.4, 33280 x 8 x 72 14.8 / 11.1,
  // 33280 x 64 x 192 19.5 / 16.8, 41472 x 9 x 72 23.3 / 13.1, 52900 x 64 x 288 32.8 / 24.6, 121000 x 64 x 288 58 / 38, 458643 x 8 x 252 144 / 62;
  // two chunks: 49000 x 128 x 576 81 / 65.  Five wide: 30208 x 8 x 200 14.8 / 14.7, 30208 x 32 x 800 37.9 / 23.8, 33280 x 16 x 80 14.9 / 11.5,
  // 53125 x 32 x 400 38.9 / 19.2, 53125 x 64 x 800 70 / 47, 125000 x 8 x 400 66 / 26, 312500 x 64 x 800 323 / 200.
  // Three chunks: 32000 x 48 x 720 45.0 / 45.8, twelve: 49000 x 64 x 1152 75 / 86, both with the filter read value by value (as vectors
  // 33024 x 48 x 720 50 / 39); they are left where they were.
  const ResidentPlan p = resident_plan(positions, columns, channels, g.kh, g.kw, cu);
  return p.chunk >= 1 && p.pairs <= 2 * p.chunk && (positions > 128 * cu || p.pairs * g.kw >= 9);
}
inline bool conv_resident_fwd_ok(const ConvGeom& g, const float* x, const float* w, const Epilogue& e, int cu) {
  return e.row_index < 0 && e.ldo == g.cout && resident_tensor_ok(x, (int64_t)g.n * g.h * g.w * g.cin) &&
         resident_tensor_ok(w, (int64_t)g.kh * g.kw * g.cin * g.cout) && resident_tensor_ok(e.out, (int64_t)g.n * g.ho * g.wo * g.cout) &&
         resident_shape_ok(g, (int64_t)g.n * g.ho * g.wo, g.wo, g.cout, g.cin, cu);
}
// The ring kernels take filter counts that are multiples of 32 and fill the chip up to 128 positions a CU (32512 x 64 x 320 20.1 / 22.1, 30208 x
// 64 x 192 16.1 / 16.5; 33280 x 64 x 320 25.1 / 23.9), onto 32 columns and fewer also well beyond (62500 x 32 x 576 32.8 / 32.1).
inline bool conv_resident_dgrad_ok(const ConvGeom& g, const float* dy, const float* w, const float* dx, int cu) {
  return resident_tensor_ok(dy, (int64_t)g.n * g.ho * g.wo * g.cout) && resident_tensor_ok(w, (int64_t)g.kh * g.kw * g.cin * g.cout) &&
         resident_tensor_ok(dx, (int64_t)g.n * g.h * g.w * g.cin) &&
         (g.cout % 32 != 0 || (int64_t)g.n * g.h * g.w > (g.cin > 32 ? 128 * cu : 79999)) && resident_shape_ok(g, (int64_t)g.n * g.h * g.w, g.w, g.cin, g.cout, cu);
}

}  // namespace sn
