// Which filter gradients conv_wgrad_split_kernels.hip takes, and how it divides them over workgroups (host only).
#pragma once
#include "common.hpp"

#include <algorithm>

namespace sn {

struct WgradSplitPlan {
  int tm = 0, tn = 0;              // tiles of 32 values of a run, of 32 filters, that a wavefront keeps
  int groups_m = 0, groups_n = 0;  // workgroups that a filter row's result is divided over
  int chunks = 0, parts = 0;       // of 16 positions; ranges of them
  float cost = 0.f;
  bool padded = false;
};
// Up to six tiles a wavefront (96 of its 256 registers).  Which division: what a workgroup's time comes to in cycles, its two
// wavefronts on a SIMD in turn - a chunk's 6 products a tile of 32 cycles, or taking tm + tn tiles apart where that is more - and 1000
// for each tile that the wavefronts add and write at the end.
inline WgradSplitPlan conv_wgrad_split_plan(const ConvGeom& g, int cu, int64_t ws_elems) {
  WgradSplitPlan p;
  const int L = g.kw * g.cin, tiles_m = (int)ceil_div(L, 32), tiles_n = (int)ceil_div(g.cout, 32);
  p.chunks = (int)ceil_div((int64_t)g.n * g.ho * g.wo, 16);
  const int64_t room = ws_elems / ((int64_t)g.kh * L * g.cout);
  p.padded = g.pt != 0 || g.pl != 0 || (g.ho - 1) * g.sh + g.kh > g.h || (g.wo - 1) * g.sw + g.kw > g.w;
  p.cost = 1e30f;
  for (int tm = 1; tm <= 3; ++tm)
    for (int tn = 1; tn <= 3; ++tn) {
      if (tm * tn > (tn == 3 ? 3 : 6)) continue;  // (2 x 3 holds three tiles of dy taken apart twice over and spills: at 28224 x 65 x 108 23 us for 19)
      const int gm = (int)ceil_div(tiles_m, tm), gn = (int)ceil_div(tiles_n, tn), groups = g.kh * gm * gn;
      const int parts = (int)std::min<int64_t>({(int64_t)std::max(1, cu / groups), (int64_t)p.chunks, room});
      if (parts < 1) continue;
      const float rounds = (float)ceil_div(groups * parts, cu), share = (float)ceil_div(p.chunks, 8 * parts);
      const float cost = rounds * (share * 2.f * std::max(192.f * (float)(tm * tn), 330.f * (float)(tm + tn)) + 1000.f * (float)(tm * tn));
      if (cost < p.cost) {
        p.cost = cost;
        p.tm = tm; p.tn = tn; p.groups_m = gm; p.groups_n = gn; p.parts = parts;
      }
    }
  return p;
}
// 32-bit byte offsets (a tile's values behind a run included), a bit for every row and column of the filter.  From 4096 positions:
// at 3136 x 128 x 576 both ways take 15.3 us, at 5760 x 8 x 144 this one 7.9 for 9.8, and below that nothing is left to gain.
// A filter row of a few values leaves most of its tile of 32 empty, once for every row, where the split products' tiles of 64 (32, if
// that is enough) hold several rows, each made up to whole vectors of four.  How much more is multiplied
// decides from half as much again on, unless the result is small enough (512 values) for the kernel of small outputs, which this one beats at
// any run.  Below 32768 positions launches and the sums at the end are most of the time, and either way is within two microseconds up to
// twice as much.  The kernels before / this one with the sums of the partial results, us, rows x columns x channels of the filter, number
// of filters, at 31104, 65124 and 250128 positions:
//   half as much again: 3 x 3 x 11, 64 24.3 / 23.1, 32.4 / 29.8, 70.6 / 63.9   3 x 3 x 12, 64 23.7 / 23.0, 31.4 / 29.3, 70.3 / 64.2
//     3 x 1 x 12, 64 18.5 / 18.5, 23.1 / 22.8, 45.5 / 46.8   6 x 1 x 20, 64 23.7 / 23.7, 30.6 / 33.2, 70.3 / 80.5 (its rows share tiles of 64 by twos)
//     tiles of 128 filters: 3 x 3 x 11, 100 31.2 / 30.0, 41.9 / 42.8, 94.6 / 110.4   3 x 1 x 12, 100 21.9 / 22.9, 29.3 / 32.8, 67.8 / 77.9
//   two thirds: 5 x 3 x 12, 64 28.4 / 28.2, 43.1 / 38.5, 88.2 / 95.7   three quarters: 7 x 3 x 12, 64 31.7 / 32.0, 43.2 / 46.8, 106.6 / 125.7
//   twice as much: 4 x 1 x 9, 64 19.5 / 20.2, 23.3 / 25.8, 45.7 / 57.7   2.25 times: 9 x 1 x 8, 64 21.9 / 27.3, 28.6 / 40.7, 69.9 / 111.6
//   a vector more than whole tiles: 3 x 3 x 14, 64 27.1 / 23.2, 44.3 / 30.0, 88.4 / 65.9   3 x 1 x 21, 64 21.7 / 19.0, 28.1 / 23.8, 69.2 / 47.7
//   small results, 392000 positions: 7 x 1 x 8, 8 124 / 93   3 x 1 x 20, 8 128 / 50
// Large results: a tile of x is fetched again for every 64 or 96 filters and one of dy for every filter row, and workgroups that leave CUs idle
// in their last round cost more than the fetches save against split products in tiles of 128 x 128 (more than 64 filters).  So not where
// a round behind the first is short of full, nor where a fifth of the only round is empty and the product is large enough (some 2e10
// multiplications) for several of those tiles on a CU.  3 x 3 taps, positions x filters x channels, split products / this one: 39200 x 256 x
// 256 350 / 399, 196000 x 512 x 128 1497 / 1899, 12544 x 512 x 512 434 / 533, 5 x 5 taps 4312 x 256 x 256 127 / 158, 12544 x 80 x 512
// 295 / 368, 1 x 1 12544 x 2048 x 2048 743 / 789; full rounds, or smaller: 25088 x 256 x 256 295 / 263, 58800 x 384 x 384 1286 / 1178, 2 x 2
// 12544 x 1024 x 512 443 / 421, 1 x 1 12544 x 1024 x 2048 402 / 400; at most 64 filters: 5 x 5 12544 x 64 x 1024 428 / 400.
inline bool conv_wgrad_split_ok(const ConvGeom& g, const float* x, const float* dy, int cu) {
  const int64_t positions = (int64_t)g.n * g.ho * g.wo, run = (int64_t)g.kw * g.cin, rows = g.kh * run;
  const auto fits = [](const float* p, int64_t elems) { return (reinterpret_cast<uintptr_t>(p) & 3u) == 0 && elems * 4 < ((int64_t)1 << 31) - 4096; };
  if (!(g.cin >= 8 && g.cin <= 4096 && g.kh <= 15 && g.kw <= 15 && fits(x, (int64_t)g.n * g.h * g.w * g.cin) && fits(dy, positions * g.cout) &&
        positions >= 4096))
    return false;
  const int64_t here = g.kh * 32 * ceil_div(run, 32), packed = g.kh * 4 * ceil_div(run, 4), there = packed <= 32 ? 32 : 64 * ceil_div(packed, 64);
  if (2 * here >= 3 * there && rows * g.cout > 512 &&
      (4 * here >= 9 * there || (positions >= 32768 && !(g.cout <= 64 && g.kh <= 5 && 3 * here <= 5 * there))))
    return false;
  if (g.cout <= 64) return true;
  const WgradSplitPlan p = conv_wgrad_split_plan(g, cu, rows * g.cout * cu);
  const int64_t items = (int64_t)g.kh * p.groups_m * p.groups_n * p.parts, places = ceil_div(items, cu) * cu, idle = places - items;
  return places > cu ? 20 * idle <= places : 5 * idle <= places || (double)positions * (double)(rows * g.cout) < 2e10;
}

// Floats of workspace for all parts of the plan, and what a model sets aside for it: by its largest batch, or by halves of that, the first
// that runs it (the rule has lines above which it does not), nothing where none does.
inline int64_t conv_wgrad_split_workspace(const ConvGeom& g, int cu) {
  const int64_t size = (int64_t)g.kh * g.kw * g.cin * g.cout;
  return conv_wgrad_split_plan(g, cu, size * cu).parts * size;
}
inline int64_t conv_wgrad_split_reserve(ConvGeom g, int cu) {
  for (; g.n > 0; g.n /= 2)
    if (conv_wgrad_split_ok(g, nullptr, nullptr, cu)) return conv_wgrad_split_workspace(g, cu);
  return 0;
}

}  // namespace sn
