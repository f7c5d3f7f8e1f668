// Which first layers conv_first_kernels.hip takes, and how it divides them over wavefronts (host only).
#pragma once
#include "common.hpp"

#include <algorithm>

namespace sn {

// Forward: up to 64 taps, whole vectors of filters.  A wavefront keeps 64 filters' weights and gathers its positions' inputs anew for
// every 64 filters, one value a lane, so many taps onto many filters are the tiled kernels': 64 taps x 256 filters over 10000 positions
// 16.3 us there and 28.9 here, 36 x 344 26.2 and 33.4, 48 x 512 30.0 and 54.9.  Up to 28 taps it is the other way round at any
// number of filters (27 x 512 over 10816: 32.2 and 27.7, 9 x 1400 95.0 and 42.7).
inline bool conv_first_fwd_ok(const ConvGeom& g, const Epilogue& e) {
  const int64_t positions = (int64_t)g.n * g.ho * g.wo, taps = (int64_t)g.kh * g.kw * g.cin;
  return g.cin <= 4 && taps <= 64 && (taps <= 28 || taps * g.cout <= 12288) && g.cout % 4 == 0 && e.ldo % 4 == 0 &&
         (reinterpret_cast<uintptr_t>(e.out) & 15u) == 0 && positions > 0 && positions < (1ll << 30) &&
         (int64_t)g.h * g.w * g.cin < (1ll << 30) && g.h < (1 << 20) && g.cout <= 4096;
}

// Tiles of 16 filters a wavefront multiplies its positions' inputs with: up to four.  Where the inputs are cheap to gather again and
// nothing of a second tile is left over, two and twice the wavefronts: the weights are there sooner and fewer registers leave more
// wavefronts in flight (9 taps x 64 filters, 67600 positions 16.5 -> 15.7 us, 18 x 64 19.3 -> 17.9, 18 x 128 28.0 -> 21.5; but 27 x 64
// over 225000 29.4 -> 30.9, 32 x 64 over 210000 36 -> 40, 56 filters at 9 taps over 225000 20.9 -> 21.0, and a training step whose
// first layer of 64 filters also forms a batch normalisation's statistics, over 500 images of 28 x 28, 159 -> 165).
inline int conv_first_fwd_tiles(int taps, int cout, bool statistics) {
  const int tiles = (int)ceil_div((int64_t)cout, (int64_t)16);
  return !statistics && taps <= 20 && cout > 32 && cout % 32 == 0 ? 2 : std::min(tiles, 4);
}

// Filter gradient: `rows` rows of `wo` output positions for at most `room` workgroups of four wavefronts.  A wavefront takes items_per_wave rows in
// turn; where there are not half as many rows as wavefronts (signals: images of one or a few long rows), rows are cut into
// segments of whole trips of 16 positions, until there is one for every wavefront.  9 taps x 32 filters with whole rows and
// with segments: 8 rows of 4088 positions 344 and 6.3 us, 64 of 2040 182 and 8.5, 128 of 504 48 and 7.6, 224 of 20 6.7 and 6.3.
struct FirstWgradCut {
  int segments = 0, segment_length = 0, items_per_wave = 0, parts = 0;  // parts: workgroups, each leaves one partial filter
};
inline FirstWgradCut conv_first_wgrad_cut(int64_t rows, int wo, int64_t room) {
  FirstWgradCut c;
  const int64_t waves = 4 * room;
  const int64_t trips = ceil_div((int64_t)wo, (int64_t)16), wanted = std::min<int64_t>(std::max<int64_t>(waves / rows, 1), trips);
  const int64_t trips_each = ceil_div(trips, wanted);
  c.segments = (int)ceil_div(trips, trips_each);
  c.segment_length = (int)(16 * trips_each);
  const int64_t items = rows * c.segments;
  c.items_per_wave = (int)ceil_div(items, waves);
  c.parts = (int)ceil_div(items, (int64_t)4 * c.items_per_wave);
  return c;
}

}  // namespace sn
