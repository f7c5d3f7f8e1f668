// How the first-layer filter gradient is divided over wavefronts (host only).
#pragma once
#include "common.hpp"

#include <algorithm>

namespace sn {

// `rows` rows of `wo` output positions for at most `room` workgroups of four wavefronts.  A wavefront takes items_per_wave rows in
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
