// Workspace rules of the batch normalisation's reductions, asked on the command line and answered without a GPU, for 256 CUs:
//   room cols batch         slices that a workspace for `batch` rows holds, and the most that a pass over 1 .. batch rows asks for
//   stream cols rows        slices asked for, and what the streaming form writes
//   written cols rows       slices asked for, and the most that a reduction over these rows writes in any of its forms
#include "../../scanet3_amd/csrc/batchnorm_rules.hpp"

#include <cstdio>
#include <cstdlib>
#include <cstring>

int main(int argc, char** argv) {
  if (argc != 4) return 2;
  const int cus = 256, cols = std::atoi(argv[2]);
  const int64_t rows = std::atoll(argv[3]);
  if (!std::strcmp(argv[1], "room")) {
    int most = 0;
    for (int64_t r = 1; r <= rows; ++r) most = std::max(most, sn::bn_max_slices(cus, r, cols));
    std::printf("%d %d\n", sn::bn_max_slices(cus, rows, cols), most);
    return 0;
  }
  if (!std::strcmp(argv[1], "stream")) {
    std::printf("%d %d\n", sn::bn_max_slices(cus, rows, cols), sn::bn_stream_of(cus, rows, cols).slices);
    return 0;
  }
  if (!std::strcmp(argv[1], "written")) {
    int most = sn::bn_row_slices(cus, rows, cols);
    if (sn::bn_stream_form(cols)) most = std::max(most, sn::bn_stream_of(cus, rows, cols).slices);
    std::printf("%d %d\n", sn::bn_max_slices(cus, rows, cols), most);
    return 0;
  }
  return 2;
}
