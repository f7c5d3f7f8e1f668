// How the first-layer filter gradient is divided, asked on the command line and answered without a GPU:
//   cut rows wo room        segments, their length, items per wavefront, workgroups
#include "../../scanet3_amd/csrc/conv_first_rules.hpp"

#include <cstdio>
#include <cstdlib>
#include <cstring>

int main(int argc, char** argv) {
  if (argc != 5 || std::strcmp(argv[1], "cut")) return 2;
  const sn::FirstWgradCut c = sn::conv_first_wgrad_cut(std::atoll(argv[2]), std::atoi(argv[3]), std::atoll(argv[4]));
  std::printf("%d %d %d %d\n", c.segments, c.segment_length, c.items_per_wave, c.parts);
  return 0;
}
