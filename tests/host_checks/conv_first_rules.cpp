// Which first layers have kernels of their own and how these divide them, asked on the command line and answered without a GPU:
//   forward kh kw cin cout  whether that product of 24 x 24 images runs there (0/1)
//   tiles taps cout stats  tiles of 16 filters a wavefront of the forward product takes
//   cut rows wo room        segments, their length, items per wavefront, workgroups
#include "../../scanet3_amd/csrc/conv_first_rules.hpp"

#include <cstdio>
#include <cstdlib>
#include <cstring>

int main(int argc, char** argv) {
  if (argc == 6 && !std::strcmp(argv[1], "forward")) {
    const int kh = std::atoi(argv[2]), kw = std::atoi(argv[3]), cin = std::atoi(argv[4]), cout = std::atoi(argv[5]);
    alignas(16) static float at[4];
    sn::Epilogue e;
    e.out = at;
    e.ldo = cout;
    std::printf("%d\n", sn::conv_first_fwd_ok(sn::ConvGeom{64, 24, 24, cin, 25 - kh, 25 - kw, cout, kh, kw, 1, 1, 0, 0}, e));
    return 0;
  }
  if (argc == 5 && !std::strcmp(argv[1], "tiles")) {
    std::printf("%d\n", sn::conv_first_fwd_tiles(std::atoi(argv[2]), std::atoi(argv[3]), std::atoi(argv[4]) != 0));
    return 0;
  }
  if (argc != 5 || std::strcmp(argv[1], "cut")) return 2;
  const sn::FirstWgradCut c = sn::conv_first_wgrad_cut(std::atoll(argv[2]), std::atoi(argv[3]), std::atoll(argv[4]));
  std::printf("%d %d %d %d\n", c.segments, c.segment_length, c.items_per_wave, c.parts);
  return 0;
}
