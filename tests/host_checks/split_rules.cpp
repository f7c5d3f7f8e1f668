// Host-side rules of the split products, asked on the command line and answered without a GPU:
//   choose m n k planes deferred                     tile (bm bn bk) and split count of a product on 256 CUs
//   defers m n plain                                 whether the optimizer's launch can add its partial results (0/1)
//   float32 m n k channels                           whether a convolution's product stays off the split kernels (0/1)
//   conv n h w cin ho wo cout kh kw sh sw pt pl      which convolution products read tensors of exactly these sizes: three 0/1
#include "../../scanet3_amd/csrc/split_launch.hpp"

#include <cstdio>
#include <cstdlib>
#include <cstring>

int main(int argc, char** argv) {
  std::vector<int> v;
  for (int i = 2; i < argc; ++i) v.push_back(std::atoi(argv[i]));
  alignas(16) static float at[4];
  if (argc == 15 && !std::strcmp(argv[1], "conv")) {
    const sn::ConvGeom g{v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8], v[9], v[10], v[11], v[12]};
    std::printf("%d %d %d\n", sn::split_conv_fwd_ok(g, at, at), sn::split_conv_dgrad_ok(g, at, at), sn::split_conv_wgrad_ok(g, at, at));
    return 0;
  }
  if (argc == 7 && !std::strcmp(argv[1], "choose")) {
    const sn::SplitChoice c = sn::split_choose(v[0], v[1], v[2], 256, 256, v[4] != 0, v[3]);
    std::printf("%d %d %d %d\n", sn::SPLIT_TILE[c.tile].bm, sn::SPLIT_TILE[c.tile].bn, sn::SPLIT_TILE[c.tile].bk, c.splits);
    return 0;
  }
  if (argc == 6 && !std::strcmp(argv[1], "float32")) {
    std::printf("%d\n", sn::conv_prefers_float32_tiles(v[0], v[1], v[2], v[3]));
    return 0;
  }
  if (argc == 5 && !std::strcmp(argv[1], "defers")) {
    std::printf("%d\n", sn::split_defers(v[2] ? at : nullptr, at, v[0], v[1]));
    return 0;
  }
  return 2;
}
