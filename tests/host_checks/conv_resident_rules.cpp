// Which convolutions conv_resident_kernels.hip takes and how it divides them, asked on the command line and answered without a GPU:
//   plan positions columns channels kh kw     units_per_row units pairs chunk tn blocks_n tiles wvk per_block lds (256 compute units)
//   takes n h w cin cout kh kw same           forward, input gradient (0/1 each)
#include "../../scanet3_amd/csrc/conv_resident_rules.hpp"

#include <cstdio>
#include <cstdlib>
#include <cstring>

int main(int argc, char** argv) {
  int v[8] = {};
  for (int i = 2; i < argc && i < 10; ++i) v[i - 2] = std::atoi(argv[i]);
  if (argc == 7 && !std::strcmp(argv[1], "plan")) {
    const sn::ResidentPlan p = sn::resident_plan(v[0], v[1], v[2], v[3], v[4], 256);
    std::printf("%d %d %d %d %d %d %d %d %d %d\n", p.units_per_row, p.units, p.pairs, p.chunk, p.tn, p.blocks_n, p.tiles, p.wvk, p.per_block, p.lds);
    return 0;
  }
  if (argc != 10 || std::strcmp(argv[1], "takes")) return 2;
  alignas(16) static float at[4];
  const int same = v[7];
  const sn::ConvGeom g{v[0], v[1], v[2], v[3], same ? v[1] : v[1] - v[5] + 1, same ? v[2] : v[2] - v[6] + 1, v[4], v[5], v[6], 1, 1, same ? (v[5] - 1) / 2 : 0,
                       same ? (v[6] - 1) / 2 : 0};
  sn::Epilogue e;
  e.out = at;
  e.ldo = g.cout;
  std::printf("%d %d\n", sn::conv_resident_fwd_ok(g, at, at, e, 256), sn::conv_resident_dgrad_ok(g, at, at, at, 256));
  return 0;
}
