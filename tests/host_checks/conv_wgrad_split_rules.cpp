// Which filter gradients conv_wgrad_split_kernels.hip takes and how it divides them, asked on the command line and answered without a GPU:
//   n h w cin cout kh kw sh same room     taken tm tn groups_m groups_n chunks parts padded workspace reserve (256 compute units; room: workspace floats, -1: its own)
#include "../../scanet3_amd/csrc/conv_wgrad_split_rules.hpp"

#include <cstdio>
#include <cstdlib>

int main(int argc, char** argv) {
  if (argc != 11) return 2;
  int v[9];
  for (int i = 0; i < 9; ++i) v[i] = std::atoi(argv[i + 1]);
  static float at[4];
  const int sh = v[7], same = v[8];
  const sn::ConvGeom g{v[0], v[1], v[2], v[3], same ? (v[1] + sh - 1) / sh : (v[1] - v[5]) / sh + 1, same ? v[2] : v[2] - v[6] + 1, v[4], v[5], v[6], sh, 1,
                       same ? (v[5] - 1) / 2 : 0, same ? (v[6] - 1) / 2 : 0};
  const int64_t workspace = sn::conv_wgrad_split_workspace(g, 256), room = std::atoll(argv[10]);
  const sn::WgradSplitPlan p = sn::conv_wgrad_split_plan(g, 256, room < 0 ? workspace : room);
  std::printf("%d %d %d %d %d %d %d %d %lld %lld\n", sn::conv_wgrad_split_ok(g, at, at, 256), p.tm, p.tn, p.groups_m, p.groups_n, p.chunks, p.parts, p.padded,
              (long long)workspace, (long long)sn::conv_wgrad_split_reserve(g, 256));
  return 0;
}
