// Dense products (forward NN, input gradient NT, weight gradient TN) on the split kernels (split_gemm.hpp).
#include "split_launch.hpp"

namespace sn {

// Both operands need one unit stride and at least four values along it (a vector of four is loaded from inside its row),
// 32-bit byte offsets; rows need no alignment.
bool split_dense_ok(const GemmDesc& g) {
  const int m = g.m - (g.a_ones_row ? 1 : 0);
  if (m < 1) return false;
  const bool akc = g.a_sk == 1, bkc = g.b_sk == 1 && g.b_sn != 1;
  if (g.a_ones_row && (akc || bkc)) return false;
  return (akc ? FlatOp<true>::ok(g.a, g.a_sm, g.a_sk, m, g.k) : FlatOp<false>::ok(g.a, g.a_sm, g.a_sk, m, g.k)) &&
         (bkc ? FlatOp<true>::ok(g.b, g.b_sn, g.b_sk, g.n, g.k) : FlatOp<false>::ok(g.b, g.b_sn, g.b_sk, g.n, g.k));
}

template <int PLANES, bool AK, bool BK>
static int launch_pair(sn_ctx* ctx, const char* name, const GemmDesc& g, const Epilogue& e, float* ws, int64_t ws_elems) {
  const int m = g.m - (g.a_ones_row ? 1 : 0);
  FlatOp<AK> al{g.a, (int)(AK ? g.a_sm : g.a_sk), m, g.k};
  FlatOp<BK> bl{g.b, (int)(BK ? g.b_sn : g.b_sk), g.n, g.k};
  return launch_split<PLANES>(ctx, name, m, g.n, g.k, g.m, g.a_ones_row ? m : -1, al, bl, StdEpilogue{e}, ws, ws_elems);
}

template <int PLANES>
static int launch_planes(sn_ctx* ctx, const char* name, const GemmDesc& g, const Epilogue& e, float* ws, int64_t ws_elems) {
  const bool akc = g.a_sk == 1, bkc = g.b_sk == 1 && g.b_sn != 1;
  if (akc && bkc) return launch_pair<PLANES, true, true>(ctx, name, g, e, ws, ws_elems);
  if (akc) return launch_pair<PLANES, true, false>(ctx, name, g, e, ws, ws_elems);
  if (bkc) return launch_pair<PLANES, false, true>(ctx, name, g, e, ws, ws_elems);
  return launch_pair<PLANES, false, false>(ctx, name, g, e, ws, ws_elems);
}

int launch_split_dense(sn_ctx* ctx, const char* name, const GemmDesc& g, const Epilogue& e, float* ws, int64_t ws_elems, bool bf16) {
  SN_REQUIRE(split_dense_ok(g), "%s: operands outside the split kernels' range", name);
  return bf16 ? launch_planes<1>(ctx, name, g, e, ws, ws_elems) : launch_planes<3>(ctx, name, g, e, ws, ws_elems);
}

// dX = dY . W^T through the gradient of the layer below's activation
int launch_split_dense_act_grad(sn_ctx* ctx, const GemmDesc& g, const ActGrad& a, float* ws, int64_t ws_elems, bool bf16) {
  SN_REQUIRE(split_dense_ok(g) && g.a_sk == 1 && g.b_sk == 1 && g.b_sn != 1 && !g.a_ones_row, "input gradient outside the split kernels' range");
  FlatOp<true> al{g.a, (int)g.a_sm, g.m, g.k}, bl{g.b, (int)g.b_sn, g.n, g.k};
  const ActGradEpilogue ep{a.out, a.y, a.ldo, a.act, a.act_param};
  return bf16 ? launch_split<1>(ctx, "gemm_bf16_and_activation_gradient", g.m, g.n, g.k, g.m, -1, al, bl, ep, ws, ws_elems)
              : launch_split<3>(ctx, "gemm_f32_and_activation_gradient", g.m, g.n, g.k, g.m, -1, al, bl, ep, ws, ws_elems);
}

}  // namespace sn
