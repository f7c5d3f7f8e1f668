// Conv2D forward, input gradient (unit strides) and filter gradient as implicit GEMMs on the split kernels (split_gemm.hpp):
// any channel count, padding and kernel size; a filter row of a position is read as one run of kw * channels floats.
#include "split_launch.hpp"

namespace sn {

static bool interior(const ConvGeom& g) {
  return g.pt == 0 && g.pl == 0 && (g.ho - 1) * g.sh + g.kh <= g.h && (g.wo - 1) * g.sw + g.kw <= g.w;
}
int launch_split_conv_fwd(sn_ctx* ctx, const ConvGeom& g, const float* x, const float* w, const Epilogue& e, float* ws, int64_t ws_elems) {
  const int L = g.kw * g.cin, Lp = (int)align_up(L, 4), M = g.n * g.ho * g.wo, K = g.kh * Lp, N = g.cout;
  const int total = g.n * g.h * g.w * g.cin;
  const StdEpilogue ep{e};
  auto run = [&](auto al) {
    al.src = x;
    al.M = M; al.ih = g.ho; al.iw = g.wo; al.sy = g.sh; al.sx = g.sw; al.oy = -g.pt; al.ox = -g.pl; al.ty = 1;
    al.H = g.h; al.W = g.w; al.C = g.cin; al.kh = g.kh; al.L = L; al.Lp = Lp; al.total = total;
    al.by_iw = fast_div((uint32_t)g.wo);
    al.by_ih = fast_div((uint32_t)g.ho);
    al.walk = run_walk(Lp);
    if (L == Lp) return launch_split<3>(ctx, "conv2d_forward", M, N, K, M, -1, al, FlatOp<false>{w, N, N, K}, ep, ws, ws_elems);
    return launch_split<3>(ctx, "conv2d_forward", M, N, K, M, -1, al, ConvRunFilterOp{w, N, g.kh, L, Lp, run_walk(Lp)}, ep, ws, ws_elems);
  };
  if (interior(g) && L == Lp) return run(ConvRunOp<false>{});
  return run(ConvRunOp<true>{});
}

int launch_split_conv_dgrad(sn_ctx* ctx, const ConvGeom& g, const float* dy, const float* w, float* dx, float* ws, int64_t ws_elems) {
  const int L = g.kw * g.cout, Lp = (int)align_up(L, 4), M = g.n * g.h * g.w, K = g.kh * Lp, N = g.cin;
  Epilogue e;
  e.out = dx;
  e.ldo = g.cin;
  const StdEpilogue ep{e};
  ConvRunOp<true> al{};
  al.src = dy;
  al.M = M; al.ih = g.h; al.iw = g.w; al.sy = 1; al.sx = 1; al.oy = g.pt; al.ox = g.pl - (g.kw - 1); al.ty = -1;
  al.H = g.ho; al.W = g.wo; al.C = g.cout; al.kh = g.kh; al.L = L; al.Lp = Lp;
  al.total = g.n * g.ho * g.wo * g.cout;
  al.by_iw = fast_div((uint32_t)g.w);
  al.by_ih = fast_div((uint32_t)g.h);
  al.walk = run_walk(Lp);
  const FastDiv by_cout = fast_div((uint32_t)g.cout);
  if (g.cout % 4 == 0)
    return launch_split<3>(ctx, "conv2d_input_gradient", M, N, K, M, -1, al, ConvDgradFilterOp<true>{w, g.cin, g.cout, g.kh, g.kw, L, Lp, by_cout, run_walk(Lp)}, ep, ws, ws_elems);
  return launch_split<3>(ctx, "conv2d_input_gradient", M, N, K, M, -1, al, ConvDgradFilterOp<false>{w, g.cin, g.cout, g.kh, g.kw, L, Lp, by_cout, run_walk(Lp)}, ep, ws, ws_elems);
}

int launch_split_conv_wgrad(sn_ctx* ctx, const ConvGeom& g, const float* x, const float* dy, float* dw, float* ws, int64_t ws_elems) {
  const int L = g.kw * g.cin, Lp = (int)align_up(L, 4), K = g.n * g.ho * g.wo, N = g.cout;
  const FlatOp<false> bl{dy, N, N, K};
  auto run = [&](auto al) {
    al.x = x; al.g = g; al.L = L; al.Lp = Lp; al.K = K; al.total = g.n * g.h * g.w * g.cin; al.rows = g.kh * Lp;
    al.by_wo = fast_div((uint32_t)g.wo);
    al.by_ho = fast_div((uint32_t)g.ho);
    al.step_ow = 32 % g.wo;
    al.step_oh = 32 / g.wo % g.ho;
    al.step_b = 32 / g.wo / g.ho;
    if (L == Lp) {
      Epilogue e;
      e.out = dw;
      e.ldo = N;
      return launch_split<3>(ctx, "conv2d_filter_gradient", g.kh * L, N, K, g.kh * L, -1, al, bl, StdEpilogue{e}, ws, ws_elems);
    }
    return launch_split<3>(ctx, "conv2d_filter_gradient", g.kh * Lp, N, K, g.kh * L, -1, al, bl, RunRowsEpilogue{dw, N, L, Lp}, ws, ws_elems);
  };
  if (interior(g) && L == Lp) return run(ConvWgradRunOp<false>{});
  return run(ConvWgradRunOp<true>{});
}

}  // namespace sn
