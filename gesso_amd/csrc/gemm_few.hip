// Which products of up to 16 rows go to the kernels of gemm_few_impl.h, and the launches of the plain ones.
#include "gemm_few_impl.h"

// Whether a wavefront's share of K is whole loads: the same number for each of a block's eight.
static bool few_takes(const SkinnyCall& c, const void* Wt, bool half) {
  return Wt && c.M <= 16 && c.K % (FEW_WAVES * 32 * (half ? 2 : 1)) == 0 && !c.ex.res;
}

FewArgs few_args(const SkinnyCall& c) {
  FewArgs g = {};
  g.W = c.w; g.X = c.x; g.M = c.M; g.N = c.N; g.K = c.K;
  g.xrow = c.ex.x_tiled ? 8 : c.ldx; g.xgroup = c.ex.x_tiled ? 128 : 8; g.xstep = c.ex.x_tiled ? 512 : 32;
  g.ssq = c.ex.ssq; g.nb = c.ex.nb; g.eps = c.ex.eps;
  g.Y = c.Y; g.ldy = c.ldy; g.tiled = c.ex.y_tiled; g.extra = c.ex.squared;
  return g;
}

template <int R, bool HALF, bool SCALED, bool ONCE>
static void few_plain_out(const SkinnyCall& c, int blocks) {
  if (c.y_dtype == GS_F32) launch_few<R, HALF, SCALED, 0, 1, ONCE, float>(blocks, few_args(c), c.stream);
  else launch_few<R, HALF, SCALED, 0, 1, ONCE, bf16>(blocks, few_args(c), c.stream);
}
template <int R, bool HALF>
static void few_plain(const SkinnyCall& c, int blocks) {
  if (skinny_once(c.N, c.K)) c.ex.ssq ? few_plain_out<R, HALF, true, true>(c, blocks) : few_plain_out<R, HALF, false, true>(c, blocks);
  else c.ex.ssq ? few_plain_out<R, HALF, true, false>(c, blocks) : few_plain_out<R, HALF, false, false>(c, blocks);
}

// A plain product (`half`: of a weight of few rows, half a tile a block), or gate and up with SwiGLU; false: not for these kernels.
bool gs_few_plain(const SkinnyCall& c, const void* Wt, bool half) {
  if (!few_takes(c, Wt, half)) return false;
  if (c.epilogue == 1) {
    if (c.y_dtype != GS_BF16) return false;
    gs_few_swiglu(c);
  } else if (half) few_plain<1, true>(c, c.N / 8);
  else if (c.N <= 8192) few_plain<1, false>(c, c.N / 16);
  else few_plain<2, false>(c, gs_ceil_div(c.N, 32));
  return true;
}

bool gs_few_gated(const SkinnyCall& c, const void* Wt) {
  if (!few_takes(c, Wt, false)) return false;
  gs_few_gated_run(c);
  return true;
}

// Into the stream: weights of few rows, half a tile a block.
bool gs_few_residual(const SkinnyCall& c, const void* Wt) {
  if (!gs_skinny_halves(c.N) || !few_takes(c, Wt, true)) return false;
  gs_few_residual_run(c);
  return true;
}

// The convolution: where every block has a compute unit to itself (three tiles' sums leave a lane's registers no room for two).
bool gs_few_conv(const SkinnyCall& c, const void* Wt) {
  if (!c.ex.conv_vec || c.N / 24 > 256 || !few_takes(c, Wt, true)) return false;
  gs_few_conv_run(c);
  return true;
}
