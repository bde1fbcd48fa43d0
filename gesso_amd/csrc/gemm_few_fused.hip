// The products of up to 16 rows with what follows them in a block (gemm_few_impl.h).
#include "gemm_few_impl.h"

template <bool ONCE>
static void swiglu(const SkinnyCall& c) {
  const int blocks = c.N / 32;
  if (c.ex.ssq) launch_few<2, false, true, 1, 1, ONCE, bf16>(blocks, few_args(c), c.stream);
  else launch_few<2, false, false, 1, 1, ONCE, bf16>(blocks, few_args(c), c.stream);
}
void gs_few_swiglu(const SkinnyCall& c) { skinny_once(c.N, c.K) ? swiglu<true>(c) : swiglu<false>(c); }

void gs_few_gated_run(const SkinnyCall& c) {
  FewArgs g = few_args(c);
  g.bias = c.ex.act_bias;
  g.extra = c.ex.act;
  if (skinny_once(c.N, c.K)) launch_few<2, false, false, 4, 1, true, bf16>(c.N / 32, g, c.stream);
  else launch_few<2, false, false, 4, 1, false, bf16>(c.N / 32, g, c.stream);
}

void gs_few_residual_run(const SkinnyCall& c) {
  FewArgs g = few_args(c);
  g.Y = c.ex.xs_out; g.w = c.ex.next_w; g.io = c.ex.res_out; g.ssq_out = c.ex.ssq_out;
  if (skinny_once(c.N, c.K)) launch_few<1, true, false, 2, 1, true, float>(c.N / 8, g, c.stream);
  else launch_few<1, true, false, 2, 1, false, float>(c.N / 8, g, c.stream);
}

template <int CW, bool ONCE>
static void conv(const SkinnyCall& c) {
  FewArgs g = few_args(c);
  g.slots = c.ex.slots; g.w = c.ex.taps; g.bias = c.ex.conv_bias; g.io = c.ex.state;
  if (c.ex.ssq) launch_few<3, true, true, 3, CW, ONCE, bf16>(c.N / 24, g, c.stream);
  else launch_few<3, true, false, 3, CW, ONCE, bf16>(c.N / 24, g, c.stream);
}
template <int CW>
static void conv_width(const SkinnyCall& c) { skinny_once(c.N, c.K) ? conv<CW, true>(c) : conv<CW, false>(c); }
void gs_few_conv_run(const SkinnyCall& c) {
  if (c.ex.conv_w == 2) conv_width<2>(c);
  else if (c.ex.conv_w == 3) conv_width<3>(c);
  else conv_width<4>(c);
}
