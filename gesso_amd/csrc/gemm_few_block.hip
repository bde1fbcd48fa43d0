// The products of up to 64 rows with what follows them in a block: the stream, the convolution, a part of K's sums (gemm_few_impl.h).
#include "gemm_few_impl.h"

void gs_few_residual_run(const SkinnyCall& c) {
  FewArgs g = few_args(c);
  g.Y = c.ex.xs_out; g.w = c.ex.next_w; g.io = c.ex.res_out; g.ssq_out = c.ex.ssq_out;
  if (skinny_once(c.N, c.K)) launch_few_rows<1, 8, 8, 2, true, false, 2, 1, true, float>(c.N / 8, g, c.stream);
  else launch_few_rows<1, 8, 8, 2, true, false, 2, 1, false, float>(c.N / 8, g, c.stream);
}

template <int CW, bool ONCE>
static void conv(const SkinnyCall& c) {
  FewArgs g = few_args(c);
  g.slots = c.ex.slots; g.w = c.ex.taps; g.bias = c.ex.conv_bias; g.io = c.ex.state;
  if (c.ex.ssq) launch_few_rows<3, 8, 8, 2, true, true, 3, CW, ONCE, bf16>(c.N / 24, g, c.stream);
  else launch_few_rows<3, 8, 8, 4, true, false, 3, CW, ONCE, bf16>(c.N / 24, g, c.stream);
}
template <int CW>
static void conv_width(const SkinnyCall& c) { skinny_once(c.N, c.K) ? conv<CW, true>(c) : conv<CW, false>(c); }
void gs_few_conv_run(const SkinnyCall& c) {
  if (c.ex.conv_w == 2) conv_width<2>(c);
  else if (c.ex.conv_w == 3) conv_width<3>(c);
  else conv_width<4>(c);
}

// Two weight tiles a block of four wavefronts.  (Four of eight, which bring in a third less of X a compute unit: 64 rows of 2048 x 8192
// in eight parts 11.6 us, so 11.5.)
void gs_few_parts_run(const SkinnyCall& c, int parts) {
  const dim3 grid(parts, gs_ceil_div(c.N, 32));
  FewArgs g = few_args(c);
  g.ldy = c.N;
  if (skinny_once(c.N, c.K)) launch_few_rows<2, 4, 4, 4, false, false, 5, 1, true, float>(grid, g, c.stream);
  else launch_few_rows<2, 4, 4, 4, false, false, 5, 1, false, float>(grid, g, c.stream);
}
