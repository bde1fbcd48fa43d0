// The products of up to 64 rows with what follows them in a block: the stream, the convolution, a part of K's sums (gemm_few_impl.h).
#include "gemm_few_impl.h"

// (loaded once from 4 M weights on: at most 2,560 rows of them are a K of 2,048, four loads a wavefront)
bool gs_few_residual_run(const SkinnyCall& c) {
  FewArgs g = few_args(c);
  g.Y = c.ex.xs_out; g.w = c.ex.next_w; g.io = c.ex.res_out; g.ssq_out = c.ex.ssq_out;
  return skinny_once(c.N, c.K) ? launch_few_rows<1, 8, 8, 2, true, false, 2, 1, true, float, 4>(c.N / 8, g, c.stream)
                               : launch_few_rows<1, 8, 8, 2, true, false, 2, 1, false, float>(c.N / 8, g, c.stream);
}

// (loaded once from 4 M weights on: at most 6,144 rows of them are a K of 1,024, two loads a wavefront)
template <int CW, bool ONCE>
static bool conv(const SkinnyCall& c) {
  FewArgs g = few_args(c);
  g.slots = c.ex.slots; g.w = c.ex.taps; g.bias = c.ex.conv_bias; g.io = c.ex.state;
  return c.ex.ssq ? launch_few_rows<3, 8, 8, 2, true, true, 3, CW, ONCE, bf16, ONCE ? 2 : 1>(c.N / 24, g, c.stream)
                  : launch_few_rows<3, 8, 8, 4, true, false, 3, CW, ONCE, bf16, ONCE ? 2 : 1>(c.N / 24, g, c.stream);
}
template <int CW>
static bool conv_width(const SkinnyCall& c) { return skinny_once(c.N, c.K) ? conv<CW, true>(c) : conv<CW, false>(c); }
bool gs_few_conv_run(const SkinnyCall& c) { return c.ex.conv_w == 2 ? conv_width<2>(c) : c.ex.conv_w == 3 ? conv_width<3>(c) : conv_width<4>(c); }

// Two weight tiles a block of four wavefronts.  (Four of eight, which bring in a third less of X a compute unit: 64 rows of 2048 x 8192
// in eight parts 11.6 us, so 11.5.)
bool gs_few_parts_run(const SkinnyCall& c, int parts) {
  const dim3 grid(parts, gs_ceil_div(c.N, 32));
  FewArgs g = few_args(c);
  g.ldy = c.N;
  return skinny_once(c.N, c.K) ? launch_few_rows<2, 4, 4, 4, false, false, 5, 1, true, float>(grid, g, c.stream)
                               : launch_few_rows<2, 4, 4, 4, false, false, 5, 1, false, float>(grid, g, c.stream);
}
