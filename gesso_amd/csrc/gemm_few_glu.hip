// Gate and up of up to 64 rows, and the head's like of them (gemm_few_impl.h).
#include "gemm_few_impl.h"

// Four tiles a block where four row tiles of X are read (skinny_fours: the rule and what it measured), else two.
int few_glu_waves(const SkinnyCall& c) { return c.M > 32 && !skinny_fours(c.M, c.N / 2, c.K) ? 4 : 8; }

template <bool ONCE>
static bool swiglu(const SkinnyCall& c) {
  const int blocks = c.N / 32;
  if (c.ex.ssq) return launch_few_rows<2, 8, 4, 2, false, true, 1, 1, ONCE, bf16>(blocks, few_args(c), c.stream);
  // (four tiles a block: from 16,384 rows of 2,048 weights on, which are loaded once and make eight loads a wavefront)
  if (ONCE && skinny_fours(c.M, c.N / 2, c.K)) return launch_few<4, 4, 8, false, false, 1, 1, true, bf16, 8>((blocks + 1) / 2, few_args(c), c.stream);
  return launch_few_rows<2, 8, 4, 4, false, false, 1, 1, ONCE, bf16>(blocks, few_args(c), c.stream);
}
bool gs_few_swiglu(const SkinnyCall& c) { return skinny_once(c.N, c.K) ? swiglu<true>(c) : swiglu<false>(c); }

bool gs_few_gated_run(const SkinnyCall& c) {
  FewArgs g = few_args(c);
  g.bias = c.ex.act_bias;
  g.extra = c.ex.act;
  return skinny_once(c.N, c.K) ? launch_few_rows<2, 8, 4, 4, false, false, 4, 1, true, bf16>(c.N / 32, g, c.stream)
                               : launch_few_rows<2, 8, 4, 4, false, false, 4, 1, false, bf16>(c.N / 32, g, c.stream);
}
