// Which products go to the kernels of gemm_few_impl.h, and the launches of the plain ones.
#include "gemm_few_impl.h"

// Whether a wavefront's share of K is whole loads, the same number for each of a block's `waves` (and for each part), and X's rows lie
// within 4 GB, which a lane's 32 bits of bytes reach (rows further apart are the older kernel's, as they were).
extern "C" int gs_gemm_few_takes(int M, int K, int ldx, int x_tiled, int waves, int half, int parts) {
  const long reach = x_tiled ? 16L * gs_ceil_div(M, 16) * K : (long)(M - 1) * ldx + K;
  return M <= 64 && K % (waves * 32 * (half ? 2 : 1) * parts) == 0 && reach <= 1L << 31;
}

// Rows weighted for their norm come up to 32 at a time: beyond, every block's reading of their partial sums is more than a pass.
static bool few_takes(const SkinnyCall& c, const void* Wt, int waves, bool half, int parts = 1) {
  return Wt && !c.ex.res && !(c.ex.ssq && c.M > 32) && gs_gemm_few_takes(c.M, c.K, c.ldx, c.ex.x_tiled, waves, half, parts);
}

FewArgs few_args(const SkinnyCall& c) {
  FewArgs g = {};
  const int tiles = gs_ceil_div(c.M, 16);
  g.W = c.w; g.X = c.x; g.M = c.M; g.N = c.N; g.K = c.K;
  g.xrow = c.ex.x_tiled ? 8 : c.ldx; g.xgroup = c.ex.x_tiled ? 128 : 8; g.xstep = c.ex.x_tiled ? 512 * tiles : 32; g.xtile = c.ex.x_tiled ? 512 : tiles > 1 ? 16 * c.ldx : 0;
  g.ssq = c.ex.ssq; g.nb = c.ex.nb; g.eps = c.ex.eps;
  g.Y = c.Y; g.ldy = c.ldy; g.tiled = c.ex.y_tiled; g.extra = c.ex.squared;
  return g;
}

// Loads a wavefront at least: halves come with a K of 2,048 (four); of one tile a block 4 M weights or more, loaded once, are a K of 512
// (8,192 rows; two), above 32 rows of X 1,024 (4,096 rows; four).
template <int R, int W34, int MOST, bool HALF, bool SCALED, bool ONCE>
static bool few_plain_out(const SkinnyCall& c, int blocks) {
  constexpr int least = HALF ? 4 : R == 1 && ONCE ? 2 : 1, least34 = R == 1 && ONCE ? 4 : 1;
  return c.y_dtype == GS_F32 ? launch_few_rows<R, 8, W34, MOST, HALF, SCALED, 0, 1, ONCE, float, least, least34>(blocks, few_args(c), c.stream)
                             : launch_few_rows<R, 8, W34, MOST, HALF, SCALED, 0, 1, ONCE, bf16, least, least34>(blocks, few_args(c), c.stream);
}
template <int R, int W34, int MOST, bool HALF>
static bool few_plain(const SkinnyCall& c, int blocks) {
  if (skinny_once(c.N, c.K)) return c.ex.ssq ? few_plain_out<R, W34, 2, HALF, true, true>(c, blocks) : few_plain_out<R, W34, MOST, HALF, false, true>(c, blocks);
  return c.ex.ssq ? few_plain_out<R, W34, 2, HALF, true, false>(c, blocks) : few_plain_out<R, W34, MOST, HALF, false, false>(c, blocks);
}

// Two tiles a block and 17 to 48 plain rows: up to a K of 4,096 and, of more than 32 rows, 10,240 weight rows.  Beyond, both wait for the same
// bytes and gemm_skinny_impl.h's kernel is as fast or faster (microseconds there and here, cold weights: gate and up 24 rows of 10240 x 2560
// 15.2 and 14.5, of 12288 x 4096 22.4 both, of 22528 x 4096 32.9 and 33.5; 48 rows of 9216 x 1024 9.0 and 8.8, of 10240 x 2560 18.2 both,
// of 16384 x 2048 16.1 and 16.3, of 28672 x 4096 50.8 and 52.1; stored, 17 rows of 12288 x 2048 12.8 and 12.5, of 16384 x 4096 25.9 and 26.6;
// 48 rows of 65536 x 2048 57.9 and 58.9).  49 rows and more: as tiled rows nothing was slower; as rows a K up
// to 4,096 (gated ones below it; 49 rows, stored, of 9472 x 4096 36.3 and 36.2, x 4608 42.7 and 43.5, x 10752 93.6 and 96.6, gated of 25344 x
// 2048 38.0 both, x 4096 70.3 and 71.6; 64 rows of 9472 x 4608 50.6 and 50.9).  More than 16 weighted for their norm: nothing was slower.  SwiGLU of up to 32
// rows that lie as rows, not in tiles: from 16,384 rows of 2,048 on (24 of 12288 x 2048 15.15 and 15.2, of 16384 x 2048 15.85 and 16.2, of 28672 x
// 2048 27.5 and 28.4, of 24576 x 1536 18.5 and 18.0).
// Up to 16 rows: but for one to three of a long K, which gain nothing here or lose (1 row weighted for its norm,
// SwiGLU of 1024 x 6144 10.5 and 10.7, x 10752 16.7 and 17.35, of 4096 x 9216 16.8 and 17.2; 2 rows, stored, of 12288 x 8192 42.3 and 43.1;
// 4 rows of 4096 x 7168 15.3 and 14.9; of the gated activation only one row from 10,240 on: 1024 x 10752 17.35
// and 17.6, x 8192 12.9 both), and but for 7 to 12 rows of a long K that lie a multiple of 16 KB apart (8 rows of 9216 x
// 8192 37.8 and 39.3, of 14336 x 8192 43.9 and 46.2; of SwiGLU and gated ones those of about a block a compute unit: 8192 x 8192
// 25.2 and 26.6, 25.6 and 26.2, but 5120 x 8192 18.5 and 18.4, 9216 x 8192 34.8 and 35.0, gated 35.4 and 35.0).
static bool few_pairs(const SkinnyCall& c) {
  if (c.M <= 16) {
    const bool gated = c.epilogue == 4;
    if (c.M <= (gated ? 1 : 3) && c.K >= (gated ? 10240 : 6144)) return false;
    if (!c.ex.x_tiled && c.M >= 7 && c.M <= 12 && c.K >= 8192 && c.ldx % 8192 == 0 && (c.epilogue == 0 || (c.N > 6144 && c.N <= 8192))) return false;
    return true;
  }
  if (c.M <= 32 && c.epilogue == 1 && !c.ex.ssq && !c.ex.x_tiled && c.N >= 16384 && c.K >= 2048) return false;
  if (c.M > 48 && !c.ex.x_tiled && (c.epilogue == 4 ? c.K >= 4096 : c.K > 4096)) return false;
  return c.M > 48 || c.ex.ssq || (c.K < 4096 && (c.M <= 32 || c.N <= 10240));
}

// A plain product (`half`: of a weight of few rows and up to 32 of X, half a tile a block), or gate and up with SwiGLU; false: not for
// these kernels.
bool gs_few_plain(const SkinnyCall& c, const void* Wt, bool half) {
  if (c.epilogue == 1) return c.y_dtype == GS_BF16 && few_pairs(c) && few_takes(c, Wt, few_glu_waves(c), false) && gs_few_swiglu(c);
  // More than 32 rows and one tile a block: where every block has a compute unit to itself.  (Microseconds there and here.  A ring of four loads for three or four row
  // tiles leaves a unit one block, gemm_skinny_impl.h's two: 48 rows of 4096 x 4096 11.6 and 11.5 us, of 3072 x 2048 6.9 and
  // 6.7, of 4112 x 2048 9.9 and 10.1, of 8192 x 1024 6.85 and 7.6, x 2048 11.7 and 12.1; 64 rows of 4096 x 2560 10.1 and 9.25, of 6144 x 2048
  // 13.0 and 13.4, of 8192 x 2048 13.6 and 14.2.  With 32-bit offsets, 103 and 128 registers where 132 and 170 were: 64 rows of 8192 x
  // 2048 14.5, of 4096 x 4096 13.8 for 13.1; with a ring of three and 108: 13.6 and 13.35, of 8192 x 1024 8.2 for 7.8.)
  const bool wide = !half && c.N > 8192;
  if (wide ? !few_pairs(c) : c.M > 32 && c.N > 4096) return false;
  if (!few_takes(c, Wt, wide && c.M > 32 ? 4 : 8, half)) return false;
  if (half) return few_plain<1, 8, 2, true>(c, c.N / 8);
  return wide ? few_plain<2, 4, 4, false>(c, gs_ceil_div(c.N, 32)) : few_plain<1, 8, 4, false>(c, c.N / 16);
}

bool gs_few_gated(const SkinnyCall& c, const void* Wt) {
  return few_pairs(c) && few_takes(c, Wt, c.M > 32 ? 4 : 8, false) && gs_few_gated_run(c);
}

// Into the stream: weights of few rows, half a tile a block, up to 32 rows (more come in parts).
bool gs_few_residual(const SkinnyCall& c, const void* Wt) {
  return c.M <= 32 && gs_skinny_halves(c.N) && few_takes(c, Wt, 8, true) && gs_few_residual_run(c);
}

// The convolution: where every block has a compute unit to itself (three tiles' sums and four channels' taps are 134 registers, 128
// would leave it room for two).
bool gs_few_conv(const SkinnyCall& c, const void* Wt) {
  return c.ex.conv_vec && c.N / 24 <= 256 && few_takes(c, Wt, 8, true) && gs_few_conv_run(c);
}

bool gs_few_parts(const SkinnyCall& c, const void* Wt, int parts) {
  return few_takes(c, Wt, 4, false, parts) && gs_few_parts_run(c, parts);
}
