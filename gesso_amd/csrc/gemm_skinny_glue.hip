// Fills the call record and hands it to the kernels that read rows or tiles.
#include "gemm_skinny_decl.h"
#include "gemm_skinny_impl.h"

void gs_skinny_plain_rows(const SkinnyCall& c);
void gs_skinny_residual_rows(const SkinnyCall& c);
void gs_skinny_conv_rows(const SkinnyCall& c);
void gs_skinny_plain_tiles(const SkinnyCall& c);
void gs_skinny_plain_half_tiles(const SkinnyCall& c);
void gs_skinny_gated_tiles(const SkinnyCall& c);
void gs_skinny_residual_tiles(const SkinnyCall& c);
void gs_skinny_residual_half_tiles(const SkinnyCall& c);
void gs_skinny_conv_tiles(const SkinnyCall& c);
void gs_skinny_parts_rows(const SkinnyCall& c, int parts);
void gs_skinny_parts_tiles(const SkinnyCall& c, int parts);
void gs_skinny_conv_half_tiles(const SkinnyCall& c);

// The tile-major weight and a K that a block's wavefronts share evenly (gemm_few.hip); false: left to the kernels above.
bool gs_few_plain(const SkinnyCall& c, const void* Wt, bool half);
bool gs_few_gated(const SkinnyCall& c, const void* Wt);
bool gs_few_residual(const SkinnyCall& c, const void* Wt);
bool gs_few_conv(const SkinnyCall& c, const void* Wt);
bool gs_few_parts(const SkinnyCall& c, const void* Wt, int parts);

static SkinnyCall base(const void* X, int ldx, int x_tiled, const void* W, const void* Wt, void* Y, int y_dtype, int ldy, int M,
                       int N, int K, int epilogue, hipStream_t stream) {
  SkinnyCall c = {};
  c.ex.x_tiled = x_tiled;
  c.x = (const bf16*)X; c.ldx = ldx; c.w = (const bf16*)(Wt ? Wt : W); c.Y = Y; c.y_dtype = y_dtype; c.ldy = ldy;
  c.M = M; c.N = N; c.K = K; c.epilogue = epilogue; c.stream = stream;
  return c;
}

static void lazy(SkinnyCall& c, const float* res, const float* ssq, int nb, const float* norm_w, float eps) {
  c.ex.res = res; c.ex.ssq = ssq; c.ex.nb = nb; c.ex.norm_w = norm_w; c.ex.eps = eps;
}

// A weight of few rows is shared out in half tiles, so that twice as many blocks stream it.
bool gs_skinny_halves(int N) { return N % 16 == 0 && N / 16 <= 160; }

void gs_skinny_run_plain(const void* X, int ldx, int x_tiled, const float* res, const float* ssq, int nb, const float* norm_w,
                         float eps, const void* W, const void* Wt, void* Y, int y_dtype, int ldy, int M, int N, int K,
                         int epilogue, int y_tiled, hipStream_t stream, int squared) {
  SkinnyCall c = base(X, ldx, x_tiled, W, Wt, Y, y_dtype, ldy, M, N, K, epilogue, stream);
  c.ex.y_tiled = y_tiled;
  c.ex.squared = squared;
  if (res || ssq) lazy(c, res, ssq, nb, norm_w, eps);
  // Half tiles (the same bits) where a block of eight weight rows still comes once to a compute unit and K is long enough for the
  // sum over the wavefronts not to bind.  Cold weights, microseconds in half and in whole tiles of gemm_few_impl.h's kernel: 1 row of 2048 x
  // 8192 8.0 and 10.1, of 1024 x 4608 5.2 and 6.5, of 2048 x 2048 3.8 and 4.1, of 1360 x 2048 3.4 and 3.7; 8 rows the same; 16 10.0 and
  // 11.5, 6.6 and 7.5, 4.3 and 4.6, 3.8 and 4.2; 32 13.2 and 15.0, 8.3 and 9.4, 5.2 and 5.9, 4.5 and 5.0, weighted for their norm 14.6 and
  // 16.3, 9.4 and 10.4, 6.4 and 6.9, 5.7 and 6.1; beyond 32 the blocks' reading of X outweighs the rest.  In whole tiles K below 2048 (2048 x
  // 1024 of 1 row 3.05 both, of 32 3.65 and 3.75, of 1024 x 1024 3.25 both) and more than 256 blocks (1 row of 2064 x 2048 4.4 and 4.1, 8 of
  // 2560 x 2560 5.6 and 5.1, 32 of it 9.2 and 7.0, of 2304 x 4608 14.3 and 10.05).  Another K goes to gemm_skinny_impl.h's kernel, in halves
  // from four rows on (1 row of 1024 x 3072 7.3 and 7.1).
  const bool half = Wt && epilogue == 0 && N % 16 == 0 && N <= 2048 && K >= 2048 && M <= 32;
  if (gs_few_plain(c, Wt, half)) return;
  if (half && M >= 4) gs_skinny_plain_half_tiles(c);
  else Wt ? gs_skinny_plain_tiles(c) : gs_skinny_plain_rows(c);
}

void gs_skinny_run_gated(const void* X, int ldx, int x_tiled, const void* Wt, const float* bias, int act, void* Y, int y_tiled, int M,
                         int N, int K, hipStream_t stream) {
  SkinnyCall c = base(X, ldx, x_tiled, Wt, Wt, Y, GS_BF16, N / 2, M, N, K, 4, stream);
  c.ex.y_tiled = y_tiled;
  c.ex.act_bias = bias;
  c.ex.act = act;
  if (!gs_few_gated(c, Wt)) gs_skinny_gated_tiles(c);
}

void gs_skinny_run_residual(const void* X, int ldx, int x_tiled, const void* W, const void* Wt, float* res, float* ssq_out,
                            const float* next_w, void* xs_out, int xs_tiled, int M, int N, int K, hipStream_t stream) {
  SkinnyCall c = base(X, ldx, x_tiled, W, Wt, nullptr, GS_F32, N, M, N, K, 2, stream);
  c.ex.y_tiled = xs_tiled;
  c.ex.res_out = res; c.ex.ssq_out = ssq_out; c.ex.next_w = next_w; c.ex.xs_out = (bf16*)xs_out;
  if (gs_few_residual(c, Wt)) return;
  if (Wt && gs_skinny_halves(N)) gs_skinny_residual_half_tiles(c);
  else Wt ? gs_skinny_residual_tiles(c) : gs_skinny_residual_rows(c);
}

void gs_skinny_run_conv(const void* X, int ldx, int x_tiled, const float* res, const float* ssq, int nb, const float* norm_w, float eps, const void* W,
                        const void* Wt, const float* taps, const float* conv_bias, float* state, const int* slots,
                        int conv_w, void* Y, int y_tiled, int M, int H, int K, hipStream_t stream) {
  SkinnyCall c = base(X, ldx, x_tiled, W, Wt, Y, GS_BF16, H, M, 3 * H, K, 3, stream);
  c.ex.y_tiled = y_tiled;
  if (res || ssq) lazy(c, res, ssq, nb, norm_w, eps);
  c.ex.taps = taps; c.ex.conv_bias = conv_bias; c.ex.state = state; c.ex.slots = slots; c.ex.conv_w = conv_w;
  c.ex.conv_vec = conv_w >= 2 && conv_w <= 4 && H % 4 == 0 && H >= 4 &&
                  (((uintptr_t)taps | (uintptr_t)conv_bias | (uintptr_t)state) & 15) == 0;
  if (gs_few_conv(c, Wt)) return;
  // c.N / 3 channels, as few as a narrow weight's rows (6144 x 2048, in whole and in half tiles: 8 rows 9.5 and 8.4 us, 40 10.9 and
  // 10.1, 64 12.7 and 11.9)
  if (Wt && gs_skinny_halves(c.N / 3)) gs_skinny_conv_half_tiles(c);
  else Wt ? gs_skinny_conv_tiles(c) : gs_skinny_conv_rows(c);
}

void gs_skinny_run_parts(const void* X, int ldx, int x_tiled, const void* W, const void* Wt, float* part, int parts, int M, int N,
                         int K, hipStream_t stream) {
  SkinnyCall c = base(X, ldx, x_tiled, W, Wt, part, GS_F32, N, M, N, K, 5, stream);
  if (gs_few_parts(c, Wt, parts)) return;
  Wt ? gs_skinny_parts_tiles(c, parts) : gs_skinny_parts_rows(c, parts);
}
