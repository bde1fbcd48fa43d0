// Y (M, N) = X (M, K) . W (N, K)^T for M <= 64 rows and the tile-major weight, K shared evenly: the products of a decode step.
//
// What binds it: the weight's bytes (5.5 to 6 TB/s), and before and after them the kernel's own chain: its arguments, the first
// loads' way, the wavefronts' sums, the epilogue.  So the code is one straight line: the epilogue's operands are asked for by the
// wavefront that runs it, and the rows' partial sums of squares; then the weight's and the rows' first loads, behind no load's arrival
// and no branch (the compiler waits for every load in flight where a branch hides how many there are); and only then does the first
// product wait.
// Arithmetic and order of sums are gemm_skinny_impl.h's, bit for bit: a block's wavefronts share K evenly, each adds its steps of 32 one
// after another, and the wavefronts' tiles are added in their order.
//
// A block owns R tiles of 16 weight rows, or R halves of 8 (HALF) where a weight has few rows.  A load of halves brings the eight rows
// at two steps of K, and the second step's rows come to the first's lanes by a move within rows of 16 lanes.
//
// Measured on cold weights in a graph, 8 rows, microseconds in gemm_skinny_impl.h's kernel, here, and a plain read of as many bytes:
// into the stream 2048 x 8192 9.0, 8.0 and 6.5, 2048 x 7168 8.75 and 7.5, 2048 x 2048 4.65, 4.0 and 4.05, 1024 x 4608 6.6, 5.3 and 4.0,
// 1024 x 1024 3.7 and 3.2; the convolution's product of 6144 x 2048 7.9, 6.8 and 6.7, 3072 x 1024 5.75, 4.4 and 3.4; gate and up of
// 16384 x 2048 12.4, 12.2 and 11.8, 9216 x 1024 6.9, 6.55 and 4.5 (288 blocks: some units have two); q, k and v of 3072 x 2048 5.15 and
// 4.6; the head of 65536 x 2048 42.4 and 41.5.  Of what that took: loads twice as wide for halves; the epilogue's operands asked for
// before the weight by its one wavefront (after it, or by all eight: 1024 x 4608 5.8); no load behind another's arrival (the
// convolution's slots came by three scalar loads one after another, before the weight).
// More rows, microseconds of a decode step's kernels before and now, 64 rows of 2,048 wide: gate and up of 16384 x 2048 16.1 and 15.0,
// K in eight parts of 2048 x 8192 12.3 and 11.5, of 2048 x 2048 5.9 and 5.2,
// the convolution's product 12.3 and 10.5, q, k and v 8.0 and 7.4.  There each block brings in all rows of X beside its weight.
#pragma once
#include "gemm_skinny_impl.h"

typedef __attribute__((ext_vector_type(4))) int i32x4_t;

struct FewArgs {
  const bf16* W;         // tile-major; K a multiple of a block's wavefronts' steps of 32 (halves: of pairs of steps)
  const bf16* X;
  int M, N, K;
  int xrow, xgroup, xstep;   // elements of X from a row to the next, from eight columns to the next, from a step of K to the next
  const float* ssq;      // SCALED: (M, nb) partial sums of squares; the rows are weighted for their norm and not yet scaled
  int nb;
  float eps;
  void* Y;
  int ldy;
  int tiled;             // Y (EPI 1, 3, 4) or xs (EPI 2) are written as tiled rows
  int extra;             // EPI 0: columns stored as the square of their relu; EPI 4: the activation
  const int* slots;      // EPI 3: (M)
  // EPI 2: the next norm's weight (N) or null, the stream (M, N) in place, its partial sums of squares (M, blocks); Y: the weighted rows
  // EPI 3: taps (H, CW), state (slots, H, CW - 1), bias (H) or null
  // EPI 4: bias (N) or null
  const float* w;
  float* io;
  float* ssq_out;
  const float* bias;
  int xtile;             // elements of X from a row tile to the next
};

// Rows 8 to 15 of a tile's piece in the places of rows 0 to 7, and the other way round.
__device__ __forceinline__ bf16x8_t other_rows(bf16x8_t v) {
  i32x4_t x = __builtin_bit_cast(i32x4_t, v);
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = __builtin_amdgcn_update_dpp(0, x[i], 0x128, 0xf, 0xf, true);   // row_ror:8
  return __builtin_bit_cast(bf16x8_t, x);
}

// p (the same for every lane) and a lane's own bytes beyond it (a register an address, not two).
__device__ __forceinline__ const bf16* at_bytes(const bf16* p, unsigned bytes) {
  return reinterpret_cast<const bf16*>(reinterpret_cast<const char*>(p) + bytes);
}

// EPI as in gemm_skinny_impl.h: 0 stored, 1 SwiGLU, 2 into the stream, 3 the convolution (of CW taps), 4 gated activation.
// FIRST: loads a weight tile that the first wait covers; the rounds after it take NEXT.
template <int R, int MT, int WAVES, bool HALF, bool SCALED, int EPI, int CW, int FIRST, bool ONCE, typename TOut>
__global__ __launch_bounds__(WAVES * 64, MT == 1 && R == 2 ? WAVES / 2 : 1) void gemm_few_kernel(FewArgs g) {
  static_assert((EPI != 2 && EPI != 3) || HALF, "the stream and the convolution come in halves");
  constexpr bool GLU = EPI == 1 || EPI == 4;
  static_assert(!GLU || (R % 2 == 0 && !HALF), "gate and up come in whole tiles");
  static_assert(WAVES >= MT, "a wavefront finishes a row tile");
  constexpr int S = HALF ? 2 : 1;                        // steps of K a load
  constexpr bool WIDE = MT > 1 && R % 2 == 0;            // (a lane's registers bind)
  constexpr int NEXT = HALF ? (R >= 3 ? 2 : 4) : 8;
  constexpr int ROWS = MT * 16 / WAVES;                  // SCALED: rows whose partial sums a wavefront adds
  extern __shared__ __align__(16) float all_sums[];      // several row tiles: WAVES x R x MT x 256 sums
  __shared__ __align__(16) float one_sums[MT == 1 ? (WAVES - 1) * R * 256 : 4];
  float* red = MT == 1 ? one_sums : all_sums;
  __shared__ float inv_s[MT * 16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, kg = lane >> 4, blk = EPI == 5 ? blockIdx.y : blockIdx.x;
  // the row that this wavefront finishes (a row past M: the last again; its column of the result is never stored)
  const int em = MT > 1 ? wave * 16 + r16 : r16, mc = em < g.M ? em : g.M - 1;
  // EPI 5: part blockIdx.x of K, its blocks' weight tiles along y
  const int ksteps = g.K >> 5, units = ksteps / (WAVES * S * (EPI == 5 ? (int)gridDim.x : 1));
  const int s0 = ((EPI == 5 ? (int)blockIdx.x * WAVES : 0) + wave) * units * S;

  int slot = 0;

  const bf16* wp[R];                                     // the same for every lane
#pragma unroll
  for (int r = 0; r < R; ++r) {
    int tile;
    if (GLU) {
      tile = blk * (R / 2) + (r >> 1);
      if (R > 2 && tile >= g.N >> 5) tile = (g.N >> 5) - 1;
      tile += (r & 1) * (g.N >> 5);
    }
    else if (EPI == 3) tile = (blk >> 1) + r * (g.N / 48);
    else if (HALF) tile = blk >> 1;
    else {
      tile = blk * R + r;                                // (past the last: the last again, never stored)
      if (R > 1 && tile >= g.N >> 4) tile = (g.N >> 4) - 1;
    }
    wp[r] = g.W + ((size_t)tile * ksteps + s0) * 512;
  }
  const unsigned wo = HALF ? (kg * 16 + (blk & 1) * 8 + (r16 & 7)) * 8 + (r16 >> 3) * 512 : lane * 8;
  unsigned xo[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = mt * 16 + r16 < g.M ? mt * 16 + r16 : g.M - 1;
    xo[mt] = (MT > 1 ? (m >> 4) * g.xtile + (m & 15) * g.xrow : m * g.xrow) + kg * g.xgroup;
  }
  const bf16* xp = g.X + (size_t)s0 * g.xstep;

  f32x4_t acc[R][MT];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[r][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  int u0 = 0;
  // C loads a weight tile and the rows' at their steps, what else is asked for, then the products.  (Macros, not closures: arrays that
  // a closure takes by reference are not always kept in registers.)
#define GS_FEW_LOAD(U, AT)                                                                                              \
  {                                                                                                                     \
    _Pragma("unroll") for (int r = 0; r < R; ++r)                                                                       \
      a[U][r] = load8w<ONCE ? SKINNY_ONCE : 0>(WIDE ? at_bytes(wp[r], 2 * wo + (unsigned)(AT) * (S * 1024)) : wp[r] + (size_t)(AT) * (S * 512) + wo); \
    _Pragma("unroll") for (int j = 0; j < S; ++j)                                                                       \
      _Pragma("unroll") for (int mt = 0; mt < MT; ++mt)                                                                 \
        b[U][j][mt] = *reinterpret_cast<const bf16x8_t*>(WIDE ? at_bytes(xp, 2 * (xo[mt] + (unsigned)((AT) * S + j) * g.xstep))  \
                                                                : xp + (size_t)((AT) * S + j) * g.xstep + xo[mt]);      \
  }
#define GS_FEW_MULTIPLY(U)                                                                                             \
  {                                                                                                                     \
    _Pragma("unroll") for (int j = 0; j < S; ++j)                                                                       \
      _Pragma("unroll") for (int r = 0; r < R; ++r) {                                                                   \
        const bf16x8_t w_ = j ? other_rows(a[U][r]) : a[U][r];                                                          \
        _Pragma("unroll") for (int mt = 0; mt < MT; ++mt)                                                               \
          acc[r][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w_, b[U][j][mt], acc[r][mt], 0, 0, 0);                   \
      }                                                                                                                 \
  }
#define GS_FEW_ROUND(C, ...)                                                                                           \
  {                                                                                                                     \
    bf16x8_t a[C][R], b[C][S][MT];                                                                                      \
    _Pragma("unroll") for (int u = 0; u < C; ++u) GS_FEW_LOAD(u, u0 + u)                                                \
    __builtin_amdgcn_sched_barrier(0);                                                                                  \
    __VA_ARGS__                                                                                                         \
    _Pragma("unroll") for (int u = 0; u < C; ++u) GS_FEW_MULTIPLY(u)                                                    \
    u0 += C;                                                                                                            \
  }
  float pre[ROWS > 0 ? ROWS : 1][4];
  f32x4_t rold, nextw, gbias[R];
  f32x4_t tq[CW], hq[CW > 1 ? CW - 1 : 1], cb;
  const int H = EPI == 3 ? g.N / 3 : 0;
  const int n0 = HALF ? blk * 8 + (kg & 1) * 4 : blk * 16 * (GLU ? R / 2 : R) + kg * 4;   // this lane's first column (halves: of kg 0 and 1)
  // What the epilogue reads besides the product is asked for before the weight, by the wavefront that runs it.
  if (wave < MT) {
    if (EPI == 2) {
      rold = *reinterpret_cast<const f32x4_t*>(g.io + (size_t)mc * g.N + n0);
      nextw = *reinterpret_cast<const f32x4_t*>(g.w ? g.w + n0 : g.io + n0);
    }
    if (EPI == 3) {
      // four channels' taps and history are runs of memory: a row of CW and of CW - 1 pieces of 16 bytes
      slot = g.slots[mc];
#pragma unroll
      for (int q = 0; q < CW; ++q) tq[q] = *reinterpret_cast<const f32x4_t*>(g.w + (size_t)n0 * CW + 4 * q);
      cb = *reinterpret_cast<const f32x4_t*>((g.bias ? g.bias : g.w) + n0);
    }
    if (EPI == 4) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        gbias[r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if (g.bias) gbias[r] = *reinterpret_cast<const f32x4_t*>(g.bias + n0 + (r & 1 ? g.N >> 1 : 0));
      }
    }
  }
  if (SCALED) {
    // the partial sums of this wavefront's rows (one that does not exist is read from one that does, and not counted)
#pragma unroll
    for (int i = 0; i < ROWS; ++i) if (MT > 1 || i == 0 || g.M > WAVES) {
      const int m = wave + i * WAVES;
      const float* row = g.ssq + (size_t)(m < g.M ? m : g.M - 1) * g.nb;
#pragma unroll
      for (int j = 0; j < 4; ++j) pre[i][j] = row[lane + 64 * j < g.nb ? lane + 64 * j : 0];
    }
  }
#define GS_FEW_HISTORY                                                                                                 \
  if (EPI == 3 && wave < MT) {                                                                                          \
    const float* hp = g.io + ((size_t)slot * H + n0) * (CW - 1);                                                        \
    _Pragma("unroll") for (int q = 0; q < CW - 1; ++q) hq[q] = *reinterpret_cast<const f32x4_t*>(hp + 4 * q);           \
  }
  if constexpr (MT == 1) {
    GS_FEW_ROUND(FIRST, GS_FEW_HISTORY)
    while (u0 + NEXT <= units) GS_FEW_ROUND(NEXT, )
    if (NEXT > 4 && u0 + 4 <= units) GS_FEW_ROUND(4, )
    if (NEXT == 4 && u0 + 3 <= units) GS_FEW_ROUND(3, )
    if (NEXT > 2 && u0 + 2 <= units) GS_FEW_ROUND(2, )
    if (u0 < units) GS_FEW_ROUND(1, )
  } else {
    // several row tiles: the rows' bytes bind, so a place in the ring is asked for again as soon as it is multiplied
    {
      bf16x8_t a[FIRST][R], b[FIRST][S][MT];
#pragma unroll
      for (int u = 0; u < FIRST; ++u) GS_FEW_LOAD(u, u)
      __builtin_amdgcn_sched_barrier(0);
      GS_FEW_HISTORY
      for (u0 = FIRST; u0 + FIRST <= units; u0 += FIRST) {
#pragma unroll
        for (int u = 0; u < FIRST; ++u) {
          GS_FEW_MULTIPLY(u)
          GS_FEW_LOAD(u, u0 + u)
        }
      }
#pragma unroll
      for (int u = 0; u < FIRST; ++u) GS_FEW_MULTIPLY(u)
    }
    if (FIRST > 2 && u0 + 2 <= units) GS_FEW_ROUND(2, )
    if (FIRST > 1 && u0 < units) GS_FEW_ROUND(1, )
  }
#undef GS_FEW_HISTORY
#undef GS_FEW_ROUND
#undef GS_FEW_MULTIPLY
#undef GS_FEW_LOAD

  if (SCALED) {
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      const int m = wave + i * WAVES;
#pragma unroll
      for (int j = 0; j < 4; ++j) pre[i][j] = lane + 64 * j < g.nb ? pre[i][j] : 0.f;
      float ss = MT == 1 && i ? ((pre[i][0] + pre[i][1]) + pre[i][2]) + pre[i][3] : (pre[i][0] + pre[i][1]) + (pre[i][2] + pre[i][3]);
      if (m < g.M) {
        for (int b = 256 + lane; b < g.nb; b += 64) ss += g.ssq[(size_t)m * g.nb + b];
        ss = wave_sum_dpp(ss);
        if (lane == 0) inv_s[m] = norm_inverse(ss, (float)g.K, g.eps);
      }
    }
  }
  f32x4_t sum[R];
  if constexpr (MT == 1) {
    if (wave > 0) {
#pragma unroll
      for (int r = 0; r < R; ++r) *reinterpret_cast<f32x4_t*>(red + (((wave - 1) * R + r) * 64 + lane) * 4) = acc[r][0];
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int r = 0; r < R; ++r) sum[r] = acc[r][0];
#pragma unroll
    for (int w = 0; w < WAVES - 1; ++w)
#pragma unroll
      for (int r = 0; r < R; ++r) sum[r] += *reinterpret_cast<const f32x4_t*>(red + ((w * R + r) * 64 + lane) * 4);
  } else {
    // wavefront w finishes row tile w: its own part of it from registers, the others' from LDS, in their order
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      if (wave != mt) {
#pragma unroll
        for (int r = 0; r < R; ++r) *reinterpret_cast<f32x4_t*>(red + (((wave * R + r) * MT + mt) * 64 + lane) * 4) = acc[r][mt];
      }
    __syncthreads();
    if (wave >= MT) return;
    f32x4_t own[R];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      if (wave == mt) {
#pragma unroll
        for (int r = 0; r < R; ++r) own[r] = acc[r][mt];
      }
    const float* src = red + (wave * 64 + lane) * 4;
#pragma unroll
    for (int w = 0; w < WAVES; ++w)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        f32x4_t v = own[r];
        if (w >= MT || w != wave) v = *reinterpret_cast<const f32x4_t*>(src + (size_t)(w * R + r) * MT * 256);
        if (w == 0) sum[r] = v; else sum[r] += v;
      }
  }
  if (SCALED) {
    const float iv = inv_s[mc];
#pragma unroll
    for (int r = 0; r < R; ++r) sum[r] *= iv;
  }

  // lane l holds, for row l % 16 of the wavefront's row tile, columns 4 (l / 16) + 0..3 of every tile (halves: of kg 0 and 1)
  const bool live = em < g.M && (!HALF || kg < 2);
  if constexpr (EPI == 0 || EPI == 5) {
    if (!live) return;
    TOut* Y = reinterpret_cast<TOut*>(g.Y) + (EPI == 5 ? (size_t)blockIdx.x * g.M * g.ldy : 0);   // (a sheet a part)
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int n = n0 + 16 * r;
      if (EPI == 0 && n < g.extra) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float z = to_f32(f32_to_bf16(sum[r][i])), v = z > 0.f ? z : 0.f;
          if (n + i < g.extra) sum[r][i] = v * v;
        }
      }
      if (n < g.N) store4<TOut>(Y + (size_t)em * g.ldy + n, sum[r], 4);
    }
  } else if constexpr (GLU) {
    if (!live) return;
#pragma unroll
    for (int r = 0; r < R; r += 2) {
      const int n = n0 + 8 * r;
      f32x4_t o;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (EPI == 1) o[i] = sum[r][i] / (1.0f + expf(-sum[r][i])) * sum[r + 1][i];
        else o[i] = gated_act(to_f32(f32_to_bf16(sum[r][i])) + gbias[r][i], g.extra) * (to_f32(f32_to_bf16(sum[r + 1][i])) + gbias[r + 1][i]);
      }
      if (R == 2 || n < g.N >> 1) store4<TOut>(reinterpret_cast<TOut*>(g.Y) + (g.tiled ? tiled_index(em, n, MT) : (size_t)em * g.ldy + n), o, 4);
    }
  } else if constexpr (EPI == 2) {
    // every lane takes part in the exchange, live or not
    float ss = 0.f;
    if (live) {
      f32x4_t nv, xv;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        // (the product is rounded to bfloat16 first, as a pass of its own would find it)
        nv[i] = rold[i] + to_f32(f32_to_bf16(sum[0][i]));
        ss = __builtin_fmaf(nv[i], nv[i], ss);
        xv[i] = nv[i] * nextw[i];
      }
      *reinterpret_cast<f32x4_t*>(g.io + (size_t)em * g.N + n0) = nv;
      if (g.Y) store4<bf16>(reinterpret_cast<bf16*>(g.Y) + (g.tiled ? tiled_index(em, n0, MT) : (size_t)em * g.N + n0), xv, 4);
    }
    ss += __shfl_xor(ss, 16, 64);
    ss += __shfl_xor(ss, 32, 64);
    if (live && kg == 0) g.ssq_out[(size_t)em * gridDim.x + blk] = ss;
  } else {
    if (!live) return;
    f32x4_t out, nh[CW - 1];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float Bv = to_f32(f32_to_bf16(sum[0][i])), Cv = to_f32(f32_to_bf16(sum[R > 1 ? 1 : 0][i])), Xv = to_f32(f32_to_bf16(sum[R > 2 ? 2 : 0][i]));
      const float u = Bv * Xv;
      float y = 0.f;
#pragma unroll
      for (int p = 0; p < CW - 1; ++p) y += tq[(i * CW + p) / 4][(i * CW + p) % 4] * hq[(i * (CW - 1) + p) / 4][(i * (CW - 1) + p) % 4];
      y += tq[(i * CW + CW - 1) / 4][(i * CW + CW - 1) % 4] * u;
      if (g.bias) y += cb[i];
      out[i] = Cv * y;
#pragma unroll
      for (int p = 0; p < CW - 1; ++p) {
        const int at = i * (CW - 1) + p;
        nh[at / 4][at % 4] = p < CW - 2 ? hq[(at + 1) / 4][(at + 1) % 4] : u;
      }
    }
    store4<TOut>(reinterpret_cast<TOut*>(g.Y) + (g.tiled ? tiled_index(em, n0, MT) : (size_t)em * g.ldy + n0), out, 4);
    float* hp = g.io + ((size_t)slot * H + n0) * (CW - 1);
#pragma unroll
    for (int q = 0; q < CW - 1; ++q) *reinterpret_cast<f32x4_t*>(hp + 4 * q) = nh[q];
  }
}

// Where a wavefront's loads start: in halves four, or five where one would be left over (a round trip of its own: 1024 x 4608, nine
// loads a wavefront, 5.6 and 5.3 us), or all there are; three tiles' halves two (as good as four) or, of three, all; whole tiles eight,
// four, two or one.
static inline int few_first(int units, bool half, bool three) {
  if (!half) return units >= 8 ? 8 : units >= 4 ? 4 : units >= 2 ? 2 : 1;
  if (three) return units == 3 ? 3 : units >= 2 ? 2 : 1;
  return units >= 4 ? (units % 4 == 1 ? 5 : 4) : units;
}

template <int R, int MT, int WAVES, bool HALF, bool SCALED, int EPI, int CW, int FIRST, bool ONCE, typename TOut>
static void launch_few_first(dim3 grid, const FewArgs& g, hipStream_t stream) {
  const size_t lds = MT > 1 ? (size_t)WAVES * R * MT * 256 * sizeof(float) : 0;
  const auto kernel = &gemm_few_kernel<R, MT, WAVES, HALF, SCALED, EPI, CW, FIRST, ONCE, TOut>;
  if (lds > 64 * 1024) {
    // more than the default limit of dynamic LDS: asked for once per kernel
    static const hipError_t asked = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    (void)asked;
  }
  kernel<<<grid, WAVES * 64, lds, stream>>>(g);
}

// LEAST: what callers' rules leave of K is that many loads a wavefront or more; shorter starts are not compiled (a call that had fewer
// would come back false, nothing launched).
template <int R, int MT, int WAVES, bool HALF, bool SCALED, int EPI, int CW, bool ONCE, typename TOut, int LEAST = 1>
static bool launch_few(dim3 grid, const FewArgs& g, hipStream_t stream) {
  const int units = (g.K >> 5) / (WAVES * (HALF ? 2 : 1) * (EPI == 5 ? (int)grid.x : 1));
#define GS_FEW(F, COMPILED)                                                                               \
  if constexpr (COMPILED) {                                                                               \
    launch_few_first<R, MT, WAVES, HALF, SCALED, EPI, CW, F, ONCE, TOut>(grid, g, stream);                \
    return true;                                                                                          \
  }
  if constexpr (MT > 1) {
    // (a ring of four loads a weight tile, three tiles' halves and four tiles of two: what a lane's registers hold beside the sums)
    if (units >= 4 && R < 3) { GS_FEW(4, R < 3) }
    else if (units >= 2) { GS_FEW(2, R >= 3 || LEAST < 4) }
    else { GS_FEW(1, LEAST < 2) }
  } else {
    switch (few_first(units, HALF, R >= 3)) {
      case 1: GS_FEW(1, LEAST < 2) break;
      case 2: GS_FEW(2, HALF ? R >= 3 || LEAST < 3 : LEAST < 4) break;
      case 3: GS_FEW(3, HALF && LEAST < 4) break;
      case 4: GS_FEW(4, R < 3) break;
      case 5: GS_FEW(5, HALF && R < 3) break;
      default: GS_FEW(8, !HALF) break;
    }
  }
  return false;
#undef GS_FEW
}

// By row tiles: one to MOST of them, in blocks of W12 wavefronts (one and two) and W34.
template <int R, int W12, int W34, int MOST, bool HALF, bool SCALED, int EPI, int CW, bool ONCE, typename TOut, int LEAST = 1, int LEAST34 = LEAST>
static bool launch_few_rows(dim3 grid, const FewArgs& g, hipStream_t stream) {
  switch ((g.M + 15) / 16) {
    case 1: return launch_few<R, 1, W12, HALF, SCALED, EPI, CW, ONCE, TOut, LEAST>(grid, g, stream);
    case 2: return launch_few<R, 2, W12, HALF, SCALED, EPI, CW, ONCE, TOut, LEAST>(grid, g, stream);
    case 3: if constexpr (MOST >= 3) return launch_few<R, 3, W34, HALF, SCALED, EPI, CW, ONCE, TOut, LEAST34>(grid, g, stream); break;
    default: if constexpr (MOST >= 4) return launch_few<R, 4, W34, HALF, SCALED, EPI, CW, ONCE, TOut, LEAST34>(grid, g, stream); break;
  }
  return false;
}

// Between the entry points (gemm_skinny_glue.hip) and the launches (gemm_few.hip, gemm_few_glu.hip, gemm_few_block.hip).
FewArgs few_args(const SkinnyCall& c);
bool gs_skinny_halves(int N);
int few_glu_waves(const SkinnyCall& c);
bool gs_few_swiglu(const SkinnyCall& c);
bool gs_few_gated_run(const SkinnyCall& c);
bool gs_few_residual_run(const SkinnyCall& c);
bool gs_few_conv_run(const SkinnyCall& c);
bool gs_few_parts_run(const SkinnyCall& c, int parts);
