// Y (M, N) = X (M, K) . W (N, K)^T for M <= 16 rows and the tile-major weight: the products of a decode step of few requests.
//
// What binds it: the weight's bytes (5.5 to 6 TB/s), and before and after them the kernel's own chain: its arguments, the first
// loads' way, the wavefronts' sums, the epilogue.  So the code is one straight line: the weight's and the rows' first loads are asked
// for as soon as the arguments are there, then what the epilogue and the rows' norm need, by every wavefront and behind no branch (the
// compiler waits for every load in flight where a branch hides how many there are), and only then the first product waits.
// Arithmetic and order of sums are gemm_skinny_impl.h's, bit for bit: eight wavefronts share K evenly, each adds its steps of 32 one
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
#pragma once
#include "gemm_skinny_impl.h"

typedef __attribute__((ext_vector_type(4))) int i32x4_t;

#define FEW_WAVES 8

struct FewArgs {
  const bf16* W;         // tile-major; K a multiple of FEW_WAVES steps of 32 (halves: of pairs of steps)
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
};

// Rows 8 to 15 of a tile's piece in the places of rows 0 to 7, and the other way round.
__device__ __forceinline__ bf16x8_t other_rows(bf16x8_t v) {
  i32x4_t x = __builtin_bit_cast(i32x4_t, v);
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = __builtin_amdgcn_update_dpp(0, x[i], 0x128, 0xf, 0xf, true);   // row_ror:8
  return __builtin_bit_cast(bf16x8_t, x);
}

// EPI as in gemm_skinny_impl.h: 0 stored, 1 SwiGLU, 2 into the stream, 3 the convolution (of CW taps), 4 gated activation.
// FIRST: loads a weight tile that the first wait covers; the rounds after it take NEXT.
template <int R, bool HALF, bool SCALED, int EPI, int CW, int FIRST, bool ONCE, typename TOut>
__global__ __launch_bounds__(FEW_WAVES * 64, R == 2 ? FEW_WAVES / 2 : 1) void gemm_few_kernel(FewArgs g) {
  static_assert((EPI != 2 && EPI != 3) || HALF, "the stream and the convolution come in halves");
  constexpr bool GLU = EPI == 1 || EPI == 4;
  static_assert(!GLU || (R == 2 && !HALF), "gate and up come as a tile each");
  constexpr int S = HALF ? 2 : 1;                        // steps of K a load
  constexpr int NEXT = HALF ? (R >= 3 ? 2 : 4) : 8;
  __shared__ __align__(16) float red[(FEW_WAVES - 1) * R * 256];
  __shared__ float inv_s[16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, kg = lane >> 4, blk = blockIdx.x;
  const int mc = r16 < g.M ? r16 : g.M - 1;              // (a row past M: the last again; its column of the result is never stored)
  const int ksteps = g.K >> 5, units = ksteps / (FEW_WAVES * S), s0 = wave * units * S;

  int slot = 0;

  const bf16* wp[R];                                     // the same for every lane
#pragma unroll
  for (int r = 0; r < R; ++r) {
    int tile;
    if (GLU) tile = blk + r * (g.N >> 5);
    else if (EPI == 3) tile = (blk >> 1) + r * (g.N / 48);
    else if (HALF) tile = blk >> 1;
    else {
      tile = blk * R + r;                                // (past the last: the last again, never stored)
      if (R > 1 && tile >= g.N >> 4) tile = (g.N >> 4) - 1;
    }
    wp[r] = g.W + ((size_t)tile * ksteps + s0) * 512;
  }
  const unsigned wo = HALF ? (kg * 16 + (blk & 1) * 8 + (r16 & 7)) * 8 + (r16 >> 3) * 512 : lane * 8;
  const unsigned xo = mc * g.xrow + kg * g.xgroup;
  const bf16* xp = g.X + (size_t)s0 * g.xstep;

  f32x4_t acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  int u0 = 0;
  // C loads a weight tile and the rows' at their steps, what else is asked for, then the products.  (Macros, not closures: arrays that
  // a closure takes by reference are not always kept in registers.)
#define GS_FEW_ROUND(C, ...)                                                                                           \
  {                                                                                                                     \
    bf16x8_t a[C][R], b[C][S];                                                                                          \
    _Pragma("unroll") for (int u = 0; u < C; ++u) {                                                                     \
      _Pragma("unroll") for (int r = 0; r < R; ++r) a[u][r] = load8w<ONCE ? SKINNY_ONCE : 0>(wp[r] + (size_t)(u0 + u) * (S * 512) + wo); \
      _Pragma("unroll") for (int j = 0; j < S; ++j)                                                                     \
        b[u][j] = *reinterpret_cast<const bf16x8_t*>(xp + (size_t)((u0 + u) * S + j) * g.xstep + xo);                     \
    }                                                                                                                   \
    __builtin_amdgcn_sched_barrier(0);                                                                                  \
    __VA_ARGS__                                                                                                         \
    _Pragma("unroll") for (int u = 0; u < C; ++u)                                                                       \
      _Pragma("unroll") for (int j = 0; j < S; ++j)                                                                     \
        _Pragma("unroll") for (int r = 0; r < R; ++r)                                                                   \
          acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(j ? other_rows(a[u][r]) : a[u][r], b[u][j], acc[r], 0, 0, 0); \
    u0 += C;                                                                                                            \
  }
  float pre[2][4];
  f32x4_t rold, nextw, gbias[2];
  f32x4_t tq[CW], hq[CW > 1 ? CW - 1 : 1], cb;
  const int H = EPI == 3 ? g.N / 3 : 0;
  const int n0 = HALF ? blk * 8 + (kg & 1) * 4 : blk * 16 * (GLU ? 1 : R) + kg * 4;   // this lane's first column (halves: of kg 0 and 1)
  // What the epilogue reads besides the product is asked for before the weight, by the wavefront that runs it.
  if (wave == 0) {
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
      for (int r = 0; r < 2; ++r) {
        gbias[r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if (g.bias) gbias[r] = *reinterpret_cast<const f32x4_t*>(g.bias + n0 + (r ? g.N >> 1 : 0));
      }
    }
  }
  if (SCALED) {
    // the partial sums of this wavefront's rows (one that does not exist is read from one that does, and not counted)
#pragma unroll
    for (int i = 0; i < 2; ++i) if (i == 0 || g.M > FEW_WAVES) {
      const int m = wave + i * FEW_WAVES;
      const float* row = g.ssq + (size_t)(m < g.M ? m : g.M - 1) * g.nb;
#pragma unroll
      for (int j = 0; j < 4; ++j) pre[i][j] = row[lane + 64 * j < g.nb ? lane + 64 * j : 0];
    }
  }
  GS_FEW_ROUND(FIRST, if (EPI == 3 && wave == 0) {
    const float* hp = g.io + ((size_t)slot * H + n0) * (CW - 1);
    _Pragma("unroll") for (int q = 0; q < CW - 1; ++q) hq[q] = *reinterpret_cast<const f32x4_t*>(hp + 4 * q);
  })
  while (u0 + NEXT <= units) GS_FEW_ROUND(NEXT, )
  if (NEXT > 4 && u0 + 4 <= units) GS_FEW_ROUND(4, )
  if (NEXT == 4 && u0 + 3 <= units) GS_FEW_ROUND(3, )
  if (NEXT > 2 && u0 + 2 <= units) GS_FEW_ROUND(2, )
  if (u0 < units) GS_FEW_ROUND(1, )
#undef GS_FEW_ROUND

  if (SCALED) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int m = wave + i * FEW_WAVES;
#pragma unroll
      for (int j = 0; j < 4; ++j) pre[i][j] = lane + 64 * j < g.nb ? pre[i][j] : 0.f;
      float ss = i ? ((pre[i][0] + pre[i][1]) + pre[i][2]) + pre[i][3] : (pre[i][0] + pre[i][1]) + (pre[i][2] + pre[i][3]);
      if (m < g.M) {
        for (int b = 256 + lane; b < g.nb; b += 64) ss += g.ssq[(size_t)m * g.nb + b];
        ss = wave_sum_dpp(ss);
        if (lane == 0) inv_s[m] = norm_inverse(ss, (float)g.K, g.eps);
      }
    }
  }
  if (wave > 0) {
#pragma unroll
    for (int r = 0; r < R; ++r) *reinterpret_cast<f32x4_t*>(red + (((wave - 1) * R + r) * 64 + lane) * 4) = acc[r];
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int w = 0; w < FEW_WAVES - 1; ++w)
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] += *reinterpret_cast<const f32x4_t*>(red + ((w * R + r) * 64 + lane) * 4);
  if (SCALED) {
    const float iv = inv_s[mc];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] *= iv;
  }

  // lane l holds, for row l % 16, columns 4 (l / 16) + 0..3 of every tile (halves: of kg 0 and 1)
  const bool live = r16 < g.M && (!HALF || kg < 2);
  if constexpr (EPI == 0) {
    if (!live) return;
    TOut* Y = reinterpret_cast<TOut*>(g.Y);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int n = n0 + 16 * r;
      if (n < g.extra) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float z = to_f32(f32_to_bf16(acc[r][i])), v = z > 0.f ? z : 0.f;
          if (n + i < g.extra) acc[r][i] = v * v;
        }
      }
      if (n < g.N) store4<TOut>(Y + (size_t)r16 * g.ldy + n, acc[r], 4);
    }
  } else if constexpr (GLU) {
    if (!live) return;
    f32x4_t o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (EPI == 1) o[i] = acc[0][i] / (1.0f + expf(-acc[0][i])) * acc[R - 1][i];
      else o[i] = gated_act(to_f32(f32_to_bf16(acc[0][i])) + gbias[0][i], g.extra) * (to_f32(f32_to_bf16(acc[R - 1][i])) + gbias[1][i]);
    }
    store4<TOut>(reinterpret_cast<TOut*>(g.Y) + (g.tiled ? tiled_index(r16, n0, 1) : (size_t)r16 * g.ldy + n0), o, 4);
  } else if constexpr (EPI == 2) {
    // every lane takes part in the exchange, live or not
    float ss = 0.f;
    if (live) {
      f32x4_t nv, xv;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        // (the product is rounded to bfloat16 first, as a pass of its own would find it)
        nv[i] = rold[i] + to_f32(f32_to_bf16(acc[0][i]));
        ss = __builtin_fmaf(nv[i], nv[i], ss);
        xv[i] = nv[i] * nextw[i];
      }
      *reinterpret_cast<f32x4_t*>(g.io + (size_t)r16 * g.N + n0) = nv;
      if (g.Y) store4<bf16>(reinterpret_cast<bf16*>(g.Y) + (g.tiled ? tiled_index(r16, n0, 1) : (size_t)r16 * g.N + n0), xv, 4);
    }
    ss += __shfl_xor(ss, 16, 64);
    ss += __shfl_xor(ss, 32, 64);
    if (live && kg == 0) g.ssq_out[(size_t)r16 * gridDim.x + blk] = ss;
  } else {
    if (!live) return;
    f32x4_t out, nh[CW - 1];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float Bv = to_f32(f32_to_bf16(acc[0][i])), Cv = to_f32(f32_to_bf16(acc[R > 1 ? 1 : 0][i])), Xv = to_f32(f32_to_bf16(acc[R > 2 ? 2 : 0][i]));
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
    store4<TOut>(reinterpret_cast<TOut*>(g.Y) + (g.tiled ? tiled_index(r16, n0, 1) : (size_t)r16 * g.ldy + n0), out, 4);
    float* hp = g.io + ((size_t)slot * H + n0) * (CW - 1);
#pragma unroll
    for (int q = 0; q < CW - 1; ++q) *reinterpret_cast<f32x4_t*>(hp + 4 * q) = nh[q];
  }
}

// Where a wavefront's loads start: in halves four, or five where one would be left over (a round trip of its own: 1024 x 4608, nine
// loads a wavefront, 5.6 and 5.3 us), or all there are; three tiles' halves two (as good as four, and a lane's registers leave room
// for two blocks a compute unit) or, of three, all; whole tiles eight, four, two or one.
static inline int few_first(int units, bool half, bool three) {
  if (!half) return units >= 8 ? 8 : units >= 4 ? 4 : units >= 2 ? 2 : 1;
  if (three) return units == 3 ? 3 : units >= 2 ? 2 : 1;
  return units >= 4 ? (units % 4 == 1 ? 5 : 4) : units;
}

template <int R, bool HALF, bool SCALED, int EPI, int CW, bool ONCE, typename TOut>
static void launch_few(int blocks, const FewArgs& g, hipStream_t stream) {
  const int units = (g.K >> 5) / (FEW_WAVES * (HALF ? 2 : 1));
#define GS_FEW(F) gemm_few_kernel<R, HALF, SCALED, EPI, CW, F, ONCE, TOut><<<blocks, FEW_WAVES * 64, 0, stream>>>(g)
  switch (few_first(units, HALF, R >= 3)) {
    case 1: GS_FEW(1); break;
    case 2: GS_FEW(2); break;
    case 3: if constexpr (HALF) GS_FEW(3); break;
    case 4: if constexpr (R < 3) GS_FEW(4); break;
    case 5: if constexpr (HALF && R < 3) GS_FEW(5); break;
    default: if constexpr (!HALF) GS_FEW(8); break;
  }
#undef GS_FEW
}

// Between the entry points (gemm_skinny_glue.hip) and the launches (gemm_few.hip, gemm_few_fused.hip).
FewArgs few_args(const SkinnyCall& c);
bool gs_skinny_halves(int N);
void gs_few_swiglu(const SkinnyCall& c);
void gs_few_gated_run(const SkinnyCall& c);
void gs_few_residual_run(const SkinnyCall& c);
void gs_few_conv_run(const SkinnyCall& c);
