// Y (M, N) = X (M, K) . W (N, K)^T for few rows (M <= 64): the weight-streaming product of decoding,
// with what stands before and after it in a block folded in.
//
// Every weight is read once from HBM; the time of this kernel is the time of that stream.  bfloat16
// inputs, float32 accumulation on the matrix cores (v_mfma_f32_16x16x32_bf16).  One MFMA takes a 16 x 32
// tile of W as its A operand, straight from global memory in the operand's own layout (lane l: row
// l % 16, eight consecutive k at 8 * (l / 16): one 16-byte load), and a 32 x 16 tile of X^T as its B
// operand (lane l: token l % 16, the same eight k).  The result tile holds, per lane, four consecutive
// output columns n for one token.
//
// A block of WAVES wavefronts owns R tiles of 16 rows of W; its wavefronts split K among themselves and
// add their partial tiles through LDS in wavefront order, each row tile's by a wavefront of its own, which
// runs that row tile's epilogue.  Rows beyond N, tokens beyond M and k beyond K
// are masked (K must be a multiple of 8 so that every 16-byte load is aligned).
//
// The weight is read either as it is stored, rows of K (SHUF = 0), or from a tile-major copy
// (SHUF = 1) in which the 16 x 32 tile of (row tile, k step) lies as 64 lanes x 16 bytes in the
// operand's own order, tiles of a row tile one after the other: then every load of a wavefront is one
// contiguous kilobyte and a wavefront streams a contiguous range, which HBM serves faster than
// sixteen rows 2 K bytes apart.
//
// X is read either as rows of ldx elements or, with x_tiled, in the order the MFMA takes it ("tiled rows",
// tiled_index in common.h: the 16 x 32 tile of (k step, row tile) as 64 lanes x 16 bytes): then every load of X is one
// contiguous kilobyte instead of sixteen pieces of rows, which is what the products of many rows are bound by.  With
// y_tiled the epilogues that write rows for a following product (SwiGLU, convolution, pre-weighted rows) write them
// in that order.
//
// A tile-major weight whose K the wavefronts share evenly, without the norm's fold (PRO 1), goes to gemm_few_impl.h's kernel, which
// gives the same bits sooner, by the rules of gemm_few.hip (gs_few_*).  Here is what they leave: besides stored rows and other K, weighted
// rows beyond 32, products into the stream beyond 32 rows or of weights not cut in halves, convolutions of more than 2,048 channels or
// unaligned state, float32 results of SwiGLU, and the sizes whose figures stand there.
//
// What feeds X (PRO):
//   0  X is given, bfloat16.
//   1  X is the RMSNorm of the float32 residual stream: x = res * inv_rms(row) * norm_weight, rounded to
//      bfloat16 as the norm kernel would store it; the row's sum of squares comes as partial sums
//      (row, nb), added in a fixed order.
//   2  X holds rows already multiplied by the norm's weight (res * norm_weight,
//      written by the product that last added to the stream, EPI 2); the row's inverse root mean square,
//      which no single block of that product knew, multiplies this product's result instead:
//      (x inv) W^T = inv (x W^T).  The norm costs no kernel and no pass of its own.
// What is done with Y (EPI):
//   0  stored (bfloat16 or float32).
//   1  SwiGLU: W holds gate rows [0, N/2) then up rows; stores silu(gate) * up, N/2 wide.
//   5  partial sums: K is shared out over gridDim.x blocks as well (the weight tiles over gridDim.y), each writes its float32 (M, N) sheet; a second
//      kernel adds the sheets.  For many rows: every block reads all rows of X for its part of K, so the fewer
//      weight rows and the more of K a block takes, the more X traffic; sharing K over blocks caps it.
//   2  added to the residual stream in place (float32), and the sums of squares of the new rows over this
//      block's columns stored as partial sums for the next norm.
//   4  gated activation: as 1, but the two products are rounded as they would be stored, then biased (float32, or none), and the
//      activation is the one asked for: the feed-forwards whose gate is no silu.
//   3  gated short convolution of a decode step: tiles are the B, C, X rows of 16 channels; u = B X,
//      y = taps . (history, u) + bias, out = C y, history shifted; one token per sequence.
#pragma once
#include "common.h"
#include <type_traits>

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

// A kernel's LAYOUT is SHUF, with SKINNY_ONCE added where the weight's pieces are loaded non-temporally.
#define SKINNY_ONCE 4
// And SKINNY_PAIRED for two row tiles whose blocks come two to a compute unit: a lane then has 128 registers.
#define SKINNY_PAIRED 8

__device__ __forceinline__ bf16x8_t load8(const bf16* p) { return *reinterpret_cast<const bf16x8_t*>(p); }

// A piece of weight.  Of a large weight's tile-major copy (skinny_once) it is loaded non-temporally: whole lines, each read by
// one compute unit and not again in the step.
template <int LAYOUT>
__device__ __forceinline__ bf16x8_t load8w(const bf16* p) {
  return LAYOUT & SKINNY_ONCE ? __builtin_nontemporal_load(reinterpret_cast<const bf16x8_t*>(p)) : load8(p);
}

__device__ __forceinline__ bf16x8_t zero8() {
  bf16x8_t z;
#pragma unroll
  for (int i = 0; i < 8; ++i) z[i] = (__bf16)0.0f;
  return z;
}

template <typename T>
__device__ __forceinline__ void store4(T* p, f32x4_t v, int valid);
template <>
__device__ __forceinline__ void store4<float>(float* p, f32x4_t v, int valid) {
  if (valid >= 4 && ((uintptr_t)p & 15) == 0) {
    *reinterpret_cast<f32x4_t*>(p) = v;
  } else {
    for (int i = 0; i < valid && i < 4; ++i) p[i] = v[i];
  }
}
template <>
__device__ __forceinline__ void store4<bf16>(bf16* p, f32x4_t v, int valid) {
  if (valid >= 4 && ((uintptr_t)p & 7) == 0) {
    uint2 o;
    o.x = (uint32_t)f32_to_bf16(v[0]).x | ((uint32_t)f32_to_bf16(v[1]).x << 16);
    o.y = (uint32_t)f32_to_bf16(v[2]).x | ((uint32_t)f32_to_bf16(v[3]).x << 16);
    *reinterpret_cast<uint2*>(p) = o;
  } else {
    for (int i = 0; i < valid && i < 4; ++i) p[i] = f32_to_bf16(v[i]);
  }
}

// Everything the prologues and epilogues need beside X, W, Y; unused fields stay null.
struct SkinnyExtra {
  // PRO 1
  const float* res;      // (M, K) float32 residual stream
  const float* ssq;      // (M, nb) partial sums of squares of res rows
  int nb;
  const float* norm_w;   // (K)
  float eps;
  // EPI 2
  float* res_out;        // (M, N) float32, updated in place
  float* ssq_out;        // (M, gridDim.x)
  const float* next_w;   // (N) weight of the norm that reads the stream next, or null
  bf16* xs_out;          // (M, N) res * next_w, for that norm's consumer
  // EPI 3
  const float* taps;     // (H, W)
  const float* conv_bias;
  float* state;          // (slots, H, W - 1)
  const int* slots;      // (M)
  int conv_w;
  int conv_vec;          // widths 2..4, H a multiple of 4, taps, bias and state 16-byte aligned: the epilogue keeps taps
                         // and history in registers and moves them sixteen bytes at a time
  // layouts
  int x_tiled;           // X comes as tiled rows (PRO 0 only; K a multiple of 32)
  // EPI 4
  const float* act_bias; // (N): the gate rows', then the up rows'; or null
  int act;
  int y_tiled;           // EPI 1, 3, 4: Y, EPI 2: xs_out are written as tiled rows (their width a multiple of 32)
  // EPI 0
  int squared;           // the first so many columns are stored as the square of their relu, of the rounded product
};

template <int R, int MT, int WAVES, int PRO, int EPI, int LAYOUT, typename TOut>
__global__ __launch_bounds__(WAVES * 64, LAYOUT & SKINNY_PAIRED ? WAVES / 2 : 1) void gemm_skinny_kernel(const bf16* __restrict__ X, int ldx,
                                                                  const bf16* __restrict__ W,
                                                                  TOut* __restrict__ Y, int ldy, int M, int N,
                                                                  int K, SkinnyExtra ex) {
  constexpr int SHUF = LAYOUT & 3;
  constexpr bool RING = MT > 1 && !(LAYOUT & SKINNY_PAIRED);     // see the loop
  constexpr bool GLU = EPI == 1 || EPI == 4;
  extern __shared__ float red[];  // WAVES (one row tile: WAVES - 1) x R x MT x 64 x 4 floats
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  static_assert(WAVES >= MT, "a wavefront for each row tile's epilogue");
  // wavefront w adds up and finishes row tile w
  const int emt = MT > 1 ? wave : 0;
  const int r16 = lane & 15, kg = lane >> 4;
  const int half = N >> 1;
  // rows of W this block owns
  int rowbase[R];
  if (GLU) {
    const int n0 = blockIdx.x * 16 * (R / 2);
#pragma unroll
    for (int r = 0; r < R; ++r) rowbase[r] = n0 + (r >> 1) * 16 + ((r & 1) ? half : 0);
  } else if (EPI == 3) {
    const int H = N / 3;
#pragma unroll
    for (int r = 0; r < R; ++r) rowbase[r] = blockIdx.x * (SHUF == 2 ? 8 : 16) + r * H;  // B, C, X rows of the same channels
  } else if (SHUF == 2) {
    rowbase[0] = blockIdx.x * 8;  // half a tile: twice the blocks for a weight of few rows
  } else {
    // (EPI 5: the grid is (parts of K, weight tiles), see below)
    const int n0 = (EPI == 5 ? blockIdx.y : blockIdx.x) * 16 * R;
#pragma unroll
    for (int r = 0; r < R; ++r) rowbase[r] = n0 + r * 16;
  }
  static_assert(SHUF != 2 || (R == 1 && (EPI == 0 || EPI == 2)) || EPI == 3, "half tiles are written for plain products and for the residual and the convolution epilogues");
  const bool wact = SHUF != 2 || r16 < 8;  // half tiles: the lanes of the other eight rows load nothing
  const bf16* wrow[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    int n = rowbase[r] + r16;
    if (GLU && !(r & 1) && n >= half) n = half - 1;  // gate rows end at N/2
    if (EPI == 3 && n >= (r + 1) * (N / 3)) n = (r + 1) * (N / 3) - 1;
    if (n >= N) n = N - 1;                                // clamped: loaded, never stored
    if (SHUF == 2)
      wrow[r] = W + ((size_t)(rowbase[r] >> 4) * ((K + 31) >> 5)) * 512 + (kg * 16 + (rowbase[r] & 8) + (r16 & 7)) * 8;
    else if (SHUF) {
      // tile-major: the 16 x 32 tile of (row tile, k step) is 64 lanes x 16 bytes in the operand's own order
      // (a tile past the weight's last, where a block's tiles outnumber what is left, reads the last: loaded, never stored)
      const int tile = (rowbase[r] >> 4) < ((N + 15) >> 4) ? (rowbase[r] >> 4) : ((N + 15) >> 4) - 1;
      wrow[r] = W + ((size_t)tile * ((K + 31) >> 5)) * 512 + lane * 8;
    }
    else
      wrow[r] = W + (size_t)n * K + kg * 8;
  }
  bool xok[MT];
  const bf16* xrow[MT];
  const float* rrow[MT];
  float inv[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    int m = mt * 16 + r16;
    xok[mt] = m < M;
    xrow[mt] = nullptr;
    rrow[mt] = nullptr;
    inv[mt] = 0.f;
    if (PRO != 1) {
      // (a row past M: the last, whose line a neighbour asks for anyway; its column of the result is never stored)
      const int mc = m < M ? m : M - 1;
      xrow[mt] = ex.x_tiled ? X + (size_t)((mc >> 4) * 64 + kg * 16 + (mc & 15)) * 8 : X + (size_t)mc * ldx + kg * 8;
    } else {
      rrow[mt] = ex.res + (size_t)(xok[mt] ? m : M - 1) * K;
    }
    if (PRO == 1) {
      // the row's sum of squares: this lane group adds every fourth partial, then the four groups are added
      float s = 0.f;
      if (xok[mt])
        for (int b = kg; b < ex.nb; b += 4) s += ex.ssq[(size_t)m * ex.nb + b];
      s += __shfl_xor(s, 16, 64);
      s += __shfl_xor(s, 32, 64);
      inv[mt] = norm_inverse(s, (float)K, ex.eps);
    }
  }

  // Pre-weighted rows: the rows' inverse root mean squares are needed only at the end.  The wavefronts share
  // the rows; a lane adds every 64th partial sum and the wavefront adds its lanes (an order that depends on
  // nothing but the number of partials).  The first row's loads start here, under the product's own.
  __shared__ float inv_s[64];
  constexpr bool scaled = PRO == 2;
  // With two row tiles all of a wavefront's rows are asked for here (where the registers allow): after the loop they were a round trip of their own
  // (20 rows of 9216 x 1024 9.3 against 8.7 us).
  constexpr int RPW = (MT * 16 + WAVES - 1) / WAVES;      // rows a wavefront
  constexpr int EARLY = MT == 2 && RING ? RPW : 1;
  float pre[EARLY][4];
  if (scaled && wave < M) {
    // (a row or a partial sum that does not exist is read from one that does and not counted: no load sits behind a branch)
#pragma unroll
    for (int i = 0; i < EARLY; ++i) {
      const int m = wave + i * WAVES;
      const float* row = ex.ssq + (size_t)(m < M ? m : M - 1) * ex.nb;
#pragma unroll
      for (int j = 0; j < 4; ++j) pre[i][j] = row[lane + 64 * j < ex.nb ? lane + 64 * j : 0];
    }
  }

  // The convolution's slots, by scalar loads (the row number is the same for every lane), each lane then picking its
  // row's: the history's addresses wait for them, and scalar loads return on a counter of their own.
  int cslot = 0;
  if (EPI == 3) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = emt * 16 + i;
      const int sv = ex.slots[row < M ? row : 0];
      cslot = r16 == i ? sv : cslot;
    }
  }

  // What the epilogue reads besides the product (the stream's old rows, the convolution's history and taps) is
  // loaded early, by the wavefront that runs the epilogue, so that these round trips pass under the product's own
  // instead of after it.  The stream's old rows are asked for here, before the weights.  The convolution's operands
  // are asked for right after the first weight loads (few row tiles), by loads that sit behind no branch and whose
  // values nothing touches before the epilogue: wherever a branch hides how many loads are in flight the compiler
  // waits for all of them, and with a test on each tap and each history value that was a round trip apiece before
  // the first weight was asked for (measured on cold weights of 6144 x 2048, 8 rows: 10.6 against 9.6 us a kernel).
  constexpr int PRE_TAPS = 4;                       // convolutions of up to this width are held in registers
  const bool half_ok = SHUF != 2 || kg < 2;
  f32x4_t rold[EPI == 2 ? R : 1], nextw[EPI == 2 ? R : 1];
  float chist[4][PRE_TAPS - 1], ctap[4][PRE_TAPS], cbias[4];
  const bool vec4 = (N & 3) == 0;
  const int em = emt * 16 + r16;                    // the epilogue's row
  if (EPI == 2 && wave < MT) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int n = rowbase[r] + kg * 4;
      const bool ok = n < N && half_ok;
      nextw[r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if (ok && ex.next_w) {
        if (vec4) nextw[r] = *reinterpret_cast<const f32x4_t*>(ex.next_w + n);
        else
          for (int i = 0; i < 4; ++i)
            if (n + i < N) nextw[r][i] = ex.next_w[n + i];
      }
      rold[r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if (ok && em < M) {
        const float* p = ex.res_out + (size_t)em * N + n;
        if (vec4) rold[r] = *reinterpret_cast<const f32x4_t*>(p);
        else
          for (int i = 0; i < 4; ++i)
            if (n + i < N) rold[r][i] = p[i];
      }
    }
  }
  f32x4_t gbias[EPI == 4 ? R : 1];
  if (EPI == 4 && wave < MT) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int n = rowbase[r] + kg * 4;               // (whole tiles: N / 2 is a multiple of 16; a tile past the last reads the last)
      const int end = r & 1 ? N : half;
      gbias[r] = ex.act_bias ? *reinterpret_cast<const f32x4_t*>(ex.act_bias + (n < end ? n : end - 4)) : f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
  }
  const bool pre_conv = EPI == 3 && ex.conv_vec != 0;
  // A lane's four channels are neighbours, so their taps (4 x width floats), their bias and, per row, their history
  // (4 x (width - 1) floats) are each one run of memory: moved sixteen bytes at a time, the width a compile-time
  // number in each of the three forms.  A block's channels past H read the last four (loaded, never used), a row
  // past M its row 0's slot.
  // (macros, not closures: arrays that a closure takes by reference are not always kept in registers, and these
  // were not: taps and history went through scratch memory, a store after each load's arrival and a load before use)
#define GS_CONV_WIDTH(BODY)                                                                                            \
  switch (ex.conv_w) {                                                                                                  \
    case 2: { constexpr int WD = 2; BODY } break;                                                                       \
    case 3: { constexpr int WD = 3; BODY } break;                                                                       \
    default: { constexpr int WD = 4; BODY } break;                                                                      \
  }
#define GS_PRELOAD_CONV_BODY                                                                                           \
  {                                                                                                                     \
    f32x4_t tq[WD];                                                                                                     \
    _Pragma("unroll") for (int q = 0; q < WD; ++q) tq[q] = *reinterpret_cast<const f32x4_t*>(ex.taps + (size_t)cc0_ * WD + 4 * q); \
    _Pragma("unroll") for (int i = 0; i < 4; ++i)                                                                       \
      _Pragma("unroll") for (int p = 0; p < WD; ++p) ctap[i][p] = tq[(i * WD + p) / 4][(i * WD + p) % 4];               \
    f32x4_t hq[WD - 1];                                                                                                 \
    const float* hp = ex.state + ((size_t)cslot * H_ + cc0_) * (WD - 1);                                                \
    _Pragma("unroll") for (int q = 0; q < WD - 1; ++q) hq[q] = *reinterpret_cast<const f32x4_t*>(hp + 4 * q);           \
    _Pragma("unroll") for (int i = 0; i < 4; ++i)                                                                       \
      _Pragma("unroll") for (int p = 0; p < WD - 1; ++p) chist[i][p] = hq[(i * (WD - 1) + p) / 4][(i * (WD - 1) + p) % 4]; \
  }
#define GS_PRELOAD_CONV()                                                                                              \
  if (EPI == 3 && wave < MT && pre_conv) {                                                                              \
    const int H_ = N / 3;                                                                                               \
    const int c0_ = blockIdx.x * (SHUF == 2 ? 8 : 16) + kg * 4;                                                         \
    const int cc0_ = c0_ + 3 < H_ ? c0_ : H_ - 4;                                                                       \
    const f32x4_t bv_ = *reinterpret_cast<const f32x4_t*>((ex.conv_bias ? ex.conv_bias : ex.taps) + cc0_);              \
    _Pragma("unroll") for (int i = 0; i < 4; ++i) cbias[i] = bv_[i];                                                    \
    GS_CONV_WIDTH(GS_PRELOAD_CONV_BODY)                                                                                 \
  }
#define GS_CONV_EPI_BODY                                                                                                \
        {                                                                                                              \
          f32x4_t out, nh[WD - 1];                                                                                     \
_Pragma("unroll")                                                                                                      \
          for (int i = 0; i < 4; ++i) {                                                                                \
            const float Bv = to_f32(f32_to_bf16(sum[0][i])), Cv = to_f32(f32_to_bf16(sum[R > 1 ? 1 : 0][i])),          \
                        Xv = to_f32(f32_to_bf16(sum[R > 2 ? 2 : 0][i]));                                               \
            const float u = Bv * Xv;                                                                                   \
            float y = 0.f;                                                                                             \
_Pragma("unroll")                                                                                                      \
            for (int p = 0; p < WD - 1; ++p) y += ctap[i][p] * chist[i][p];                                            \
            y += ctap[i][WD - 1] * u;                                                                                  \
            if (ex.conv_bias) y += cbias[i];                                                                           \
            out[i] = Cv * y;                                                                                           \
_Pragma("unroll")                                                                                                      \
            for (int p = 0; p < WD - 1; ++p)                                                                           \
              nh[(i * (WD - 1) + p) / 4][(i * (WD - 1) + p) % 4] = p < WD - 2 ? chist[i][p + 1] : u;                   \
          }                                                                                                            \
          store4<TOut>(Y + (ex.y_tiled ? tiled_index(em, c0, MT) : (size_t)em * ldy + c0), out, 4);                    \
          float* hp = ex.state + ((size_t)cslot * H + c0) * (WD - 1);                                                  \
_Pragma("unroll")                                                                                                      \
          for (int q = 0; q < WD - 1; ++q) *reinterpret_cast<f32x4_t*>(hp + 4 * q) = nh[q];                            \
        }
  if (EPI == 3 && MT >= 2) GS_PRELOAD_CONV()   // the loop of many row tiles keeps its order
  f32x4_t acc[R][MT];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[r][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int xstep = ex.x_tiled ? MT * 512 : 32;   // elements between a row tile's consecutive k steps
  auto load_x = [&](int mt, int s) -> bf16x8_t {
    if (PRO != 1) {
      return load8(xrow[mt] + (size_t)s * xstep);
    } else {
      const int k = (s << 5) + kg * 8;
      const f32x4_t a0 = *reinterpret_cast<const f32x4_t*>(rrow[mt] + k);
      const f32x4_t a1 = *reinterpret_cast<const f32x4_t*>(rrow[mt] + k + 4);
      const f32x4_t w0 = *reinterpret_cast<const f32x4_t*>(ex.norm_w + k);
      const f32x4_t w1 = *reinterpret_cast<const f32x4_t*>(ex.norm_w + k + 4);
      union {
        bf16x8_t v;
        uint16_t u[8];
      } o;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        o.u[i] = f32_to_bf16(a0[i] * inv[mt] * w0[i]).x;
        o.u[4 + i] = f32_to_bf16(a1[i] * inv[mt] * w1[i]).x;
      }
      return o.v;
    }
  };

  // this wavefront's share of K, in steps of 32
  // (EPI 5: the blocks that own the same weight rows share K among themselves first, blockIdx.x taking its part.  The part
  // runs fastest in launch order and blocks go to the eight XCDs in turn, so with eight parts every XCD works on one
  // part of K and holds that part of X alone in its L2; with four, two XCDs a part.)
  const int ksteps_all = (K + 31) >> 5;
  int kbeg = 0, kend = ksteps_all;
  if (EPI == 5) {
    const int part = (ksteps_all + (int)gridDim.x - 1) / (int)gridDim.x;
    kbeg = blockIdx.x * part;
    kend = kbeg + part < ksteps_all ? kbeg + part : ksteps_all;
    if (kend < kbeg) kend = kbeg;
  }
  const int per = (kend - kbeg + WAVES - 1) / WAVES;
  const int s0 = kbeg + wave * per, s1 = (s0 + per < kend) ? s0 + per : kend;
  int s = s0;
  // steps whose loads are issued together: as many as about a hundred registers hold (16 bytes a lane per tile)
  constexpr int UQ = (WAVES >= 16 ? 12 : 24) / (R + MT);   // sixteen wavefronts leave a lane 128 registers
  constexpr int U = UQ >= 8 ? 8 : (UQ >= 4 ? 4 : (UQ >= 2 ? 2 : 1));
  constexpr int WSTEP = SHUF ? 512 : 32;  // elements between a row tile's consecutive k steps
  const bool whole = SHUF || (K & 31) == 0;
  // C steps, their loads issued together, then multiplied.  (One row tile: the lanes without a row load nothing.  A macro, as above.)
#define GS_BATCH(C, BETWEEN)                                                                                           \
  {                                                                                                                     \
    bf16x8_t a[C][R], b[C][MT];                                                                                         \
    _Pragma("unroll") for (int u = 0; u < C; ++u) {                                                                     \
      _Pragma("unroll") for (int r = 0; r < R; ++r)                                                                     \
        a[u][r] = MT > 1 || wact ? load8w<LAYOUT>(wrow[r] + (size_t)(s + u) * WSTEP) : zero8();                         \
      _Pragma("unroll") for (int mt = 0; mt < MT; ++mt) b[u][mt] = MT > 1 || xok[mt] ? load_x(mt, s + u) : zero8();     \
    }                                                                                                                   \
    BETWEEN                                                                                                             \
    _Pragma("unroll") for (int u = 0; u < C; ++u)                                                                       \
      _Pragma("unroll") for (int r = 0; r < R; ++r)                                                                     \
        _Pragma("unroll") for (int mt = 0; mt < MT; ++mt)                                                               \
          acc[r][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][r], b[u][mt], acc[r][mt], 0, 0, 0);                 \
    s += C;                                                                                                             \
  }
  if (!RING) {
    // few rows: the steps' loads are issued U at a time, then multiplied (the ring below costs registers, and with
    // them a resident wavefront per SIMD, which these shapes need more; two row tiles: all loads before the first product, which
    // the compiler would else move up between them to save registers)
    if (EPI == 3) {
      if (whole && s + U <= s1) GS_BATCH(U, GS_PRELOAD_CONV())
      else GS_PRELOAD_CONV()
    }
    if (whole)
      while (s + U <= s1) GS_BATCH(U, if (MT > 1) __builtin_amdgcn_sched_barrier(0);)
  } else if (whole && s1 - s0 >= U) {
    // many rows: a ring of U steps in registers: a step is multiplied as soon as it has arrived and its place is
    // asked for again at once, U steps ahead, so that loads are in flight the whole time (loads return in order).
    // Measured against issuing U steps at a time, both builds run in turn on one GPU, six repeats each, gate|up of
    // 16384 x 2048: 18.6-18.7 against 19.3-19.4 us at 64 rows, 16.8-16.9 against 17.2-17.3 us at 48 rows; two row tiles: the
    // convolution's input product of 6144 x 2048 10.5 against 11.5 us at 32 rows, 2048 x 8192 13.9 against 14.8.
    bf16x8_t a[U][R], b[U][MT];
    auto fetch = [&](int u, int step) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        // every lane loads (its address is a valid one): a load under a lane mask would hide from the
        // compiler how many loads are in flight, and it would wait for all of them (half tiles: the lanes of
        // the other eight rows load the first eight's again; those rows are never stored)
        a[u][r] = load8w<LAYOUT>(wrow[r] + (size_t)step * WSTEP);
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) b[u][mt] = load_x(mt, step);
    };
    auto multiply = [&](int u) {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[r][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][r], b[u][mt], acc[r][mt], 0, 0, 0);
    };
#pragma unroll
    for (int u = 0; u < U; ++u) fetch(u, s0 + u);
    const int groups = (s1 - s0) / U;
    for (int g = 1; g < groups; ++g) {
      const int base = s0 + g * U;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        multiply(u);
        fetch(u, base + u);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) multiply(u);
    s = s0 + groups * U;
  }
  // What is left of a wavefront's share: four and two steps together where U is more.  K = 1024 is four steps a wavefront, and
  // one by one each was a round trip of its own (8 rows, microseconds one by one and together: 1024 x 1024 4.35 and 3.6, 2048 x
  // 1024 4.4 and 3.5, gate and up of 9216 x 1024 8.2 and 7.1; 1024 x 4608, eighteen steps, 7.2 and 6.7).
  if (whole) {
    if (U > 4 && s + 4 <= s1) GS_BATCH(4, )
    if (U > 2 && EPI != 3 && s + 2 <= s1) GS_BATCH(2, )
  }
  for (; s < s1; ++s) {
    const int k = (s << 5) + kg * 8;
    const bool kin = k < K;
    bf16x8_t b[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) b[mt] = kin ? load_x(mt, s) : zero8();
#pragma unroll
    for (int r = 0; r < R; ++r) {
      bf16x8_t a = ((kin || SHUF) && wact) ? load8w<LAYOUT>(wrow[r] + (size_t)s * WSTEP) : zero8();
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[r][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[mt], acc[r][mt], 0, 0, 0);
    }
  }

  if (scaled) {
    // a wavefront's first row was asked for at the start; its further rows (row wave + WAVES, ...) are asked for here
    // in batches, every load of a batch in flight before the first is added, at addresses that always exist (a row
    // or a partial sum that does not is read from the first and counted as zero): no load sits behind a branch
    constexpr int BATCH = RPW - 1 < 8 ? (RPW > 1 ? RPW - 1 : 1) : 8;
#pragma unroll
    for (int i = 0; i < EARLY; ++i) {
      const int m = wave + i * WAVES;
      if (m < M) {
#pragma unroll
        for (int j = 0; j < 4; ++j) pre[i][j] = lane + 64 * j < ex.nb ? pre[i][j] : 0.f;
        float ssum = (pre[i][0] + pre[i][1]) + (pre[i][2] + pre[i][3]);
        for (int b = 256 + lane; b < ex.nb; b += 64) ssum += ex.ssq[(size_t)m * ex.nb + b];
        ssum = wave_sum_dpp(ssum);
        if (lane == 0) inv_s[m] = norm_inverse(ssum, (float)K, ex.eps);
      }
    }
    if (MT == 1) {   // at most one further row: the plain loop is the smallest code, and the step of few rows feels it
      for (int m = wave + WAVES; m < M; m += WAVES) {
        float ssum = 0.f;
        for (int b = lane; b < ex.nb; b += 64) ssum += ex.ssq[(size_t)m * ex.nb + b];
        ssum = wave_sum_dpp(ssum);
        if (lane == 0) inv_s[m] = norm_inverse(ssum, (float)K, ex.eps);
      }
    }
#pragma unroll
    for (int i0 = 1; MT > 1 && EARLY == 1 && i0 < RPW; i0 += BATCH) {
      if (wave + i0 * WAVES < M) {
        float q[BATCH][4];
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
          const int m = wave + (i0 + i) * WAVES;
          const float* row = ex.ssq + (size_t)(m < M ? m : wave) * ex.nb;
#pragma unroll
          for (int j = 0; j < 4; ++j) q[i][j] = row[lane + 64 * j < ex.nb ? lane + 64 * j : 0];
        }
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
          const int m = wave + (i0 + i) * WAVES;
#pragma unroll
          for (int j = 0; j < 4; ++j) q[i][j] = lane + 64 * j < ex.nb ? q[i][j] : 0.f;
          float ssum = (q[i][0] + q[i][1]) + (q[i][2] + q[i][3]);
          if (ex.nb > 256 && m < M)
            for (int b = 256 + lane; b < ex.nb; b += 64) ssum += ex.ssq[(size_t)m * ex.nb + b];
          ssum = wave_sum_dpp(ssum);
          if (lane == 0 && i0 + i < RPW && m < M) inv_s[m] = norm_inverse(ssum, (float)K, ex.eps);
        }
      }
    }
    if (WAVES == 1) __syncthreads();
  }

  // Add the wavefronts' partial tiles, in wavefront order: wavefront w takes row tile w, its own part of it from registers and
  // the others' from LDS.  (With one wavefront for all of them: gate and up of 16384 x 2048 at 64 rows 19.1 against 17.9 us, the
  // convolution's input product of 6144 x 2048 15.0 against 13.0.)
  f32x4_t sum[R];
#pragma unroll
  for (int r = 0; r < R; ++r) sum[r] = acc[r][0];
  if (MT == 1 && WAVES > 1) {
    if (wave > 0) {
#pragma unroll
      for (int r = 0; r < R; ++r) *reinterpret_cast<f32x4_t*>(red + (((wave - 1) * R + r) * 64 + lane) * 4) = acc[r][0];
    }
    __syncthreads();
    if (wave > 0) return;
    for (int w = 0; w < WAVES - 1; ++w)
#pragma unroll
      for (int r = 0; r < R; ++r) sum[r] += *reinterpret_cast<const f32x4_t*>(red + ((w * R + r) * 64 + lane) * 4);
  } else if (WAVES > 1) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      if (wave != mt) {
#pragma unroll
        for (int r = 0; r < R; ++r)
          *reinterpret_cast<f32x4_t*>(red + (((wave * R + r) * MT + mt) * 64 + lane) * 4) = acc[r][mt];
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
    const float* src = red + (emt * 64 + lane) * 4;
#pragma unroll
    for (int w = 0; w < WAVES; ++w)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        f32x4_t v = own[r];
        if (w >= MT || w != wave) v = *reinterpret_cast<const f32x4_t*>(src + (size_t)(w * R + r) * MT * 256);
        if (w == 0) sum[r] = v; else sum[r] += v;
      }
  }

  // rows that came pre-weighted get their inverse root mean square now
  if (scaled) {
    const float iv = inv_s[em < M ? em : 0];
#pragma unroll
    for (int r = 0; r < R; ++r) sum[r] *= iv;
  }

  // lane l holds, for token 16 wave + l%16, columns rowbase + 4*(l/16) + 0..3 of every tile
  const bool live = em < M;
  if (EPI == 0 || EPI == 5) {
    if (!live) return;
    TOut* Yp = EPI == 5 ? Y + (size_t)blockIdx.x * M * ldy : Y;   // partial sums: one (M, N) sheet per part of K
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int n = rowbase[r] + kg * 4;
      if (EPI == 0 && n < ex.squared) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float z = to_f32(f32_to_bf16(sum[r][i])), u = z > 0.f ? z : 0.f;
          if (n + i < ex.squared) sum[r][i] = u * u;
        }
      }
      if (N - n > 0 && half_ok) store4<TOut>(Yp + (size_t)em * ldy + n, sum[r], N - n);
    }
  } else if (EPI == 4) {
    if (!live) return;
#pragma unroll
    for (int r = 0; r < R; r += 2) {
      const int n = rowbase[r] + kg * 4;
      f32x4_t o;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        o[i] = gated_act(to_f32(f32_to_bf16(sum[r][i])) + gbias[r][i], ex.act) * (to_f32(f32_to_bf16(sum[r + 1][i])) + gbias[EPI == 4 ? r + 1 : 0][i]);
      if (half - n > 0) store4<TOut>(Y + (ex.y_tiled ? tiled_index(em, n, MT) : (size_t)em * ldy + n), o, half - n);
    }
  } else if (EPI == 1) {
    if (!live) return;
#pragma unroll
    for (int r = 0; r < R; r += 2) {
      const int n = rowbase[r] + kg * 4;  // output column in [0, N/2)
      f32x4_t g = sum[r], u = sum[r + 1], o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = g[i] / (1.0f + expf(-g[i])) * u[i];
      if (half - n > 0) store4<TOut>(Y + (ex.y_tiled ? tiled_index(em, n, MT) : (size_t)em * ldy + n), o, half - n);
    }
  } else if (EPI == 2) {
    // every lane takes part in the shuffles, live or not
    float ss = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int n = rowbase[r] + kg * 4;
      if (live && n < N && half_ok) {
        float* p = ex.res_out + (size_t)em * N + n;
        f32x4_t nv, xv;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          // the product is rounded to bfloat16 first, as the unfused path stores it before the add
          nv[i] = rold[r][i] + to_f32(f32_to_bf16(sum[r][i]));
          if (n + i < N) ss += nv[i] * nv[i];
          xv[i] = nv[i] * nextw[r][i];
        }
        if (vec4) *reinterpret_cast<f32x4_t*>(p) = nv;
        else
          for (int i = 0; i < 4; ++i)
            if (n + i < N) p[i] = nv[i];
        if (ex.xs_out) store4<bf16>(ex.xs_out + (ex.y_tiled ? tiled_index(em, n, MT) : (size_t)em * N + n), xv, N - n);
      }
    }
    ss += __shfl_xor(ss, 16, 64);
    ss += __shfl_xor(ss, 32, 64);
    if (live && kg == 0) ex.ssq_out[(size_t)em * gridDim.x + blockIdx.x] = ss;
  } else if (EPI == 3) {
    if (!live) return;
    const int H = N / 3, Wd = ex.conv_w;
    const int c0 = blockIdx.x * (SHUF == 2 ? 8 : 16) + kg * 4;
    if (pre_conv) {
      if (c0 >= H || !half_ok) return;
      GS_CONV_WIDTH(GS_CONV_EPI_BODY)
      return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = c0 + i;
      if (c >= H || !half_ok) break;
      const float Bv = to_f32(f32_to_bf16(sum[0][i])), Cv = to_f32(f32_to_bf16(sum[R > 1 ? 1 : 0][i])),
                  Xv = to_f32(f32_to_bf16(sum[R > 2 ? 2 : 0][i]));
      const float u = Bv * Xv;
      float* hist = ex.state + ((size_t)cslot * H + c) * (Wd - 1);
      const float* wt = ex.taps + (size_t)c * Wd;
      float y = 0.f;
      for (int p = 0; p < Wd - 1; ++p) y += wt[p] * hist[p];
      y += wt[Wd - 1] * u;
      if (ex.conv_bias) y += ex.conv_bias[c];
      Y[ex.y_tiled ? tiled_index(em, c, MT) : (size_t)em * ldy + c] = from_f32<TOut>(Cv * y);
      for (int p = 0; p < Wd - 2; ++p) hist[p] = hist[p + 1];
      hist[Wd - 2] = u;
    }
  }
}

template <int R, int MT, int WAVES, int PRO, int EPI, int LAYOUT, typename TOut>
static void launch_skinny(int blocks, const bf16* X, int ldx, const bf16* W, TOut* Y, int ldy, int M, int N, int K,
                          const SkinnyExtra& ex, hipStream_t stream) {
  const size_t lds = (size_t)(MT > 1 ? WAVES : WAVES - 1) * R * MT * 256 * sizeof(float);
  if (lds > 64 * 1024) {
    // more than the default limit of dynamic LDS: asked for once per kernel
    static const hipError_t asked = hipFuncSetAttribute(
        reinterpret_cast<const void*>(&gemm_skinny_kernel<R, MT, WAVES, PRO, EPI, LAYOUT, TOut>),
        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    (void)asked;
  }
  gemm_skinny_kernel<R, MT, WAVES, PRO, EPI, LAYOUT, TOut>
      <<<blocks, WAVES * 64, lds, stream>>>(X, ldx, W, Y, ldy, M, N, K, ex);
}

template <int R, int MT, int WAVES, int LAYOUT>
static void launch_skinny_parts(int blocks, int parts, const bf16* X, int ldx, const bf16* W, float* Y, int M, int N,
                                int K, const SkinnyExtra& ex, hipStream_t stream) {
  const size_t lds = (size_t)(MT > 1 ? WAVES : WAVES - 1) * R * MT * 256 * sizeof(float);
  gemm_skinny_kernel<R, MT, WAVES, 0, 5, LAYOUT, float>
      <<<dim3(parts, blocks), WAVES * 64, lds, stream>>>(X, ldx, W, Y, N, M, N, K, ex);
}

// MT from M; the wavefronts per block are given per MT so that the LDS for the partial tiles,
// WAVES * R * MT KB, leaves a compute unit room
#define GS_BY_MT4(R, W1, W2, W3, W4, PRO, EPI, TOut, blocks)                                                            \
  switch ((M + 15) / 16) {                                                                                              \
    case 1: launch_skinny<R, 1, W1, PRO, EPI, LAYOUT, TOut>(blocks, x, ldx, w, (TOut*)Y, ldy, M, N, K, ex, stream); break;  \
    case 2: launch_skinny<R, 2, W2, PRO, EPI, LAYOUT, TOut>(blocks, x, ldx, w, (TOut*)Y, ldy, M, N, K, ex, stream); break;  \
    case 3: launch_skinny<R, 3, W3, PRO, EPI, LAYOUT, TOut>(blocks, x, ldx, w, (TOut*)Y, ldy, M, N, K, ex, stream); break;  \
    default: launch_skinny<R, 4, W4, PRO, EPI, LAYOUT, TOut>(blocks, x, ldx, w, (TOut*)Y, ldy, M, N, K, ex, stream); break; \
  }
#define GS_BY_MT(R, WAVES, PRO, EPI, TOut, blocks) GS_BY_MT4(R, WAVES, WAVES, WAVES, WAVES, PRO, EPI, TOut, blocks)

// Whether a weight's tile-major copy is loaded non-temporally: from 8 MB on.  Where the weights of a step pass through the
// last-level cache (256 MB) such loads shorten products of 20 MB and more by 1 to 7 % (8 rows: 2048 x 8192 12.5 us, with plain loads
// 12.9; gate and up 16384 x 2048 17.0 and 17.6) and leave the cache to what a step reads again (64 requests at LFM2-1.2B
// sizes, 64 tokens: 95.9 ms, with plain loads below 20 MB 96.6); below 8 MB they are within 1 % of plain ones.  Where the weights
// stay in the cache from step to step, as a small model's do, they cost up to a fifth (2048 x 3072, 8 rows: 6.1 and 5.3; 3072 x
// 1024 4.65 and 4.21).  (The decode attention's keys, whose lines two loads share, loaded like that: 2 to 3 % longer.)
static inline bool skinny_once(int N, int K) { return (long)N * K >= 4L << 20; }

// Four tiles a block where four row tiles of X are read: a block reads as much of W as of X then, not half as much.  Such a
// block has a compute unit to itself, so the last round of them has to be nearly full, and K long enough for what a block
// starts and ends with (64 rows, microseconds with two and with four tiles, the blocks of four in brackets: 16384 x 2048 17.9
// and 17.1 (256), x 1024 11.6 and 12.8; 16416 x 2048 23.2 and 26.4 (257); 20480 x 2048 25.7 and 29.1 (320); 24576 x 4096 48.7 and
// 52.4 (384); 28672 x 2048 and x 4096 0.98 and 0.89 of the time with two (448), 32768 x 2048 0.96 (512); with three row tiles
// 16384 x 2048 16.2 and 16.5, with 144 such blocks, 9216 x 1024, 9.6 and 10.1).
static inline bool skinny_fours(int M, int cols, int K) {
  const int blocks = gs_ceil_div(cols, 16), fours = (blocks + 1) / 2;
  return M > 48 && blocks >= 512 && K >= 2048 && 8 * fours >= 7 * 256 * gs_ceil_div(fours, 256);
}

// What the entry points pass on after their checks.
struct SkinnyCall {
  const bf16* x;
  int ldx;
  const bf16* w;   // row-major (SHUF = 0) or tile-major (SHUF = 1, 2)
  void* Y;
  int y_dtype, ldy, M, N, K, epilogue;
  SkinnyExtra ex;
  hipStream_t stream;
};

template <int LAYOUT, int PRO>
static void skinny_plain_pro(const SkinnyCall& c) {
  const bf16 *x = c.x, *w = c.w;
  void* Y = c.Y;
  const int ldx = c.ldx, ldy = c.ldy, M = c.M, N = c.N, K = c.K;
  const SkinnyExtra& ex = c.ex;
  hipStream_t stream = c.stream;
  const bool f32 = c.y_dtype == GS_F32;
  const int cols = c.epilogue == 1 ? N / 2 : N;
  const bool narrow = cols <= 8192;
  // few output columns: more wavefronts per block split K further, so that the whole chip streams
  if (c.epilogue == 1) {
    const int blocks = gs_ceil_div(cols, 16);
    if (skinny_fours(M, cols, K)) {
      const int fours = (blocks + 1) / 2;
      if (f32) launch_skinny<4, 4, 8, PRO, 1, LAYOUT, float>(fours, x, ldx, w, (float*)Y, ldy, M, N, K, ex, stream);
      else launch_skinny<4, 4, 8, PRO, 1, LAYOUT, bf16>(fours, x, ldx, w, (bf16*)Y, ldy, M, N, K, ex, stream);
    } else if (f32) { GS_BY_MT4(2, 8, 8, 4, 4, PRO, 1, float, blocks) } else { GS_BY_MT4(2, 8, 8, 4, 4, PRO, 1, bf16, blocks) }
  } else if (narrow) {
    const int blocks = gs_ceil_div(cols, 16);
    // Two row tiles and more blocks than compute units: the ring's registers would leave a unit one block, so that a few blocks
    // more are a round more (rows weighted before, 20 rows, microseconds with the ring and with batches: 6144 x 4096 19.4 and 17.6,
    // 5120 x 1024 9.2 and 7.5; plain rows 8192 x 1024 7.7 and 6.6).  Plain rows of up to 24 and a K from 4,096 on: the ring (17
    // rows of 6144 x 8192 27.4 and 28.0).
    const bool paired = PRO != 1 && M > 16 && M <= 32 && blocks > 256 && (PRO == 2 || M > 24 || K < 4096);
    if (paired) {
      constexpr int PAIRED = LAYOUT | (PRO != 1 ? SKINNY_PAIRED : 0);
      if (f32) launch_skinny<1, 2, 8, PRO, 0, PAIRED, float>(blocks, x, ldx, w, (float*)Y, ldy, M, N, K, ex, stream);
      else launch_skinny<1, 2, 8, PRO, 0, PAIRED, bf16>(blocks, x, ldx, w, (bf16*)Y, ldy, M, N, K, ex, stream);
    } else if (f32) { GS_BY_MT(1, 8, PRO, 0, float, blocks) } else { GS_BY_MT(1, 8, PRO, 0, bf16, blocks) }
  } else {
    const int blocks = gs_ceil_div(cols, 32);
    if (f32) { GS_BY_MT4(2, 8, 8, 4, 4, PRO, 0, float, blocks) } else { GS_BY_MT4(2, 8, 8, 4, 4, PRO, 0, bf16, blocks) }
  }
}

template <int LAYOUT>
static void skinny_plain(const SkinnyCall& c) {
  if (c.ex.res) skinny_plain_pro<LAYOUT, 1>(c);
  else if (c.ex.ssq) skinny_plain_pro<LAYOUT, 2>(c);
  else skinny_plain_pro<LAYOUT, 0>(c);
}

// A plain product of a weight of few rows, half a tile a block (up to 32 rows of X: two row tiles).
template <int LAYOUT>
static void skinny_plain_halves(const SkinnyCall& c) {
  const int blocks = gs_ceil_div(c.N, 8);
#define GS_HALF(MT, PRO, TOut) \
  launch_skinny<1, MT, 8, PRO, 0, LAYOUT, TOut>(blocks, c.x, c.ldx, c.w, (TOut*)c.Y, c.ldy, c.M, c.N, c.K, c.ex, c.stream)
#define GS_HALF_PRO(MT, TOut) \
  if (c.ex.res) GS_HALF(MT, 1, TOut); else if (c.ex.ssq) GS_HALF(MT, 2, TOut); else GS_HALF(MT, 0, TOut)
  if (c.y_dtype == GS_F32) {
    if (c.M <= 16) { GS_HALF_PRO(1, float); } else { GS_HALF_PRO(2, float); }
  } else {
    if (c.M <= 16) { GS_HALF_PRO(1, bf16); } else { GS_HALF_PRO(2, bf16); }
  }
#undef GS_HALF_PRO
#undef GS_HALF
}

// Gate and up with biases and an activation of choice (EPI 4): bfloat16 rows in and out, the tile-major weight.
template <int LAYOUT>
static void skinny_gated(const SkinnyCall& c) {
  const bf16 *x = c.x, *w = c.w;
  void* Y = c.Y;
  const int ldx = c.ldx, ldy = c.ldy, M = c.M, N = c.N, K = c.K;
  const SkinnyExtra& ex = c.ex;
  hipStream_t stream = c.stream;
  const int blocks = gs_ceil_div(N / 2, 16);
  GS_BY_MT4(2, 8, 8, 4, 4, 0, 4, bf16, blocks)
}

template <int LAYOUT>
static void skinny_residual(const SkinnyCall& c) {
  const bf16 *x = c.x, *w = c.w;
  float* Y = nullptr;
  const int ldx = c.ldx, ldy = c.N, M = c.M, N = c.N, K = c.K;
  const SkinnyExtra& ex = c.ex;
  hipStream_t stream = c.stream;
  const int blocks = gs_ceil_div(N, (LAYOUT & 3) == 2 ? 8 : 16);
  if ((LAYOUT & 3) == 2) { GS_BY_MT(1, 8, 0, 2, float, blocks) }
  else if (K >= 4096) { GS_BY_MT(1, 16, 0, 2, float, blocks) } else { GS_BY_MT(1, 8, 0, 2, float, blocks) }
}

// Partial sums over `parts` parts of K into Y (parts, M, N) float32: two weight tiles a block, four wavefronts.
template <int LAYOUT>
static void skinny_parts(const SkinnyCall& c, int parts) {
  const int blocks = gs_ceil_div(c.N, 32);
  switch ((c.M + 15) / 16) {
    case 1: launch_skinny_parts<2, 1, 4, LAYOUT>(blocks, parts, c.x, c.ldx, c.w, (float*)c.Y, c.M, c.N, c.K, c.ex, c.stream); break;
    case 2: launch_skinny_parts<2, 2, 4, LAYOUT>(blocks, parts, c.x, c.ldx, c.w, (float*)c.Y, c.M, c.N, c.K, c.ex, c.stream); break;
    case 3: launch_skinny_parts<2, 3, 4, LAYOUT>(blocks, parts, c.x, c.ldx, c.w, (float*)c.Y, c.M, c.N, c.K, c.ex, c.stream); break;
    default: launch_skinny_parts<2, 4, 4, LAYOUT>(blocks, parts, c.x, c.ldx, c.w, (float*)c.Y, c.M, c.N, c.K, c.ex, c.stream); break;
  }
}

template <int LAYOUT>
static void skinny_conv(const SkinnyCall& c) {
  const bf16 *x = c.x, *w = c.w;
  void* Y = c.Y;
  const int ldx = c.ldx, ldy = c.ldy, M = c.M, N = c.N, K = c.K;
  const SkinnyExtra& ex = c.ex;
  hipStream_t stream = c.stream;
  const int blocks = gs_ceil_div(N / 3, (LAYOUT & 3) == 2 ? 8 : 16);
  if (ex.res) { GS_BY_MT4(3, 8, 8, 4, 4, 1, 3, bf16, blocks) }
  else if (ex.ssq) { GS_BY_MT4(3, 8, 8, 8, 8, 2, 3, bf16, blocks) }
  else { GS_BY_MT4(3, 8, 8, 8, 8, 0, 3, bf16, blocks) }
}
