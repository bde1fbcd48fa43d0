// Y (M, N) = X (M, K) . W (N, K)^T for some hundred rows, with an optional SwiGLU epilogue: prompt portions of a few hundred
// tokens, the decode loop of more requests than the weight-streaming products take.
//
// bfloat16 inputs, float32 accumulation (v_mfma_f32_16x16x32_bf16), bfloat16 output.  Neither the matrix cores nor the weights'
// bytes bind here but the chain of steps over K and what a compute unit can bring in a step: 150 rows of 1024 x 1024 are
// 0.1 us of products and 0.4 us of weights.  So the weight is read from its tile-major copy, each load a contiguous kilobyte
// straight in the operand's order, by the one wavefront that owns those rows (four wavefronts side by side in N, NT tiles of
// 16 rows each), and only the rows of X go through LDS, for all four (rows of 64 + 8 elements: the sixteen rows that a read
// touches lie in different banks).  The loads of a step of 64 k are issued four steps ahead, into registers.  Where the tiles
// alone do not fill the chip a block's KG groups of four wavefronts share K out, their sums added through LDS in group order.
// (Both operands through LDS, 64 x 64 tiles: 0.3 us a step however many groups, 350M sizes at 192 rows: gate and up 13.3 us.)
//
// W's rows are the products' rows, so that a lane ends with four neighbouring columns of Y.  Rows beyond M are read from the
// last and never stored; K is a multiple of 32, pieces beyond it count as zeros.
//
// EPI 1 (SwiGLU): W holds gate rows [0, N/2), then up rows, N / 2 a multiple of 16; a wavefront owns NT / 2 tiles of gate rows
// and the up rows of the same columns.  silu(gate) * up is taken of the values as they would have been stored.
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 gd_bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float gd_f32x4_t;
typedef __attribute__((ext_vector_type(4))) unsigned gd_u32x4_t;

constexpr int GD_BK = 64, GD_LDR = GD_BK + 8, GD_AHEAD = 4;

template <int BM, int NT, int KG, int EPI>
__global__ __launch_bounds__(KG * 256) void gemm_mid_kernel(const bf16* __restrict__ X, int ldx, const bf16* __restrict__ Wt,
                                                            bf16* __restrict__ Y, int ldy, int M, int N, int K) {
  constexpr int TM = BM / 16, LA = BM / 32, STAGE = BM * GD_LDR;           // 16-byte loads of X a thread and step
  constexpr int COLS = 64 * (EPI == 1 ? NT / 2 : NT);                      // columns of Y a block
  static_assert(EPI == 0 || NT % 2 == 0, "SwiGLU pairs gate tiles with up tiles");
  extern __shared__ __align__(16) uint16_t gd_lds[];
  const int tid = threadIdx.x & 255, lane = tid & 63, r16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kg = KG > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
  const int F = N >> 1, width = EPI == 1 ? F : N;
  // Blocks go to the eight XCDs in turn, each with an L2 of its own: a run of consecutive tile numbers goes to one XCD, row
  // tiles fastest, so that the tiles that read the same weights read them from one L2.
  const int tiles_m = (M + BM - 1) / BM;
  int bm, bn;
  {
    const int nb = (int)gridDim.x, per = nb / 8, rem = nb % 8, xcd = (int)blockIdx.x % 8;
    const int t = xcd * per + (xcd < rem ? xcd : rem) + (int)blockIdx.x / 8;
    bm = t % tiles_m;
    bn = t / tiles_m;
  }
  const int m0 = bm * BM, n0 = bn * COLS + wave * (COLS / 4);               // the wavefront's first column
  const int r0 = tid >> 3, c = tid & 7;                                     // this thread's loads: row r0 + 32 i, piece c of eight k
  const bf16* ap[LA];
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    const int m = m0 + r0 + 32 * i;
    ap[i] = X + (size_t)(m < M ? m : M - 1) * ldx;
  }
  const int ksteps = K >> 5;
  const bf16* wp[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    int n = EPI == 1 ? n0 + 16 * (j % (NT / 2)) : n0 + 16 * j;
    n = n < width ? n : width - 16;                                         // (a tile past the last reads the last and stores nothing)
    if (EPI == 1 && j >= NT / 2) n += F;
    wp[j] = Wt + (size_t)(n >> 4) * ksteps * 512 + lane * 8;
  }
  // the groups' steps: a run each; as many for every group (steps beyond K: zeros)
  const int steps = (K + GD_BK - 1) / GD_BK, per = (steps + KG - 1) / KG, first = kg * per;
  struct Step {
    gd_u32x4_t a[LA];
    gd_bf16x8_t w[2][NT];
  };
  auto load = [&](Step& s, int step) __attribute__((always_inline)) {
    const int k0 = (first + (step < per ? step : per - 1)) * GD_BK;
    const int k = k0 + c * 8 < K ? k0 + c * 8 : 0;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int at = (k0 >> 5) + ks < ksteps ? (k0 >> 5) + ks : ksteps - 1; // (beyond K: any weights, X's pieces are zeros)
#pragma unroll
      for (int j = 0; j < NT; ++j) s.w[ks][j] = *reinterpret_cast<const gd_bf16x8_t*>(wp[j] + (size_t)at * 512);
    }
#pragma unroll
    for (int i = 0; i < LA; ++i) s.a[i] = *reinterpret_cast<const gd_u32x4_t*>(ap[i] + k);
  };
  uint16_t* mine = gd_lds + (size_t)kg * 2 * STAGE;
  // (zeros for what lies beyond K are put in here: where the load is issued they would wait for it)
  auto put = [&](const Step& s, int buf, int step) __attribute__((always_inline)) {
    const bool in = (first + step) * GD_BK + c * 8 < K;
    uint16_t* to = mine + buf * STAGE + r0 * GD_LDR + c * 8;
#pragma unroll
    for (int i = 0; i < LA; ++i) *reinterpret_cast<gd_u32x4_t*>(to + 32 * i * GD_LDR) = in ? s.a[i] : gd_u32x4_t{0u, 0u, 0u, 0u};
  };
  gd_f32x4_t acc[TM][NT];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = gd_f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const Step& s, int buf) __attribute__((always_inline)) {
    const uint16_t* a = mine + buf * STAGE + r16 * GD_LDR + g * 8;
    gd_bf16x8_t x[2][TM];                                  // all asked for before the first is used
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < TM; ++i) x[ks][i] = *reinterpret_cast<const gd_bf16x8_t*>(a + 16 * i * GD_LDR + 32 * ks);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(s.w[ks][j], x[ks][i], acc[i][j], 0, 0, 0);
  };
  Step s[GD_AHEAD];
#pragma unroll
  for (int d = 0; d < GD_AHEAD; ++d) load(s[d], d);
  put(s[0], 0, 0);
  __syncthreads();
  int it = 0;
  for (; it + GD_AHEAD <= per; it += GD_AHEAD) {
#pragma unroll
    for (int d = 0; d < GD_AHEAD; ++d) {
      multiply(s[d], d & 1);
      load(s[d], it + d + GD_AHEAD);
      __builtin_amdgcn_sched_barrier(0);
      put(s[(d + 1) % GD_AHEAD], (d + 1) & 1, it + d + 1);
      __syncthreads();
    }
  }
#pragma unroll
  for (int d = 0; d < GD_AHEAD - 1; ++d)
    if (it + d < per) {                                    // (the same for the whole block)
      multiply(s[d], d & 1);
      put(s[d + 1], (d + 1) & 1, it + d + 1);
      __syncthreads();
    }
  if (KG > 1) {
    // the other groups' sums, tile after tile, in group order
    float* sums = reinterpret_cast<float*>(gd_lds);
    if (kg > 0) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          *reinterpret_cast<gd_f32x4_t*>(sums + (((kg - 1) * TM * NT + i * NT + j) * 256 + tid) * 4) = acc[i][j];
    }
    __syncthreads();
    if (kg > 0) return;
    for (int q = 0; q < KG - 1; ++q)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[i][j] += *reinterpret_cast<const gd_f32x4_t*>(sums + ((q * TM * NT + i * NT + j) * 256 + tid) * 4);
  }
  // element e of lane l: row 4 (l / 16) + e of W, row l % 16 of X
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + 16 * i + r16;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < (EPI == 1 ? NT / 2 : NT); ++j) {
      const int n = n0 + 16 * j + 4 * g;
      if (n >= width) continue;                            // (whole tiles: the width is a multiple of 16)
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = acc[i][j][e];
        if (EPI == 1) {
          const float gv = to_f32(f32_to_bf16(v[e])), u = to_f32(f32_to_bf16(acc[i][j + (EPI == 1 ? NT / 2 : 0)][e]));
          v[e] = gv / (1.0f + expf(-gv)) * u;
        }
      }
      uint2 o;
      o.x = (uint32_t)f32_to_bf16(v[0]).x | ((uint32_t)f32_to_bf16(v[1]).x << 16);
      o.y = (uint32_t)f32_to_bf16(v[2]).x | ((uint32_t)f32_to_bf16(v[3]).x << 16);
      *reinterpret_cast<uint2*>(Y + (size_t)m * ldy + n) = o;
    }
  }
}

template <int BM, int NT, int KG, int EPI>
static void run_mid(const bf16* X, int ldx, const bf16* Wt, bf16* Y, int ldy, int M, int N, int K, hipStream_t stream) {
  const int cols = 64 * (EPI == 1 ? NT / 2 : NT), width = EPI == 1 ? N / 2 : N;
  const long tiles = (long)gs_ceil_div(M, BM) * gs_ceil_div(width, cols);
  const size_t held = (size_t)KG * 2 * BM * GD_LDR * sizeof(uint16_t), sums = (size_t)(KG - 1) * BM * 64 * NT * sizeof(float);
  const size_t lds = held > sums ? held : sums;
  static const hipError_t asked = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_mid_kernel<BM, NT, KG, EPI>),
                                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  (void)asked;
  gemm_mid_kernel<BM, NT, KG, EPI><<<(unsigned)tiles, KG * 256, lds, stream>>>(X, ldx, Wt, Y, ldy, M, N, K);
}

// Which tile, and whether this kernel at all.  What a compute unit brings in (some 55 bytes a nanosecond, however the tile is
// cut) is what a product takes beyond 3 to 4 us: the rows of X and W of a block times K, times the blocks a unit works off one
// after the other.  So the tile with the least of that is taken, and none where it comes to more than 2^19 rows times k, some
// 28 us: from there on the vendor's larger tiles read less (512 rows of 6144 x 2048: 28.5 us here, 26.3 there; 333 of gate
// and up, 16384 x 2048: 43 and 40 with the SwiGLU pass), nor for K beyond 2048, where it shares K out over blocks (192 rows
// of 1024 x 4608: 17.1 and 13.5).  Below, microseconds here and there (gate and up with the SwiGLU pass), 192 rows:
//   3072 x 1024 8.1 / 13.2, 1024 x 1024 5.6 / 8.0, 9216 x 1024 gate and up 11.5 / 19.3;
//   6144 x 2048 16.5 / 22.4, 2048 x 2048 9.8 / 12.0, 16384 x 2048 gate and up 27 / 34;
// 96 rows: 7.4 / 11.9, 5.6 / 8.0, 10.0 / 16.4; 13.2 / 14.3, 9.9 / 11.4, 22.6 / 24.1;
// 333 rows: 10.3 / 13.7, 5.8 / 8.5, 16.0 / 21.1; 22.8 / 25.5, 11.3 / 12.8.
struct MidTile {
  int bm, nt;
};
static const MidTile mid_plain[] = {{32, 1}, {64, 1}, {96, 1}, {64, 2}, {96, 2}};
static const MidTile mid_swiglu[] = {{32, 2}, {64, 2}, {96, 2}, {64, 4}};

static int mid_choice(int M, int N, int K, int epilogue) {
  if (M <= 64 || K > 2048) return -1;
  const MidTile* t = epilogue == 1 ? mid_swiglu : mid_plain;
  const int n = epilogue == 1 ? 4 : 5, width = epilogue == 1 ? N / 2 : N;
  int best = -1;
  long least = (1L << 19) + 1;
  for (int i = 0; i < n; ++i) {
    const long blocks = (long)gs_ceil_div(M, t[i].bm) * gs_ceil_div(width, 64 * (epilogue == 1 ? t[i].nt / 2 : t[i].nt));
    const long cost = (blocks + 255) / 256 * (t[i].bm + 64 * t[i].nt) * K;
    if (cost < least) {
      least = cost;
      best = i;
    }
  }
  return best;
}

// Whether the product is this kernel's: M rows against a tile-major weight (N, K).
extern "C" int gs_gemm_mid_takes(int M, int N, int K, int epilogue) {
  return K > 0 && K % 32 == 0 && N > 0 && N % (epilogue == 1 ? 32 : 16) == 0 && mid_choice(M, N, K, epilogue) >= 0;
}

// epilogue 0: Y (M, N) = X W^T; epilogue 1: Y (M, N / 2) = silu(X Wg^T) * (X Wu^T).  Wt: the weight's tile-major copy.
extern "C" int gs_gemm_mid(const void* X, int ldx, const void* Wt, void* Y, int ldy, int M, int N, int K, int epilogue,
                           hipStream_t stream) {
  GS_REQUIRE(epilogue == 0 || epilogue == 1, "gemm_mid: unknown epilogue %d", epilogue);
  GS_REQUIRE(gs_gemm_mid_takes(M, N, K, epilogue), "gemm_mid: not a product of this kernel (M=%d N=%d K=%d)", M, N, K);
  GS_REQUIRE(ldx >= K && ldx % 8 == 0 && ((uintptr_t)X & 15) == 0 && ((uintptr_t)Wt & 15) == 0,
             "gemm_mid: X and W must be 16-byte aligned, the row stride of X a multiple of 8");
  GS_REQUIRE(ldy >= (epilogue == 1 ? N / 2 : N) && ldy % 4 == 0 && ((uintptr_t)Y & 7) == 0,
             "gemm_mid: rows of Y too short or not aligned (stride %d)", ldy);
  const bf16 *x = (const bf16*)X, *w = (const bf16*)Wt;
  bf16* y = (bf16*)Y;
#define GD_RUN(BM, NT, KG, EPI) run_mid<BM, NT, KG, EPI>(x, ldx, w, y, ldy, M, N, K, stream)
  // (two or four groups share K where a block's registers allow: 96 rows by two weight tiles leave no room for a second)
  const int i = mid_choice(M, N, K, epilogue);
  if (epilogue == 1) {
    if (i == 0) GD_RUN(32, 2, 2, 1); else if (i == 1) GD_RUN(64, 2, 1, 1); else if (i == 2) GD_RUN(96, 2, 1, 1); else GD_RUN(64, 4, 1, 1);
  } else {
    if (i == 0) GD_RUN(32, 1, 4, 0); else if (i == 1) GD_RUN(64, 1, 2, 0); else if (i == 2) GD_RUN(96, 1, 2, 0);
    else if (i == 3) GD_RUN(64, 2, 2, 0); else GD_RUN(96, 2, 1, 0);
  }
#undef GD_RUN
  GS_LAUNCH_CHECK("gemm_mid");
  return 0;
}
