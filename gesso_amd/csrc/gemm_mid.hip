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
// last and never stored; K is a multiple of 32, and what a step or a group holds beyond it is loaded but not multiplied (an
// infinite weight times a zero put in its place would be no zero).
//
// EPI 2 (a K too long for one block's chain: a feed-forward's last product): K is shared out over blocks as well, and each stores its
// float32 sums as its part's sheet (parts, M, N); the pass that adds the product to the stream adds the sheets.
//
// EPI 1 (SwiGLU): W holds gate rows [0, N/2), then up rows, N / 2 a multiple of 16; a wavefront owns NT / 2 tiles of gate rows
// and the up rows of the same columns.  silu(gate) * up is taken of the values as they would have been stored.
//
// EPI 3 (a sub-layer's last product): the sums are added to the float32 stream where they arise, and the new rows go out
// weighted for the norm that reads them next, each wavefront's sum of their squares beside them; SCALED: such rows come in, the
// partial sums of squares are asked for before the first weights and added while those travel, and the results are multiplied
// by the rows' inverse root mean squares.  Between the two stands no pass: a layer's output projection, gate and up, and down product
// (1024 wide, 4608 inside; weights in turn, a graph) take 160 rows 32.4 us with the norm's pass and 31.4 without, 72 rows 29.0 and
// 27.5, 333 rows 41.3 and 40.1; 2048 wide and 8192 inside, 72 rows 47.4 and 45.9, 160 rows 56.3 and 55.6.  (Projection, norm, gate and
// up alone, 260 sizes of 65 to 1,000 rows, 512 to 2,048 wide: 0.93 of the three launches in the mean, none more than 1 % above them.)
//
// The groups' sums (KG > 1) are added by two groups, half of the block's rows each: the wavefronts that add, and their loads from
// LDS, are twice as many as with one.  (With room in LDS for all groups' sums, not for the others' alone, a K of 32 to 96 was up to
// 5 % slower than with one group adding: 136 rows of 5472 x 32 4.23 us, so 4.44.)
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 gd_bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float gd_f32x4_t;
typedef __attribute__((ext_vector_type(4))) unsigned gd_u32x4_t;

constexpr int GD_BK = 64, GD_LDR = GD_BK + 8, GD_AHEAD = 4;

// Bytes of LDS: two steps' rows of X a group, and in their place at the end the groups' sums.
constexpr size_t mid_lds(int BM, int NT, int KG) {
  const size_t held = (size_t)KG * 2 * BM * GD_LDR * sizeof(uint16_t), sums = (size_t)(KG - 1) * BM * 64 * NT * sizeof(float);
  return held > sums ? held : sums;
}

constexpr int GD_SSQ_MAX = 128;         // partial sums of squares a row that a SCALED product takes

// What EPI 3 writes (the stream, the next norm's weight, the rows weighted with it, their partial sums of squares) and what SCALED
// reads (partial sums of squares, eps).
struct MidNorm {
  float* res;
  const float* weight;
  bf16* rows;
  float* ssq_out;
  const float* ssq;
  int nssq;
  float eps;
};

template <int BM, int NT, int KG, int EPI, bool SCALED>
__global__ __launch_bounds__(KG * 256) void gemm_mid_kernel(const bf16* __restrict__ X, int ldx, const bf16* __restrict__ Wt,
                                                            bf16* __restrict__ Y, int ldy, int M, int N, int K, int part_steps,
                                                            MidNorm norm) {
  constexpr int TM = BM / 16, LA = BM / 32, STAGE = BM * GD_LDR;           // 16-byte loads of X a thread and step
  constexpr int COLS = 64 * (EPI == 1 ? NT / 2 : NT);                      // columns of Y a block
  constexpr int UM = KG > 1 ? TM / 2 : TM;                                 // row tiles that a group finishes
  constexpr size_t AFTER = mid_lds(BM, NT, KG);                            // bytes of LDS before the rows' inverses
  static_assert(EPI != 1 || NT % 2 == 0, "SwiGLU pairs gate tiles with up tiles");
  extern __shared__ __align__(16) uint16_t gd_lds[];
  const int tid = threadIdx.x & 255, lane = tid & 63, r16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kg = KG > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
  const int F = N >> 1, width = EPI == 1 ? F : N;
  // Blocks go to the eight XCDs in turn, each with an L2 of its own: a run of consecutive tile numbers goes to one XCD, row
  // tiles fastest, so that the tiles that read the same weights read them from one L2.
  const int tiles_m = (M + BM - 1) / BM;
  int bm, bn, part = 0;
  {
    const int nb = (int)gridDim.x, per = nb / 8, rem = nb % 8, xcd = (int)blockIdx.x % 8;
    const int t = xcd * per + (xcd < rem ? xcd : rem) + (int)blockIdx.x / 8;
    bm = t % tiles_m;
    bn = t / tiles_m;
    if (EPI == 2) {
      const int tiles_n = (N + COLS - 1) / COLS;
      part = bn / tiles_n;
      bn %= tiles_n;
    }
  }
  const int m0 = bm * BM, n0 = bn * COLS + wave * (COLS / 4);               // the wavefront's first column
  const int mu = KG > 1 ? m0 + (kg & 1) * (BM / 2) : m0;                    // the first of the rows its group finishes
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
  // the groups' steps: a run each; as many for every group (what lies beyond K is not multiplied)
  const int steps = EPI == 2 ? part_steps : (K + GD_BK - 1) / GD_BK, per = (steps + KG - 1) / KG, first = part * part_steps + kg * per;
  const int kend = EPI == 2 && 2 * (part + 1) * part_steps < ksteps ? 2 * (part + 1) * part_steps : ksteps;
  struct Step {
    gd_u32x4_t a[LA];
    gd_bf16x8_t w[2][NT];
  };
  auto load = [&](Step& s, int step) __attribute__((always_inline)) {
    const int k0 = (first + (step < per ? step : per - 1)) * GD_BK;
    const int k = k0 + c * 8 < K ? k0 + c * 8 : 0;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int at = (k0 >> 5) + ks < ksteps ? (k0 >> 5) + ks : ksteps - 1; // (beyond K: the last weights, not used)
#pragma unroll
      for (int j = 0; j < NT; ++j) s.w[ks][j] = *reinterpret_cast<const gd_bf16x8_t*>(wp[j] + (size_t)at * 512);
    }
#pragma unroll
    for (int i = 0; i < LA; ++i) s.a[i] = *reinterpret_cast<const gd_u32x4_t*>(ap[i] + k);
  };
  uint16_t* mine = gd_lds + (size_t)kg * 2 * STAGE;
  auto put = [&](const Step& s, int buf) __attribute__((always_inline)) {
    uint16_t* to = mine + buf * STAGE + r0 * GD_LDR + c * 8;
#pragma unroll
    for (int i = 0; i < LA; ++i) *reinterpret_cast<gd_u32x4_t*>(to + 32 * i * GD_LDR) = s.a[i];
  };
  gd_f32x4_t acc[TM][NT];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = gd_f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const Step& s, int buf, int step) __attribute__((always_inline)) {
    const int left = kend - 2 * (first + step);          // runs of 32 k from here on (the same for the whole wavefront)
    const uint16_t* a = mine + buf * STAGE + r16 * GD_LDR + g * 8;
    gd_bf16x8_t x[2][TM];                                  // all asked for before the first is used
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < TM; ++i) x[ks][i] = *reinterpret_cast<const gd_bf16x8_t*>(a + 16 * i * GD_LDR + 32 * ks);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      if (ks >= left) break;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(s.w[ks][j], x[ks][i], acc[i][j], 0, 0, 0);
    }
  };
  // EPI 3: the stream's values and the next norm's weights, asked for first: they are there when the sums are
  gd_f32x4_t held[EPI == 3 ? UM : 1][EPI == 3 ? NT : 1], nw[EPI == 3 ? NT : 1];
  constexpr bool ROOM = KG == 1 || NT == 1;               // (else the weights come when the groups' sums are added)
  auto next_weights = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int n = n0 + 16 * j + 4 * g < N ? n0 + 16 * j + 4 * g : N - 4;
      nw[j] = *reinterpret_cast<const gd_f32x4_t*>(norm.weight + n);
    }
  };
  if constexpr (EPI == 3) {
    if constexpr (ROOM) next_weights();
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int n = n0 + 16 * j + 4 * g < N ? n0 + 16 * j + 4 * g : N - 4;
#pragma unroll
      for (int i = 0; i < UM; ++i) {
        const int m = mu + 16 * i + r16 < M ? mu + 16 * i + r16 : M - 1;
        held[i][j] = *reinterpret_cast<const gd_f32x4_t*>(norm.res + (size_t)m * N + n);
      }
    }
  }
  // SCALED: four threads a row, a quarter of its partial sums each (what lies beyond them is loaded from the first and not added;
  // the second half only where there are more than half as many as there may be)
  constexpr int NTH = KG * 256, SR = SCALED ? (BM * 4 + NTH - 1) / NTH : 1, SP = GD_SSQ_MAX / 16;
  gd_f32x4_t sq[SR][SP];
  auto squares_of = [&](int half) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < SR; ++i) {
      const int at = (int)threadIdx.x + i * NTH, m = m0 + (at >> 2) < M ? m0 + (at >> 2) : M - 1;
#pragma unroll
      for (int q = half * SP / 2; q < (half + 1) * SP / 2; ++q) {
        const int p = 4 * ((at & 3) + 4 * q);
        sq[i][q] = *reinterpret_cast<const gd_f32x4_t*>(norm.ssq + (size_t)m * norm.nssq + (p < norm.nssq ? p : 0));
      }
    }
  };
  if constexpr (SCALED) {
#pragma unroll
    for (int i = 0; i < SR; ++i)
#pragma unroll
      for (int q = SP / 2; q < SP; ++q) sq[i][q] = gd_f32x4_t{0.f, 0.f, 0.f, 0.f};
    squares_of(0);
    if (norm.nssq > GD_SSQ_MAX / 2) squares_of(1);
  }
  Step s[GD_AHEAD];
#pragma unroll
  for (int d = 0; d < GD_AHEAD; ++d) load(s[d], d);
  float* inverse = reinterpret_cast<float*>(reinterpret_cast<char*>(gd_lds) + AFTER);       // (SCALED: BM floats)
  if constexpr (SCALED) {
#pragma unroll
    for (int i = 0; i < SR; ++i) {
      const int at = (int)threadIdx.x + i * NTH;
      float sum = 0.f;
#pragma unroll
      for (int q = 0; q < SP; ++q) {
        const float four = (sq[i][q][0] + sq[i][q][1]) + (sq[i][q][2] + sq[i][q][3]);
        sum += 4 * ((at & 3) + 4 * q) < norm.nssq ? four : 0.f;
      }
      sum += dpp_move<0xB1>(sum);
      sum += dpp_move<0x4E>(sum);
      if ((at & 3) == 0 && at < BM * 4) inverse[at >> 2] = norm_inverse(sum, (float)K, norm.eps);
    }
  }
  put(s[0], 0);
  __syncthreads();
  int it = 0;
  // (the last turn asks for the group's last step four times more, which nothing uses: no test stands between the loads)
  for (; it + GD_AHEAD <= per; it += GD_AHEAD) {
#pragma unroll
    for (int d = 0; d < GD_AHEAD; ++d) {
      multiply(s[d], d & 1, it + d);
      load(s[d], it + d + GD_AHEAD);
      __builtin_amdgcn_sched_barrier(0);
      put(s[(d + 1) % GD_AHEAD], (d + 1) & 1);
      __syncthreads();
    }
  }
#pragma unroll
  for (int d = 0; d < GD_AHEAD - 1; ++d)
    if (it + d < per) {                                    // (the same for the whole block)
      multiply(s[d], d & 1, it + d);
      put(s[d + 1], (d + 1) & 1);
      __syncthreads();
    }
  if constexpr (EPI == 3 && !ROOM) next_weights();
  gd_f32x4_t out[UM][NT];
  if constexpr (KG > 1) {
    // the groups' sums, in group order: two groups finish half of the block's rows each.  A half's own group keeps its sums, so
    // the others' have a place each, in order
    float* sums = reinterpret_cast<float*>(gd_lds);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int half = i / UM, place = kg > half ? kg - 1 : kg;
      if (kg == half) continue;                              // (the same for the whole wavefront)
#pragma unroll
      for (int j = 0; j < NT; ++j) *reinterpret_cast<gd_f32x4_t*>(sums + ((place * TM * NT + i * NT + j) * 256 + tid) * 4) = acc[i][j];
    }
    __syncthreads();
    if (kg > 1) return;
#pragma unroll
    for (int i = 0; i < UM; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const float* at = sums + (((kg * UM + i) * NT + j) * 256 + tid) * 4;
        const gd_f32x4_t first = acc[i][j], second = acc[UM + i][j];
        gd_f32x4_t own, each[KG - 1];
#pragma unroll
        for (int e = 0; e < 4; ++e) own[e] = kg == 0 ? first[e] : second[e];       // (of values: of places it would leave the registers)
#pragma unroll
        for (int q = 0; q < KG - 1; ++q) each[q] = *reinterpret_cast<const gd_f32x4_t*>(at + q * TM * NT * 1024);
        out[i][j] = kg == 0 ? own + each[0] : each[0] + own;
#pragma unroll
        for (int q = 1; q < KG - 1; ++q) out[i][j] += each[q];
      }
  } else {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) out[i][j] = acc[i][j];
  }
  // element e of lane l: row 4 (l / 16) + e of W, row l % 16 of X
  if constexpr (EPI == 3) {
    const int tiles_n = (N + COLS - 1) / COLS;
#pragma unroll
    for (int i = 0; i < UM; ++i) {
      const int m = mu + 16 * i + r16;
      float squares = 0.f;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int n = n0 + 16 * j + 4 * g;
        const gd_f32x4_t v = held[i][j] + out[i][j];
        if (m >= M || n >= N) continue;
        *reinterpret_cast<gd_f32x4_t*>(norm.res + (size_t)m * N + n) = v;
        squares += (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
        uint2 o;
        o.x = (uint32_t)f32_to_bf16(v[0] * nw[j][0]).x | ((uint32_t)f32_to_bf16(v[1] * nw[j][1]).x << 16);
        o.y = (uint32_t)f32_to_bf16(v[2] * nw[j][2]).x | ((uint32_t)f32_to_bf16(v[3] * nw[j][3]).x << 16);
        *reinterpret_cast<uint2*>(norm.rows + (size_t)m * N + n) = o;
      }
      squares = group4_sum(squares);                       // (a row's columns lie in four lanes; a tile past the last adds zero)
      if (g == 0 && m < M) norm.ssq_out[(size_t)m * (4 * tiles_n) + bn * 4 + wave] = squares;
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < UM; ++i) {
    const int m = mu + 16 * i + r16;
    if (m >= M) continue;
    const float inv = SCALED ? inverse[mu - m0 + 16 * i + r16] : 1.0f;
#pragma unroll
    for (int j = 0; j < (EPI == 1 ? NT / 2 : NT); ++j) {
      const int n = n0 + 16 * j + 4 * g;
      if (n >= width) continue;                            // (whole tiles: the width is a multiple of 16)
      if (EPI == 2) {
        *reinterpret_cast<gd_f32x4_t*>(reinterpret_cast<float*>(Y) + ((size_t)part * M + m) * N + n) = out[i][j];
        continue;
      }
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = out[i][j][e];
        if (EPI == 1) {
          float uv = out[i][j + (EPI == 1 ? NT / 2 : 0)][e];
          if (SCALED) {
            v[e] *= inv;
            uv *= inv;
          }
          const float gv = to_f32(f32_to_bf16(v[e])), u = to_f32(f32_to_bf16(uv));
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

template <int BM, int NT, int KG, int EPI, bool SCALED = false>
static void run_mid(const bf16* X, int ldx, const bf16* Wt, bf16* Y, int ldy, int M, int N, int K, hipStream_t stream, int parts = 1,
                    MidNorm norm = MidNorm()) {
  const int cols = 64 * (EPI == 1 ? NT / 2 : NT), width = EPI == 1 ? N / 2 : N;
  const long tiles = (long)gs_ceil_div(M, BM) * gs_ceil_div(width, cols) * parts;
  const size_t lds = mid_lds(BM, NT, KG) + (SCALED ? BM * sizeof(float) : 0);
  static const hipError_t asked = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_mid_kernel<BM, NT, KG, EPI, SCALED>),
                                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  (void)asked;
  gemm_mid_kernel<BM, NT, KG, EPI, SCALED><<<(unsigned)tiles, KG * 256, lds, stream>>>(X, ldx, Wt, Y, ldy, M, N, K,
                                                                                       gs_ceil_div(gs_ceil_div(K, GD_BK), parts), norm);
}

// Which tile, and whether this kernel at all.  What a compute unit brings in (some 55 bytes a nanosecond, however the tile is
// cut) is what a product takes beyond 3 to 4 us: the rows of X and W of a block times K, times the rounds in which a unit works
// off its blocks.  So the tile with the least of that is taken.  None for K beyond 2048, where the vendor and the products in parts below share K out over
// blocks (192 rows of 1024 x 4608: 17.1 us here, 13.5 there), and none where the vendor's larger tiles, which read less, win.
// Microseconds here / there (gate and up: with the SwiGLU pass), weights that lie in no cache:
// - plain, one round, up to 2^18 rows times k a unit: 192 rows of 3072 x 1024 8.7 / 13.5, 1024 x 1024 7.1 / 11.0, 2048 x 2048
//   10.5 / 12.4; 1,024 rows of 1024 x 2048 11.9 / 12.5.  Beyond it narrow weights lose (3072 x 2048, 333 rows 15.9 / 15.1, 512
//   17.5 / 15.9), those of 4,096 rows and more win up to 2^19 (6144 x 2048, 150 rows 17.4 / 23.3, 400 23.7 / 24.8).
// - plain, beyond 1,024 rows: up to 3/4 of that to 2,048 rows (2,048 of 1024 x 1024 11.5 / 12.4; 1,280 of 2048 x 1024, 7/8 of it,
//   13.5 / 13.4), half of it beyond (3,072 of 512 x 512 7.7 / 10.2; of 512 x 1024 12.3 / 11.9, of 1024 x 1024 14.3 / 13.4).
// - plain, more than a round: never (2,048 rows of 2048 x 1024 21.8 / 14.4, 512 of 9216 x 1024 26.3 / 20.3, 333 of 9216 x 96
//   10.2 / 7.2).
// - gate and up, one round: up to 2^19 (333 rows of 9216 x 1024 17.3 / 22.0, 192 of 16384 x 2048 28.2 / 35.4; the worst found:
//   128 rows of 1024 x 2048 14.1 / 13.4).  Two and three: up to 7/8 of it (512 of 12288 x 768 22.0 / 24.6; 512 of 9216 x 1024, at
//   7/8, 26.9 / 25.5).  More: no (1,280 of 8192 x 384 28.5 / 27.5, 640 of 16384 x 160 23.6 / 21.6).
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
  long least = (1L << 19) + 1, rounds = 0;
  for (int i = 0; i < n; ++i) {
    const long blocks = (long)gs_ceil_div(M, t[i].bm) * gs_ceil_div(width, 64 * (epilogue == 1 ? t[i].nt / 2 : t[i].nt));
    const long r = (blocks + 255) / 256, cost = r * (t[i].bm + 64 * t[i].nt) * K;
    if (cost < least) {
      least = cost;
      rounds = r;
      best = i;
    }
  }
  if (epilogue == 1) return rounds == 1 || (rounds <= 3 && least < 7L << 16) ? best : -1;
  const long limit = M > 2048 ? 1L << 17 : M > 1024 ? 3L << 16 : N < 4096 ? 1L << 18 : 1L << 19;
  return rounds == 1 && least <= limit ? best : -1;
}

// Whether the product is this kernel's, M rows against a tile-major weight (N, K): the number of its tile, from 1 on, or 0.
extern "C" int gs_gemm_mid_takes(int M, int N, int K, int epilogue) {
  return K > 0 && K % 32 == 0 && N > 0 && N % (epilogue == 1 ? 32 : 16) == 0 ? mid_choice(M, N, K, epilogue) + 1 : 0;
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

// Y (M, N / 2) = silu(X Wg^T) * (X Wu^T) of rows that are weighted for a norm but not yet scaled: ssq (M, nssq) holds partial sums of
// the rows' squares, nssq a multiple of four up to 128.  The products of gs_gemm_mid's epilogue 1.
extern "C" int gs_gemm_mid_swiglu_scaled(const void* X, int ldx, const float* ssq, int nssq, float eps, const void* Wt, void* Y, int ldy,
                                         int M, int N, int K, hipStream_t stream) {
  GS_REQUIRE(gs_gemm_mid_takes(M, N, K, 1), "gemm_mid_swiglu_scaled: not a product of this kernel (M=%d N=%d K=%d)", M, N, K);
  GS_REQUIRE(ldx >= K && ldx % 8 == 0 && (((uintptr_t)X | (uintptr_t)Wt | (uintptr_t)ssq) & 15) == 0,
             "gemm_mid_swiglu_scaled: X, W and the sums must be 16-byte aligned, the row stride of X a multiple of 8");
  GS_REQUIRE(ssq && nssq > 0 && nssq % 4 == 0 && nssq <= GD_SSQ_MAX && eps > 0.f, "gemm_mid_swiglu_scaled: %d partial sums a row, eps %g", nssq, eps);
  GS_REQUIRE(ldy >= N / 2 && ldy % 4 == 0 && ((uintptr_t)Y & 7) == 0, "gemm_mid_swiglu_scaled: rows of Y too short or not aligned (stride %d)", ldy);
  const bf16 *x = (const bf16*)X, *w = (const bf16*)Wt;
  bf16* y = (bf16*)Y;
  MidNorm norm = {};
  norm.ssq = ssq;
  norm.nssq = nssq;
  norm.eps = eps;
#define GD_RUN(BM, NT, KG) run_mid<BM, NT, KG, 1, true>(x, ldx, w, y, ldy, M, N, K, stream, 1, norm)
  const int i = mid_choice(M, N, K, 1);
  if (i == 0) GD_RUN(32, 2, 2); else if (i == 1) GD_RUN(64, 2, 1); else if (i == 2) GD_RUN(96, 2, 1); else GD_RUN(64, 4, 1);
#undef GD_RUN
  GS_LAUNCH_CHECK("gemm_mid_swiglu_scaled");
  return 0;
}

// How many partial sums of squares a row gs_gemm_mid_residual leaves; 0: the product is not its, or they are more than the product that
// reads them takes.
extern "C" int gs_gemm_mid_residual_sums(int M, int N, int K) {
  if (!gs_gemm_mid_takes(M, N, K, 0)) return 0;
  const int sums = 4 * gs_ceil_div(N, 64 * mid_plain[mid_choice(M, N, K, 0)].nt);
  return sums <= GD_SSQ_MAX ? sums : 0;
}

// res (M, N) += X W^T in float32; rows (M, N) = res * next_weight in bfloat16 and ssq (M, gs_gemm_mid_residual_sums) partial sums of the
// new rows' squares.
extern "C" int gs_gemm_mid_residual(const void* X, int ldx, const void* Wt, float* res, const float* next_weight, void* rows, float* ssq,
                                    int M, int N, int K, hipStream_t stream) {
  GS_REQUIRE(gs_gemm_mid_residual_sums(M, N, K) > 0, "gemm_mid_residual: not a product of this kernel (M=%d N=%d K=%d)", M, N, K);
  GS_REQUIRE(ldx >= K && ldx % 8 == 0 && (((uintptr_t)X | (uintptr_t)Wt | (uintptr_t)res | (uintptr_t)next_weight) & 15) == 0 && ((uintptr_t)rows & 7) == 0,
             "gemm_mid_residual: X, W, the stream and the weight must be 16-byte aligned, the row stride of X a multiple of 8");
  GS_REQUIRE(res && next_weight && rows && ssq, "gemm_mid_residual: needs the stream, the next norm's weight, its rows and their sums");
  const bf16 *x = (const bf16*)X, *w = (const bf16*)Wt;
  MidNorm norm = {};
  norm.res = res;
  norm.weight = next_weight;
  norm.rows = (bf16*)rows;
  norm.ssq_out = ssq;
#define GD_RUN(BM, NT, KG) run_mid<BM, NT, KG, 3>(x, ldx, w, nullptr, 0, M, N, K, stream, 1, norm)
  switch (mid_choice(M, N, K, 0)) {
    case 0: GD_RUN(32, 1, 4); break;
    case 1: GD_RUN(64, 1, 2); break;
    case 2: GD_RUN(96, 1, 2); break;
    case 3: GD_RUN(64, 2, 2); break;
    default: GD_RUN(96, 2, 1); break;
  }
#undef GD_RUN
  GS_LAUNCH_CHECK("gemm_mid_residual");
  return 0;
}

// The product in parts of K: which tile and how many parts.  As above, a unit's rows of X and W times k bind, and a sheet is written
// and read once more (counted as the rows times k that take as long; at a quarter of that, 160 rows of 1024 x 4608 took 15 parts and 15.8
// us); none beyond what one round of blocks holds.
struct MidParts {
  int tile, parts;
};
static MidParts mid_parts_choice(int M, int N, int K) {
  MidParts best = {-1, 0};
  if (M <= 64 || K <= 2048 || N > 4096 || M > (N <= 2048 ? 768 : 256)) return best;
  const int steps = gs_ceil_div(K, GD_BK);
  long least = 0;
  for (int i = 0; i < 5; ++i) {
    const long tiles = (long)gs_ceil_div(M, mid_plain[i].bm) * gs_ceil_div(N, 64 * mid_plain[i].nt);
    for (int parts = 2; parts <= 16 && parts * tiles <= 256; ++parts) {
      const int each = gs_ceil_div(steps, parts);
      if (each < 4 || (long)(parts - 1) * each >= steps) continue;      // (no part without a step)
      const long cost = (long)(mid_plain[i].bm + 64 * mid_plain[i].nt) * each * GD_BK + (long)parts * M * N / 16;
      if (best.parts == 0 || cost < least) {
        least = cost;
        best = {i, parts};
      }
    }
  }
  return best;
}

// Into how many parts of K the product of M rows with a tile-major weight (N, K) is shared out; 0: it is not this kernel's.
extern "C" int gs_gemm_mid_parts_takes(int M, int N, int K) {
  return K > 0 && K % 32 == 0 && N > 0 && N % 16 == 0 ? mid_parts_choice(M, N, K).parts : 0;
}

// Whether that is faster than the vendor's product and the plain pass, by measurement of both with the pass that adds and norms:
// 1,242 products of 65 to 768 rows, 14 widths of W from 256 to 4,096 and K from 2,304 to 14,336, weights that lie in no cache (700 MB of
// them in turn; where some 200 MB stay in the last-level cache the vendor's gain more).  Of the 877 taken here 5 are slower,
// by 2 % at most; together they take 0.75 of the vendor's time, the others would take 1.02.  The vendor's time over this one's:
// - up to 1,024 rows of W: 1.02 and more, at any K (1024 x 4608: 65 rows 1.49, 160 1.31, 768 1.18);
// - 2,048 and 4,096 rows: the more rows of X the longer K has to be (2048 x 8192, 65 rows 1.46, 512 1.04; 2048 x 2304, 320 rows 1.05,
//   448 0.93; 2048 x 3072, 512 rows 1.02, 768 0.96; 4096 x 2304, 160 rows 1.23, 256 0.93);
// - others up to 2,048 rows, whose tiles suit the vendor: from a K of 6,144 on, for up to 96 rows of X of 10,240 (1280 x 4608,
//   65 rows 0.95, 320 0.95; 1280 x 7168, 128 rows 1.23; 1280 x 8192, 65 rows 0.85; 1536 x 6144, 512 rows 1.00, 768 0.97);
// - others beyond: the vendor's step from 96 to 128 rows of X is large (2560 x 3072, 96 rows 0.80, 128 1.38; 3584 x 3072, 160 rows 1.25,
//   200 0.90); else from a K of 4,608, 6,144 or 10,240 on (2304 x 4608, 65 rows 0.97, 2304 x 6144 1.10; 3072 x 3072, 256 rows 0.90, 3072 x
//   11008 1.15).
static bool mid_parts_pay(int M, int N, int K) {
  if (N <= 1024) return true;
  if ((N & (N - 1)) == 0) return M <= (N > 2048 ? 160 : 320) || (M <= 512 && K >= 3072) || K >= 4096;
  if (N < 2048) return (M > 96 && M <= 384 && K >= 6144) || (M <= 640 && K >= 10240);
  if (M > 96 && M <= (N < 3328 ? 128 : 160)) return true;
  return N < 2816 ? K >= 6144 : (M <= 128 && K >= 4608) || (M <= 160 && K >= 6144) || K >= 10240;
}

// The same, 0 also where the vendor's product is the faster one.
extern "C" int gs_gemm_mid_parts_pay(int M, int N, int K) { return mid_parts_pay(M, N, K) ? gs_gemm_mid_parts_takes(M, N, K) : 0; }

// part (parts, M, N) float32 = partial sums of X W^T over gs_gemm_mid_parts_takes parts of K; gs_residual_from_parts adds them up.
extern "C" int gs_gemm_mid_parts(const void* X, int ldx, const void* Wt, float* part, int parts, int M, int N, int K, hipStream_t stream) {
  GS_REQUIRE(parts > 0 && gs_gemm_mid_parts_takes(M, N, K) == parts, "gemm_mid_parts: not a product of this kernel in %d parts (M=%d N=%d K=%d)", parts, M, N, K);
  GS_REQUIRE(ldx >= K && ldx % 8 == 0 && (((uintptr_t)X | (uintptr_t)Wt | (uintptr_t)part) & 15) == 0,
             "gemm_mid_parts: X, W and the sheets must be 16-byte aligned, the row stride of X a multiple of 8");
  const bf16 *x = (const bf16*)X, *w = (const bf16*)Wt;
  bf16* y = (bf16*)part;
#define GD_RUN(BM, NT, KG) run_mid<BM, NT, KG, 2>(x, ldx, w, y, N, M, N, K, stream, parts)
  switch (mid_parts_choice(M, N, K).tile) {
    case 0: GD_RUN(32, 1, 4); break;
    case 1: GD_RUN(64, 1, 2); break;
    case 2: GD_RUN(96, 1, 2); break;
    case 3: GD_RUN(64, 2, 2); break;
    default: GD_RUN(96, 2, 1); break;
  }
#undef GD_RUN
  GS_LAUNCH_CHECK("gemm_mid_parts");
  return 0;
}
