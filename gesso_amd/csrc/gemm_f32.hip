// y = x W^T (+ bias), everything float32, on the matrix cores: the true 32-bit path's product.
//
// v_mfma_f32_16x16x4_f32 multiplies float32 operands without rounding them and adds its four products to the accumulator
// one after the other in ascending k, each with one rounding: a chain of FMAs.  So an output here is summed in the order of
// the tiled FMA kernel (gemm_tiled.hip): k in chunks of GS_SUM_CHUNK = 64, each from zero in ascending k, the chunks' sums
// added in ascending order.  Its value depends neither on which kernel computed it nor on the rows beside it.
//
// The instruction wants row l % 16 and k = l / 16 of a tile in lane l.  Loaded like that from rows in memory, sixteen lanes
// in a row of the wavefront ask sixteen lines at a time, and a compute unit gets some 8 bytes a cycle whatever it loads
// (2048 x 8192 weights, 6 rows: 28 us, of which the weights alone 21); so a wavefront loads whole runs of a row, sixteen
// lanes 256 bytes, and puts them in order through LDS (rows 4 numbers further apart than their length: no bank twice).
//
// Few rows (up to 64): gemm_f32_rows_kernel.  The weights bind, so each is read once: a block owns 8 or 16 rows of W and
// its eight wavefronts take the chunks in turns, one or two at a time, D turns in flight each; the chunk sums go to LDS, and one thread an output
// adds them in order.  W is loaded non-temporally (six requests, a prompt of 150 and sixteen tokens each at LFM2-1.2B sizes: 42.7 ms against 46.1).
//
// A few rows where that kernel's blocks bind, or the way through LDS and sixteen products in a chain: gemm_f32_lanes_kernel, by
// FMAs, a lane a chunk.  With a K of a chunk or two most of a block of eight wavefronts has nothing to do, and there are many blocks
// (1 row, 65536 x 64: 20 us, by lanes 6.6); with few weight rows and a long K there are too few blocks to hide the chain.
//
// Many rows: gemm_f32_tiles_kernel.  The matrix cores bind (157 TFLOP/s): a block's 2 x WN wavefronts own MT x NT tiles of 16 x 16
// each.  A wavefront always has products to issue: rows are asked for two steps of 32 k ahead (or four), the next step's rows go to LDS half
// way through a step, operands are read from LDS under the products of the k before, and the step's barrier stands before its last
// products, with the next step's first operands asked for behind it.  (Written without fences between these, the compiler moved
// the loads down to where their values are stored: 680 rows of 2048 x 8192 292 us, now 231.)  32 x 32 x 2 instructions give the same
// chains and, alone, 3 % more; with their operands through LDS they were slower (2,048 rows of 16384 x 2048 1,130 us, these 1,050).
#include "common.h"

typedef __attribute__((ext_vector_type(4))) float gf_f32x4_t;

#define GF_WAVES 8

// Four values from k on of a row of K (K a multiple of 4); nothing beyond K is read.  TAIL: k may lie beyond K (zeros).
// ONCE: no other compute unit reads the line.
template <bool TAIL, bool ONCE = false>
__device__ __forceinline__ gf_f32x4_t gf_load(const float* __restrict__ row, int k, int K) {
  const gf_f32x4_t* p = reinterpret_cast<const gf_f32x4_t*>(row + (!TAIL || k < K ? k : 0));
  const gf_f32x4_t v = ONCE ? __builtin_nontemporal_load(p) : *p;
  if (!TAIL) return v;
  return k < K ? v : gf_f32x4_t{0.f, 0.f, 0.f, 0.f};
}

// WR: rows of W a block owns (8 or 16), XR: rows of X (4, 8, or tiles of 16), D: turns a wavefront holds in flight, of CH chunks each.
// GLU: W holds N / 2 gate rows, then as many up rows; a block takes WR / 2 of each, a gate's sum and its up's end WR / 2 lanes apart, and
// silu(gate) * up is stored, N / 2 wide.  SPARE: sums that nobody keeps are stored behind the others, not left out.  (A pass of its own was a launch a layer and the 16384-wide rows
// out and in again: a decode step of 6 requests, 16 such layers, LFM2-1.2B sizes in float32, 1.295 ms, now 1.257.)
template <int WR, int XR, int D, int CH, bool TAIL, typename TO, bool GLU, bool SPARE = false>
__global__ __launch_bounds__(GF_WAVES * 64) void gemm_f32_rows_kernel(const float* __restrict__ X, int ldx,
                                                                      const float* __restrict__ W,
                                                                      const float* __restrict__ bias, TO* __restrict__ Y,
                                                                      int ldy, int M, int N, int K, int room) {
  constexpr int MT = XR > 16 ? XR / 16 : 1, XT = XR < 16 ? XR : 16;       // tiles of X, rows used of each
  // CH = 2, half a tile of W and half a tile of X: two chunks share the instructions, the second in the tiles' other halves; its sums come out in
  // the opposite quarter, the other two hold nothing.  (One chunk at a time is sixteen products of 32 cycles in a chain, more than the
  // weights take: a decode step's kernels of 6 rows, microseconds one and two at a time: 2048 x 8192 and 2048 x 2048 13.0 and 10.7 in
  // the mean, 6144 x 2048 14.1 and 12.1, 3072 x 2048 10.0 and 8.3.)
  static_assert(CH == 1 || (CH == 2 && WR == 8 && XR <= 8), "two chunks share the halves of a tile");
  constexpr int OUT = MT * XT * WR, PER = (OUT + GF_WAVES * 64 - 1) / (GF_WAVES * 64);
  constexpr int LD = GS_SUM_CHUNK + 4;
  extern __shared__ float sums[];                                         // chunk sums of a pass: `room` of OUT numbers
  __shared__ float order[GF_WAVES][16 * LD];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * (GLU ? WR / 2 : WR), rows = GLU ? N >> 1 : N;      // the block's first output, and how many there are
  // lane l loads the four k at 4 (l % 16) of row l / 16 of four
  const float* wp[WR / 4];
  const float* xp[MT][XT / 4];
#pragma unroll
  for (int j = 0; j < WR / 4; ++j) {
    const int up = GLU && j >= WR / 8, n = n0 + 4 * j + g - up * (WR / 2);
    wp[j] = W + (size_t)(up * rows + (n < rows ? n : rows - 1)) * K;
  }
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < XT / 4; ++j) xp[i][j] = X + (size_t)(16 * i + 4 * j + g < M ? 16 * i + 4 * j + g : M - 1) * ldx;
  const int chunks = (K + GS_SUM_CHUNK - 1) / GS_SUM_CHUNK;

  struct Chunk {
    gf_f32x4_t w[CH][WR / 4], x[CH][MT][XT / 4];
  };
  auto load = [&](Chunk& b, int c, int last) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < CH; ++h) {
      const int k = (CH == 1 || c + h < last ? c + h : last) * GS_SUM_CHUNK + 4 * r16;
#pragma unroll
      for (int j = 0; j < WR / 4; ++j) b.w[h][j] = gf_load<TAIL, true>(wp[j], k, K);
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < XT / 4; ++j) b.x[h][i][j] = gf_load<TAIL>(xp[i][j], k, K);
    }
  };
  float* mine = order[wave];
  float* put = mine + g * LD + 4 * r16;           // where a lane leaves what it loaded, four rows a load
  const float* get = mine + r16 * LD + g;         // and where it finds its operands, four numbers apart
  // (a tile of fewer rows than sixteen leaves the others as they are: they end in outputs nobody keeps)
  auto multiply = [&](Chunk& b, int c, int keep) __attribute__((always_inline)) {     // keep: how many of the chunks from c on are there
    float w[16];
#pragma unroll
    for (int h = 0; h < CH; ++h)
#pragma unroll
      for (int j = 0; j < WR / 4; ++j) *reinterpret_cast<gf_f32x4_t*>(put + (8 * h + 4 * j) * LD) = b.w[h][j];
#pragma unroll
    for (int q = 0; q < 16; ++q) w[q] = get[4 * q];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      float x[16];
#pragma unroll
      for (int h = 0; h < CH; ++h)
#pragma unroll
        for (int j = 0; j < XT / 4; ++j) *reinterpret_cast<gf_f32x4_t*>(put + (8 * h + 4 * j) * LD) = b.x[h][i][j];
#pragma unroll
      for (int q = 0; q < 16; ++q) x[q] = get[4 * q];
      gf_f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q < 16; ++q) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[q], x[q], acc, 0, 0, 0);
      // element e of lane l: row 4 (l / 16) + e of W, row l % 16 of X: X's row after X's row, WR numbers each
      const int h = CH == 2 ? r16 >> 3 : 0, m = CH == 2 ? r16 & 7 : r16, n = CH == 2 ? 4 * g - 8 * h : 4 * g;
      const bool kept = h < keep && n >= 0 && n < WR && m < XT;
      float* at = sums + (c + h) * OUT + (i * XT + m) * WR + n;
      if (SPARE) at = kept ? at : sums + room * OUT + 4 * lane;
      if (SPARE || kept) *reinterpret_cast<gf_f32x4_t*>(at) = acc;
    }
  };
  float tot[PER];
#pragma unroll
  for (int p = 0; p < PER; ++p) tot[p] = 0.f;
  for (int c0 = 0; c0 < chunks; c0 += room) {     // (one pass where LDS holds all chunks' sums)
    // the wavefront's turns (of CH chunks): wave, + GF_WAVES, ...; as many rounds for every wavefront, D turns in flight, no load
    // behind a branch (a round beyond the last turn loads that turn again and leaves nothing)
    const int held = chunks - c0 < room ? chunks - c0 : room, turns = (held + CH - 1) / CH, n = (turns + GF_WAVES - 1) / GF_WAVES;
    auto chunk = [&](int i) __attribute__((always_inline)) { return CH * (wave + i * GF_WAVES < turns ? wave + i * GF_WAVES : turns - 1); };
    const int last = c0 + held - 1;
    Chunk b[D];
#pragma unroll
    for (int d = 0; d < D; ++d) load(b[d], c0 + chunk(d), last);
    int i = 0;
    for (; i + D < n; i += D)
#pragma unroll
      for (int d = 0; d < D; ++d) {
        multiply(b[d], chunk(i + d), CH);
        load(b[d], c0 + chunk(i + d + D), last);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (i + d < n) multiply(b[d], chunk(i + d), wave + (i + d) * GF_WAVES < turns ? held - chunk(i + d) : 0);
    __syncthreads();
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int o = threadIdx.x + p * GF_WAVES * 64;
      if (o < OUT) {
        // (sixteen sums asked for at a time, four where fewer are left: one by one, eight of K = 512 were 0.4 us)
        int c = 0;
        for (; c + 16 <= held; c += 16)
#pragma unroll
          for (int e = 0; e < 16; ++e) tot[p] += sums[(c + e) * OUT + o];
        for (; c + 4 <= held; c += 4)
#pragma unroll
          for (int e = 0; e < 4; ++e) tot[p] += sums[(c + e) * OUT + o];
        for (; c < held; ++c) tot[p] += sums[c * OUT + o];
      }
    }
    if (c0 + room < chunks) __syncthreads();
  }
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int o = threadIdx.x + p * GF_WAVES * 64;
    if (o >= OUT) continue;
    const int n = n0 + o % WR, m = o / WR;
    float t = tot[p];
    if constexpr (GLU) {
      const float up = __shfl_xor(t, WR / 2);
      if (o % WR < WR / 2 && n < rows && m < M) Y[(size_t)m * ldy + n] = from_f32<TO>(t / (1.0f + expf(-t)) * up);
    } else if (n < N && m < M) {
      if (bias) t += bias[n];
      Y[(size_t)m * ldy + n] = from_f32<TO>(t);
    }
  }
}

#define GF_LANES_WAVES 2
// (room for more chunks than lanes_take leaves, 72: the LDS keeps a compute unit to fewer wavefronts, whose lines then stay in its cache; 8 rows
// of 65536 x 128 22.7 us with 72, 19.3)
#define GF_LANES_CHUNKS 128

// A wavefront owns pairs of rows of W, 64 / span of them: the span lanes of a pair (a power of two, as many as there are chunks,
// at most 64) take chunks l, l + span, ... each, sum a chunk of both rows from zero in ascending k and leave the sums in LDS; then
// a lane an output adds them in ascending order.
template <int MB, typename TO>
__global__ __launch_bounds__(GF_LANES_WAVES * 64) void gemm_f32_lanes_kernel(const float* __restrict__ X, int ldx,
                                                                             const float* __restrict__ W,
                                                                             const float* __restrict__ bias, TO* __restrict__ Y,
                                                                             int ldy, int M, int N, int K, int span) {
  __shared__ float cs[GF_LANES_WAVES][2 * MB][GF_LANES_CHUNKS + 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int pairs = 64 / span;               // pairs of rows per wavefront
  const int grp = lane / span, sub = lane - grp * span;
  const int nw = (blockIdx.x * GF_LANES_WAVES + wave) * 2 * pairs;   // first row of W of this wavefront
  if (nw >= N) return;                       // whole wavefronts leave; no block-wide barrier follows
  const int n0 = nw + 2 * grp;
  const bool live = n0 < N, two = n0 + 1 < N;
  const float* w0 = W + (size_t)(live ? n0 : N - 1) * K;
  const float* w1 = W + (size_t)(two ? n0 + 1 : (live ? n0 : N - 1)) * K;
  const float* xr[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m) xr[m] = X + (size_t)(m < M ? m : M - 1) * ldx;
  const int chunks = (K + GS_SUM_CHUNK - 1) / GS_SUM_CHUNK;
  for (int c = sub; c < chunks; c += span) {
    const int k0 = c * GS_SUM_CHUNK;
    const int len4 = ((K - k0 < GS_SUM_CHUNK ? K - k0 : GS_SUM_CHUNK) + 3) >> 2;   // K is a multiple of 4
    float a0[MB], a1[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m) a0[m] = a1[m] = 0.f;
#pragma unroll 4
    for (int j = 0; j < len4; ++j) {
      const float4 u = *reinterpret_cast<const float4*>(w0 + k0 + 4 * j);
      const float4 v = *reinterpret_cast<const float4*>(w1 + k0 + 4 * j);
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        const float4 x = *reinterpret_cast<const float4*>(xr[m] + k0 + 4 * j);
        a0[m] = fmaf(x.x, u.x, a0[m]); a0[m] = fmaf(x.y, u.y, a0[m]); a0[m] = fmaf(x.z, u.z, a0[m]); a0[m] = fmaf(x.w, u.w, a0[m]);
        a1[m] = fmaf(x.x, v.x, a1[m]); a1[m] = fmaf(x.y, v.y, a1[m]); a1[m] = fmaf(x.z, v.z, a1[m]); a1[m] = fmaf(x.w, v.w, a1[m]);
      }
    }
    // pair grp keeps its chunk sums at columns [grp * span, grp * span + chunks) when span < 64 (then chunks <= span)
    const int col = pairs > 1 ? grp * span + c : c;
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      cs[wave][2 * m][col] = a0[m];
      cs[wave][2 * m + 1][col] = a1[m];
    }
  }
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_s_waitcnt(0xc07f);        // this wavefront's LDS writes are visible to its own lanes
  // one lane per output (pair g, row m of x, row r of the pair) adds that output's chunk sums in ascending order
  for (int o = lane; o < pairs * 2 * MB; o += 64) {
    const int g = o / (2 * MB), q = o - g * 2 * MB, m = q >> 1, r = q & 1;
    const int n = nw + 2 * g + r;
    float t = 0.f;
    for (int c = 0; c < chunks; ++c) t += cs[wave][q][pairs > 1 ? g * span + c : c];
    if (m < M && n < N) {
      if (bias) t += bias[n];
      Y[(size_t)m * ldy + n] = from_f32<TO>(t);
    }
  }
}

// SHORT: a K of one chunk, whose rows are all asked for at once (333 rows of 2048 x 48 6.3 us as of a longer K, 5.2 here).
template <int WN, int MT, int NT, bool TAIL, bool SHORT, typename TO>
__global__ __launch_bounds__(WN * 128, WN == 2 ? 2 : 1) void gemm_f32_tiles_kernel(const float* __restrict__ X, int ldx,
                                                                                   const float* __restrict__ W,
                                                                                   const float* __restrict__ bias, TO* __restrict__ Y,
                                                                                   int ldy, int M, int N, int K) {
  constexpr int KS = 32, LD = KS + 4, BM = 32 * MT, BN = 16 * NT * WN, RPL = WN * 16;       // RPL: rows the block loads at a time
  constexpr int LX = (BM + RPL - 1) / RPL, LW = (BN + RPL - 1) / RPL;
  constexpr int G = MT * NT >= 4 ? 1 : MT * NT == 1 ? 4 : 2, NG = KS / 4 / G;               // fours of k read from LDS at a time
  __shared__ __align__(16) float xs[2][BM * LD], ws[2][BN * LD];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r16 = lane & 15, g = lane >> 4;
  // (row tiles fastest, all in x: it takes as many tiles as there can be, y only 65,535; the blocks of an XCD, every eighth, are
  // neighbours, which share rows of W and X in its L2.  Not from 8,192 blocks on: an XCD meets all row tiles then over and over, and
  // some 2,000 rows of X no longer stay in its L2; as they come it meets an eighth of them (64 x 64, 2,048 rows of 16384 x 512 317 us
  // in neighbours, 278 as they come; x 1024 580 and 532))
  const int tiles_m = (M + BM - 1) / BM;
  const unsigned per = gridDim.x >> 3, rest = gridDim.x & 7, xcd = blockIdx.x & 7;
  const unsigned tile = gridDim.x >= 8192 ? blockIdx.x : xcd * per + (xcd < rest ? xcd : rest) + (blockIdx.x >> 3);
  const int mb = (int)(tile % tiles_m) * BM, nb = (int)(tile / tiles_m) * BN, mw = (wave & 1) * 16 * MT, nw = (wave >> 1) * 16 * NT;
  // thread t loads the four k at 4 (t % 8) of row t / 8, RPL rows a load
  const int lr = threadIdx.x >> 3, lk = 4 * (threadIdx.x & 7);
  const float* xp[LX];
  const float* wp[LW];
#pragma unroll
  for (int i = 0; i < LX; ++i) xp[i] = X + (size_t)(mb + RPL * i + lr < M ? mb + RPL * i + lr : M - 1) * ldx;
#pragma unroll
  for (int j = 0; j < LW; ++j) wp[j] = W + (size_t)(nb + RPL * j + lr < N ? nb + RPL * j + lr : N - 1) * K;
  struct Rows {
    gf_f32x4_t x[LX], w[LW];
  };
  constexpr int D = !SHORT && MT * NT == 1 ? 4 : 2;        // steps under way (blocks this small stand alone: 32 rows of 6144 x 2048 24.5, 22.0)
  Rows rows[D];
  auto load = [&](Rows& v, int k) __attribute__((always_inline)) {
    const int from = (TAIL ? k + lk : k) < K ? k + lk : (TAIL ? 0 : lk);      // (what lies beyond K is not used)
#pragma unroll
    for (int i = 0; i < LX; ++i) v.x[i] = gf_load<false>(xp[i], from, K);
#pragma unroll
    for (int j = 0; j < LW; ++j) v.w[j] = gf_load<false>(wp[j], from, K);
  };
  // the rows at k into buffer s: zeros beyond K (told only here, where the values have to be there)
  auto put = [&](const Rows& v, int s, int k) __attribute__((always_inline)) {
    const bool in = !TAIL || k + lk < K;
    const gf_f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < LX; ++i)
      if (BM % RPL == 0 || RPL * i + lr < BM) *reinterpret_cast<gf_f32x4_t*>(&xs[s][(RPL * i + lr) * LD + lk]) = in ? v.x[i] : zero;
#pragma unroll
    for (int j = 0; j < LW; ++j)
      if (BN % RPL == 0 || RPL * j + lr < BN) *reinterpret_cast<gf_f32x4_t*>(&ws[s][(RPL * j + lr) * LD + lk]) = in ? v.w[j] : zero;
  };
  gf_f32x4_t acc[MT][NT], tot[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = tot[i][j] = gf_f32x4_t{0.f, 0.f, 0.f, 0.f};
  struct Operands {
    float x[G][MT], w[G][NT];
  };
  Operands held[2];
  auto read = [&](Operands& o, int s, int q) __attribute__((always_inline)) {
    const float* x = &xs[s][(mw + r16) * LD + g + 4 * G * q];
    const float* w = &ws[s][(nw + r16) * LD + g + 4 * G * q];
#pragma unroll
    for (int u = 0; u < G; ++u) {
#pragma unroll
      for (int i = 0; i < MT; ++i) o.x[u][i] = x[16 * i * LD + 4 * u];
#pragma unroll
      for (int j = 0; j < NT; ++j) o.w[u][j] = w[16 * j * LD + 4 * u];
    }
  };
  // (first: of a chunk; what the last chunk left is added before its sum begins)
  auto multiply = [&](const Operands& o, bool first) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < G; ++u)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          gf_f32x4_t c = acc[i][j];
          if (first && u == 0) {
#pragma unroll
            for (int e = 0; e < 4; ++e) tot[i][j][e] += c[e];
            c = gf_f32x4_t{0.f, 0.f, 0.f, 0.f};
          }
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.w[u][j], o.x[u][i], c, 0, 0, 0);
        }
  };
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (!SHORT || d * KS < K) load(rows[d], d * KS);
  put(rows[0], 0, 0);
  __syncthreads();
  read(held[0], 0, 0);
  // the step at k from buffer s.  Nothing of buffer s is read behind the step's barrier, where the next step's rows may replace it
  auto step = [&](int s, int k, Rows& later, const Rows& next, bool first) __attribute__((always_inline)) {
    if (!SHORT) load(later, k + D * KS);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < NG - 1; ++q) {
      read(held[(q + 1) & 1], s, q + 1);
      if (q == (NG - 1) / 2) put(next, s ^ 1, k + KS);
      __builtin_amdgcn_sched_barrier(0);
      multiply(held[q & 1], first && q == 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    read(held[0], s ^ 1, 0);
    __builtin_amdgcn_sched_barrier(0);
    multiply(held[(NG - 1) & 1], false);
    __builtin_amdgcn_sched_barrier(0);
  };
  for (int k = 0; k < K;) {
#pragma unroll
    for (int d = 0; d < D && k < K; d += 2, k += GS_SUM_CHUNK) {      // a chunk: two steps of 32 k (beyond K: zeros)
      step(0, k, rows[d], rows[d + 1], true);
      step(1, k + KS, rows[d + 1], rows[(d + 2) % D], false);
    }
  }
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) tot[i][j][e] += acc[i][j][e];
  // element e of lane l: row 4 (l / 16) + e of W, row l % 16 of X
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = mb + mw + 16 * i + r16;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int n = nb + nw + 16 * j + 4 * g + e;
        if (n >= N) continue;
        float t = tot[i][j][e];
        if (bias) t += bias[n];
        Y[(size_t)m * ldy + n] = from_f32<TO>(t);
      }
  }
}

// Whether the matrix-core kernels take the operands: K and the row stride in whole pieces of 16 bytes, both aligned.  What
// needs more blocks than a launch holds (2^32 threads) stays with the FMA kernel, and so does what that refuses for its rows.
extern "C" int gs_gemm_f32_supports(int M, int N, int K, int ldx, const void* X, const void* W) {
  const long blocks = M <= 16 ? gs_ceil_div(N, 16) : (long)gs_ceil_div(M, 64) * gs_ceil_div(N, 64);
  return M >= 1 && N > 0 && K > 0 && K % 4 == 0 && (M == 1 || ldx % 4 == 0) && ((uintptr_t)X & 15) == 0 && ((uintptr_t)W & 15) == 0 &&
         blocks < 1L << 23 && gs_ceil_div(M, 64) <= 65535;
}

// Whether the FMA kernel is the faster one all the same: many outputs of a short K, of which it takes 16 at a time and the tiles 64
// (that kernel and this one: 65 rows of 20000 x 16 6.2 us and 12.2, 1,000 of 4096 x 16 11.2 and 15.5, 40 of 20000 x 16 5.6 and 7.0;
// 300 of 65536 x 36 51 and 58, of 8192 x 36 12.7 both, of 65536 x 64 89 and 84).
static bool fma_faster(int M, int N, int K) {
  if (M <= 16) return false;
  if (K <= 16) return (long)M * N >= 700000;
  if (M <= 64) return K <= 32 && (long)M * N >= 1100000;
  return K <= 48 && N >= 12000;
}

// Whether the product is for these kernels: they can take it, and the FMA kernel is not the faster one.
extern "C" int gs_gemm_f32_takes(int M, int N, int K, int ldx, const void* X, const void* W) {
  return gs_gemm_f32_supports(M, N, K, ldx, X, W) && !fma_faster(M, N, K);
}

template <int WR, int XR, int D, int CH, typename TO, bool GLU>
static void launch_rows(const float* X, int ldx, const float* W, const float* bias, TO* Y, int ldy, int M, int N, int K,
                     hipStream_t stream) {
  // LDS for the chunk sums, beside 34 KB: 32 KB, which leaves a compute unit room for two blocks, or 64 KB where there is no more than
  // one a unit.  A pass that ends before K does drains every load in flight and adds up before it asks for the next
  // (28 KB for all: 6 rows of 16384 x 2048, 28 of 32 chunks, 33.3 against 27.5 us; of 2048 x 8192 21.4 against 20.5; 40 rows of it
  // 70 against 57, of 2048 x 2048 18.4 against 14.6).
  constexpr int out = XR * WR;
  const int blocks = GLU ? gs_ceil_div(N / 2, WR / 2) : gs_ceil_div(N, WR), chunks = gs_ceil_div(K, GS_SUM_CHUNK), most = (blocks <= 256 ? 16384 : 8192) / out;
  const int room = chunks < most ? chunks : most;
  size_t lds = (size_t)room * out * sizeof(float);
  auto kernel = K % GS_SUM_CHUNK == 0 ? &gemm_f32_rows_kernel<WR, XR, D, CH, false, TO, GLU> : &gemm_f32_rows_kernel<WR, XR, D, CH, true, TO, GLU>;
  if (lds + sizeof(float) * GF_WAVES * 16 * (GS_SUM_CHUNK + 4) > 64 * 1024) {
    // more than the default limit of LDS: asked for once per kernel
    static const hipError_t asked[2] = {
        hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_f32_rows_kernel<WR, XR, D, CH, false, TO, GLU>), hipFuncAttributeMaxDynamicSharedMemorySize, 65536),
        hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_f32_rows_kernel<WR, XR, D, CH, true, TO, GLU>), hipFuncAttributeMaxDynamicSharedMemorySize, 65536)};
    (void)asked;
  }
  if constexpr (WR == 16 && XR == 8) {
    // (what nobody keeps goes to a spare place: behind a branch for it the compiler asks for the operands of one instruction after the
    // other, which up to sixteen chunks, one cut short, do not hide: 8 rows of 65536 x 132 29.0 us, with the branch 31.4, of 40000 x 964 34.1
    // and 34.5, x 1028 54.9 and 49.0; 5 rows of gate and
    // up, 20352 x 676 18.1 and 19.6, 40000 x 516 27.4 and 30.5)
    if (K % GS_SUM_CHUNK != 0 && chunks <= 16) {
      kernel = &gemm_f32_rows_kernel<WR, XR, D, CH, true, TO, GLU, true>;
      lds += 64 * sizeof(gf_f32x4_t);
    }
  }
  kernel<<<blocks, GF_WAVES * 64, lds, stream>>>(X, ldx, W, bias, Y, ldy, M, N, K, room);
}

// Whether a wavefront takes two chunks a turn (blocks of eight weight rows, up to eight of X; the same bits).  Up to a K of 512 a chunk for
// each of the eight wavefronts is one round either way, and two cost registers and, beside them, blocks a compute unit; more than two
// rows of more than 2,048 weight rows stay so up to 1,024.  (Microseconds one and two at a time: 1 row of 1024 x 512 3.2 and 3.5, of
// 8192 x 512 6.2 and 7.6, x 576 8.9 and 8.1; 4 rows of 3072 x 1024 5.7 and 5.9, x 1088 7.5 and 6.8; 8 rows of 2048 x 768 4.5 and 4.4, of
// 6144 x 1024 8.0 and 8.8, x 1088 11.2 and 10.3; 6 rows of 8192 x 512 6.5 and 8.6.)
// Of a K whose last chunk is cut short (84 and 106 registers for 67 and 94) one at a time also up to 1,024, but for two rows of up to 2,048,
// and just above 2,048, but for two rows of up to 5,120: 1 row of 6144 x 900 8.1 and 9.8, x 1028 11.0 and 10.7, x 2308 16.9 and 19.0, of
// 512 x 2052 7.1 and 6.3; 8 rows of 2048 x 2308 8.7 and 9.2.  And three rows and more of 23 and 24 chunks, of 21 on for seven and eight, which one at a
// time are three full rounds of the wavefronts: 8 rows of 2048 x 1532 6.3 and 6.85, x 1412 6.4 and 6.6, x 1540 7.1 and 6.75; 3 rows 5.8 and 6.0; likewise five rows and more
// of 39 and 40 whole ones: 8 rows of 2048 x 2560 7.3 and 7.65, 5 rows 7.2 and 7.4, 8 of 4096 x 2560 12.0 and 12.6.
static bool two_chunks(int M, int N, int K) {
  if (K % GS_SUM_CHUNK != 0 && M > 2 && K > (M > 6 ? 1280 : 1408) && K < 1536) return false;
  if (M > 4 && K > 2432 && K <= 2560) return false;
  if (K % GS_SUM_CHUNK != 0 && ((K <= 1024 && (M > 2 || N > 2048)) || (K > 2048 && K <= 2560 && (M > 2 || N > 5120)))) return false;
  return K > (M > 2 && N > 2048 ? 1024 : 512);
}

template <int WR, int XR, int D, typename TO, bool GLU = false>
static void run_rows(const float* X, int ldx, const float* W, const float* bias, TO* Y, int ldy, int M, int N, int K, hipStream_t stream) {
  if constexpr (WR == 8 && XR <= 8) {
    if (two_chunks(M, N, K)) return launch_rows<WR, XR, D, 2, TO, GLU>(X, ldx, W, bias, Y, ldy, M, N, K, stream);
  }
  launch_rows<WR, XR, D, 1, TO, GLU>(X, ldx, W, bias, Y, ldy, M, N, K, stream);
}

template <int MB, typename TO>
static void run_lanes(const float* X, int ldx, const float* W, const float* bias, TO* Y, int ldy, int M, int N, int K,
                      hipStream_t stream) {
  int span = 1;
  while (span * GS_SUM_CHUNK < K && span < 64) span *= 2;
  const int blocks = gs_ceil_div(N, 128 / span * GF_LANES_WAVES);
  gemm_f32_lanes_kernel<MB, TO><<<blocks, GF_LANES_WAVES * 64, 0, stream>>>(X, ldx, W, bias, Y, ldy, M, N, K, span);
}

template <int WN, int MT, int NT, typename TO>
static void run_tiles(const float* X, int ldx, const float* W, const float* bias, TO* Y, int ldy, int M, int N, int K,
                      hipStream_t stream) {
  const unsigned grid = (unsigned)gs_ceil_div(M, 32 * MT) * (unsigned)gs_ceil_div(N, 16 * NT * WN);
  auto kernel = K % GS_SUM_CHUNK == 0 ? &gemm_f32_tiles_kernel<WN, MT, NT, false, false, TO> : &gemm_f32_tiles_kernel<WN, MT, NT, true, false, TO>;
  if constexpr (WN == 2)                                     // (a short K never comes to the two largest tiles)
    if (K <= GS_SUM_CHUNK) kernel = &gemm_f32_tiles_kernel<WN, MT, NT, true, true, TO>;
  kernel<<<grid, WN * 128, 0, stream>>>(X, ldx, W, bias, Y, ldy, M, N, K);
}

// Which tiles: those whose rounds of blocks take the least.  A round (a block for each of the 256 compute units) of so many rows of
// X by so many of W takes `each` tenths of a microsecond for 2,048 k, whether blocks run beside or after one another, the first
// `first` more.  (Measured on cold weights; microseconds by this and by the rule and kernel before: 680 rows of 2048 x 2048 66 and
// 74, 6144 x 2048 172 and 197, 16384 x 2048 363 and 399, 2048 x 8192 230 and 280; 100 rows of 2048 x 2048 20 and 41, x 8192 80 and
// 178; 1,024 rows of 16384 x 2048 529 and 563, 2,048 rows of 2048 x 8192 517 and 564.)
// Up to a K of 1,024 blocks are over too soon for the eight wavefronts of the two largest tiles (2,048 rows of 16384 x 192 by
// 64 x 128 156 us, by 64 x 64 138, before 140; 1,024 of 8192 x 512 82, 76, 81; 1,024 of 16384 x 1024 281, 272, 288); the others'
// order does not change with K: over 17 to 2,048 rows of 256 to 16,384 weight rows the choice is 0.8 % above the best of the five on
// average at a K of 192, 0.3 % at 512 and 1,024, 0.9 % at 2,048, 0.7 % at 8,192 (with `each` in proportion to K, and the fixed part
// not, 9 % at 192 and 256, 3 % at 512).
struct Tiles {
  int rows, cols, first, each;
};
static const Tiles f32_tiles[] = {{64, 128, 80, 650}, {96, 64, 80, 535}, {64, 64, 105, 345}, {32, 64, 70, 195}, {32, 32, 85, 112}};

static int tiles_choice(int M, int N, int K) {
  // (a chunk or two are over before rounds are: the largest of the smaller tiles that make two blocks a compute unit; 2,100 rows of
  // 8192 x 64 by 64 x 128 59.8 us, by 64 x 64 49)
  if (K <= 2 * GS_SUM_CHUNK)
    return (long)gs_ceil_div(M, 64) * gs_ceil_div(N, 64) >= 512 ? 2 : (long)gs_ceil_div(M, 32) * gs_ceil_div(N, 64) >= 512 ? 3 : 4;
  const int from = K <= 1024 ? 2 : 0;
  int best = from;
  long least = 0;
  for (int i = from; i < 5; ++i) {
    const long blocks = (long)gs_ceil_div(M, f32_tiles[i].rows) * gs_ceil_div(N, f32_tiles[i].cols);
    const long takes = f32_tiles[i].first + (blocks + 255) / 256 * f32_tiles[i].each;
    if (i == from || takes < least) {
      least = takes;
      best = i;
    }
  }
  return best;
}

// Which kernel, by sizes (microseconds on cold weights, one MI355X; the FMA kernels that ran before: 63 on average for the
// products of a decode step of 6 rows, 729 for those of a prompt portion of 900 tokens, 2048 x 2048 to 16384 x 2048).
// Up to 16 rows, a lane a chunk: see lanes_take.
// Up to 16 rows: blocks of 8 rows of W up to N = 8192, which then still are no more than four a compute unit (6 rows,
//   2048 x 8192: 21.8, blocks of 16 rows 30.7; 6144 x 2048: 15.1 and 17.2); of 16 rows beyond (two chunks a turn in blocks of 8, and blocks of
//   16: 6 rows of 9216 x 1024 12.6 and 10.4, x 2048 17.5 and 17.6, x 4608 36.0 and 36.2; of 16384 x 2048 27.2 and 23.9; 1 row of 10240 x 4608
//   32.7 and 33.9, of 16384 x 4608 50.3 and 47.6).
// Up to 64 rows: every block of the rows kernel reads all rows of X for its few of W, so wide weights go to the tiles (rows kernel and
//   tiles; 20 rows: 4096 x 2048 13.2 and 23.6, 6144 x 512 9.3 and 7.5; 64 rows: 3072 x 1024 12.8 and 11.5, 8192 x 2048 52 and 32;
//   33 rows: 4096 x 512 7.1 and 7.6, x 2048 22.7 and 23.9, 3072 x 2048 21.9 and 23.9, x 8192 75 and 82, but 4096 x 192 6.6 and 5.0,
//   3072 x 256 6.6 and 5.5), narrow ones do not fill the chip there (64 rows of 2048 x 2048 18.4 and 19.2, of 2048 x 8192 63 and 81).
//   Nor do wavefronts that share out one chunk fill a block of the rows kernel (64 rows of 8192 x 36 21.3, tiles 4.0; of 100 x 16 6.6
//   and 3.0).
// More: tiles.
//
// Whether a lane a chunk.  Long K: one and two rows of a weight of few, whose blocks of the rows kernel leave the chip idle either way (lanes
// and rows; 1 row of 32 x 2560 4.4 and 5.5, x 4096 5.7 and 6.4, x 4608 8.0 and 7.4; of 64 x 2560 5.3 and 5.5, x 2816 5.8 and 5.55; of
// 128 x 2560 5.8 and 5.4, of 1024 x 4608 10.3 and 8.3; 2 rows of 32 x 3584 5.9 and 6.55, x 4096 6.7 and 6.5, of 64 x 2304 5.45 and 5.5, x
// 2560 6.0 and 5.6, of 1024 x 8192 16.8 and 11.8; 3 rows of 16 x 2304 6.1 and 5.4; 1 row of 32 x 2048 5.0 and 4.05;
// 1 row of 200 x 2052 6.0 and 6.1, x 2304 5.5 and 5.3, of 64 x 4100 8.1 and 8.4, of 16 x 4100 5.7 and 8.2;
// just above 2,048 one row takes as long by either, and by lanes less where the weight lies in a cache: of 96 x 2112 5.05 and 5.25, in a cache 4.2
// and 5.5, of 512 x 2304 5.55 and 5.45, in a cache 5.2 and 5.7, of 768 x 2304 5.85 and 5.6; of 8 x 8192 9.3 and 9.85, of 20 x 8192 9.45 and 10.15, of 32 x 8192 11.8 and 10.15).
// Short K (weights in the last-level cache): what a lane does one after the other is K, at most a chunk of it, times the rows; what
// the rows kernel does is so many blocks.  1 row of 65536 x 4 2.4 us, rows kernel 19.8, 16 rows of 65536 x 128 25.3 and 27.9, x 192
// 55 and 30; 16 rows of 24000 x 32 10.6 and 11.4, 8 of 24000 x 64 8.2 and 8.3; 4 rows of 8192 x 48 5.3 and 5.8, x 64 6.1 and 5.5;
// 2 rows of 4096 x 32 3.75 and 3.91; 1 row of 2048 x 16 2.7 and 2.95, of 2048 x 32 3.3 and 3.0; of 20 x 48 2.5 and 2.7.
static bool lanes_take(int M, int N, int K) {
  if (M > 16) return false;
  if (K > GS_SUM_CHUNK * GF_LANES_CHUNKS) return false;
  if (M <= 2 && K > 2048) {
    const bool cut = K % GS_SUM_CHUNK != 0;                        // (a chunk cut short costs the rows kernel 0.9)
    if (M == 1 && (N <= 20 || (N <= 512 && K <= 2304))) return true;
    if (N <= 32) return K < 4608;
    return M == 1 ? (N <= 64 && K <= 2560) || (cut && N <= 256 && K < 4608) : N <= 64 && (K <= 2304 || (cut && K < 3072));
  }
  const int rows = M <= 2 ? M : M <= 4 ? 4 : M <= 8 ? 8 : 16, chain = (K < GS_SUM_CHUNK ? K : GS_SUM_CHUNK) * rows;
  if (K > 2 * GS_SUM_CHUNK) {
    // (rows of whole 256 bytes begin in the same channels)
    const bool even = K % GS_SUM_CHUNK == 0;
    return N > 4096 && K <= (rows == 1 ? (even ? 384 : 448) : rows == 2 ? (even ? 192 : 224) : rows == 4 && N > 12288 && !even ? 160 : 0);
  }
  const bool part = K > GS_SUM_CHUNK && K < 2 * GS_SUM_CHUNK;      // (two lanes a pair, rows that begin in different channels)
  if (N >= 40000) return true;
  if (N >= 20000) return chain <= (N >= 28000 ? 768 : 512);
  if (N >= 14000) return chain <= 320;
  if (N > 4096) return chain <= ((N > 8192 && K <= 32) || part ? 256 : 192);
  if (N > 2048) return (K <= 48 || part) && rows <= 4 && chain <= 64;
  return rows <= 2 && chain <= (N <= 128 ? 48 : 20);
}

// Tiles 0 to 4 (f32_tiles); rows kernel: weight rows a block times 100 plus rows; a lane a chunk: 10000 plus rows.
static int f32_choice(int M, int N, int K) {
  const int up = M <= 1 ? 1 : M <= 2 ? 2 : M <= 4 ? 4 : M <= 8 ? 8 : M <= 16 ? 16 : M <= 32 ? 32 : M <= 48 ? 48 : 64;
  if (lanes_take(M, N, K)) return 10000 + up;
  if (M <= 16) return (N <= 8192 ? 800 : 1600) + (up < 4 ? 4 : up);
  if (M <= 64 && K > GS_SUM_CHUNK && N <= (M <= 32 || (M <= 48 && K > 256) ? 4096 : 2048)) return (N <= 2048 ? 800 : 1600) + up;
  return tiles_choice(M, N, K);
}

// The choice for these sizes, for tests of every branch.
extern "C" int gs_gemm_f32_choice(int M, int N, int K) { return f32_choice(M, N, K); }

template <typename TO>
static void run(const float* X, int ldx, const float* W, const float* bias, TO* Y, int ldy, int M, int N, int K,
                hipStream_t stream) {
#define GF_TILES(I, WN, MT, NT) case I: return run_tiles<WN, MT, NT, TO>(X, ldx, W, bias, Y, ldy, M, N, K, stream)
#define GF_ROWS(WR, XR) case 100 * WR + XR: return run_rows<WR, XR, 2, TO>(X, ldx, W, bias, Y, ldy, M, N, K, stream)
#define GF_LANES(MB) case 10000 + MB: return run_lanes<MB, TO>(X, ldx, W, bias, Y, ldy, M, N, K, stream)
  switch (f32_choice(M, N, K)) {
    GF_TILES(0, 4, 2, 2); GF_TILES(1, 4, 3, 1); GF_TILES(2, 2, 2, 2); GF_TILES(3, 2, 1, 2); GF_TILES(4, 2, 1, 1);
    GF_ROWS(8, 4); GF_ROWS(8, 8); GF_ROWS(8, 16); GF_ROWS(8, 32); GF_ROWS(8, 48); GF_ROWS(8, 64);
    GF_ROWS(16, 4); GF_ROWS(16, 8); GF_ROWS(16, 16); GF_ROWS(16, 32); GF_ROWS(16, 48);
    GF_LANES(1); GF_LANES(2); GF_LANES(4); GF_LANES(8); GF_LANES(16);
  }
#undef GF_LANES
#undef GF_ROWS
#undef GF_TILES
}

extern "C" int gs_gemm_f32(const float* X, int ldx, const float* W, const float* bias, void* Y, int y_dtype, int ldy,
                           int M, int N, int K, hipStream_t stream) {
  GS_REQUIRE(N > 0 && K > 0 && ldy >= N && (M <= 1 || ldx >= K), "gemm_f32: bad sizes N=%d K=%d ldx=%d ldy=%d", N, K, ldx, ldy);
  GS_REQUIRE(gs_gemm_f32_supports(M, N, K, ldx, X, W), "gemm_f32: needs rows, K and strides a multiple of 4, aligned operands, no more than a launch holds (M=%d N=%d K=%d)", M, N, K);
  GS_REQUIRE(y_dtype == GS_F32 || y_dtype == GS_BF16, "gemm_f32: unknown output dtype %d", y_dtype);
  if (y_dtype == GS_F32)
    run<float>(X, ldx, W, bias, (float*)Y, ldy, M, N, K, stream);
  else
    run<bf16>(X, ldx, W, bias, (bf16*)Y, ldy, M, N, K, stream);
  GS_LAUNCH_CHECK("gemm_f32");
  return 0;
}

// Whether gate and up rows, side by side in W (N of them, half each), go through gs_gemm_f32_swiglu: what the rows kernel takes of
// such a product.  The tiles' outputs of a gate and its up lie in blocks far apart, and of so many rows the pass between is little
// (728 rows: 12 us beside 450).
extern "C" int gs_gemm_f32_swiglu_takes(int M, int N, int K, int ldx, const void* X, const void* W) {
  if (N % 2 || !gs_gemm_f32_takes(M, N, K, ldx, X, W)) return 0;
  const int choice = f32_choice(M, N, K);
  return choice >= 800 && choice < 10000;
}

// Y = silu(X Wg^T) * (X Wu^T), N / 2 wide: the sums of gs_gemm_f32 and the activation of gs_swiglu, bit for bit.
extern "C" int gs_gemm_f32_swiglu(const float* X, int ldx, const float* W, float* Y, int ldy, int M, int N, int K, hipStream_t stream) {
  GS_REQUIRE(N > 0 && K > 0 && ldy >= N / 2 && (M <= 1 || ldx >= K), "gemm_f32_swiglu: bad sizes N=%d K=%d ldx=%d ldy=%d", N, K, ldx, ldy);
  GS_REQUIRE(gs_gemm_f32_swiglu_takes(M, N, K, ldx, X, W), "gemm_f32_swiglu: not a product of these sizes and operands (M=%d N=%d K=%d)", M, N, K);
#define GF_GLU(WR, XR) case 100 * WR + XR: run_rows<WR, XR, 2, float, true>(X, ldx, W, nullptr, Y, ldy, M, N, K, stream); break
  switch (f32_choice(M, N, K)) {
    GF_GLU(8, 4); GF_GLU(8, 8); GF_GLU(8, 16); GF_GLU(8, 32); GF_GLU(8, 48); GF_GLU(8, 64);
    GF_GLU(16, 4); GF_GLU(16, 8); GF_GLU(16, 16); GF_GLU(16, 32); GF_GLU(16, 48);
  }
#undef GF_GLU
  GS_LAUNCH_CHECK("gemm_f32_swiglu");
  return 0;
}
