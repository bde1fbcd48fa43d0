// Attention through a cached latent row: the kernels around the products, and the general attention kernel.
//
// A token's cache row is [z | k_rot]: z = the normed key/value latent (c numbers), k_rot = the rotated key features
// that all heads share (r numbers).  Head h's key is (W_uk[h] z | k_rot) and its value W_uv[h] z, so with
// q~ = (W_uk[h]^T q_plain | q_rot) the score is q~ . [z | k_rot] and the head's output W_uv[h] (sum_j p_j z_j):
// every head attends over the same rows (one key head of width c + r whose first c columns are also its values),
// and neither keys nor values of single heads are ever formed.
//
//   latent_prep       per token: RMS norm of the query latent -> rows for the query product; RMS norm of the
//                     key/value latent, rotation of the shared key features, both into the token's cache row
//   latent_q_rot      rotates the rotated part of every head's query into its place behind the absorbed part
//   heads_product     Y[t, h, :] = W[h] X[t, h, :] for all heads in one launch, with an optional gate: times
//                     sigmoid(G[t, h]), or times sigmoid(G[t, h N + n]) for output n (a gate each); float32 FMAs in a
//                     fixed summation order, or the matrix cores for bfloat16
//   attention_latent  the general attention kernel over such rows: any sizes, float32 arithmetic
//
// All norms, angles, scores, softmax weights and the gate's sigmoid are float32.
#include "common.h"

#define LP_HELD 4        // values of a latent a thread holds

template <typename T>
__global__ void latent_prep_kernel(const T* __restrict__ down, int ld, int q_off, int q_rank, int kv_off, int c, int r,
                                   const float* __restrict__ qw, const float* __restrict__ kvw, float eps,
                                   const float* __restrict__ cos_t, const float* __restrict__ sin_t,
                                   const int* __restrict__ positions, const int* __restrict__ seq_of_token,
                                   const int* __restrict__ block_table, int max_blocks, int page_size,
                                   T* __restrict__ cache, T* __restrict__ a_out, int write_kv) {
  __shared__ float red[17];
  const int t = blockIdx.x, tid = threadIdx.x, nt = blockDim.x;
  const T* row = down + (size_t)t * ld;
  if (write_kv && q_rank <= LP_HELD * nt && c <= LP_HELD * nt && r <= 2 * nt) {
    // everything a thread needs is asked for at once, the two sums are taken together (8 rows, ranks of 768 and 512: 4.5 us;
    // one norm after the other, each value asked for twice: 6.9)
    float q[LP_HELD], qv[LP_HELD], k[LP_HELD], kv[LP_HELD];
    const int pos = positions[t], seq = seq_of_token[t];
#pragma unroll
    for (int i = 0; i < LP_HELD; ++i) {
      const int jq = tid + i * nt < q_rank ? tid + i * nt : 0, jc = tid + i * nt < c ? tid + i * nt : 0;
      q[i] = to_f32(row[q_off + jq]);
      qv[i] = qw[jq];
      k[i] = to_f32(row[kv_off + jc]);
      kv[i] = kvw[jc];
    }
    const int half = r / 2, jr = tid < half ? tid : 0;
    float u = 0.f, v = 0.f, cs = 0.f, sn = 0.f;
    if (half) {
      u = to_f32(row[kv_off + c + jr]);
      v = to_f32(row[kv_off + c + jr + half]);
      cs = cos_t[(size_t)pos * half + jr];
      sn = sin_t[(size_t)pos * half + jr];
    }
    const int page = block_table[(size_t)seq * max_blocks + pos / page_size];
    float sq = 0.f, sk = 0.f;
#pragma unroll
    for (int i = 0; i < LP_HELD; ++i) {
      if (tid + i * nt < q_rank) sq += q[i] * q[i];
      if (tid + i * nt < c) sk += k[i] * k[i];
    }
    sq = wave_sum(sq);
    sk = wave_sum(sk);
    const int wave = tid >> 6, nw = nt >> 6;
    if ((tid & 63) == 0) {
      red[wave] = sq;
      red[8 + wave] = sk;
    }
    __syncthreads();
    sq = sk = 0.f;
    for (int i = 0; i < nw; ++i) {
      sq += red[i];
      sk += red[8 + i];
    }
    const float iq = norm_inverse(sq, (float)q_rank, eps), ik = norm_inverse(sk, (float)c, eps);
    T* dst = cache + ((size_t)page * page_size + pos % page_size) * (size_t)(c + r);
#pragma unroll
    for (int i = 0; i < LP_HELD; ++i) {
      const int j = tid + i * nt;
      if (j < q_rank) a_out[(size_t)t * q_rank + j] = from_f32<T>(q[i] * iq * qv[i]);
      if (j < c) dst[j] = from_f32<T>(k[i] * ik * kv[i]);
    }
    if (tid < half) {
      dst[c + tid] = from_f32<T>(u * cs - v * sn);
      dst[c + tid + half] = from_f32<T>(v * cs + u * sn);
    }
    return;
  }
  float ss = 0.f;
  for (int j = tid; j < q_rank; j += nt) {
    const float v = to_f32(row[q_off + j]);
    ss += v * v;
  }
  ss = block_sum(ss, red);
  float inv = norm_inverse(ss, (float)q_rank, eps);
  for (int j = tid; j < q_rank; j += nt)
    a_out[(size_t)t * q_rank + j] = from_f32<T>(to_f32(row[q_off + j]) * inv * qw[j]);
  if (!write_kv) return;
  ss = 0.f;
  for (int j = tid; j < c; j += nt) {
    const float v = to_f32(row[kv_off + j]);
    ss += v * v;
  }
  ss = block_sum(ss, red);
  inv = norm_inverse(ss, (float)c, eps);
  const int pos = positions[t];
  const int page = block_table[(size_t)seq_of_token[t] * max_blocks + pos / page_size];
  T* dst = cache + ((size_t)page * page_size + pos % page_size) * (size_t)(c + r);
  for (int j = tid; j < c; j += nt) dst[j] = from_f32<T>(to_f32(row[kv_off + j]) * inv * kvw[j]);
  const int half = r / 2;
  for (int j = tid; j < half; j += nt) {
    const float u = to_f32(row[kv_off + c + j]), v = to_f32(row[kv_off + c + j + half]);
    const float cs = cos_t[(size_t)pos * half + j], sn = sin_t[(size_t)pos * half + j];
    dst[c + j] = from_f32<T>(u * cs - v * sn);
    dst[c + j + half] = from_f32<T>(v * cs + u * sn);
  }
}

extern "C" int gs_latent_prep(const void* down, int dtype, int ld, int q_off, int q_rank, int kv_off, int c, int r,
                              const float* qw, const float* kvw, float eps, const float* cos_t, const float* sin_t,
                              const int* positions, const int* seq_of_token, const int* block_table, int max_blocks,
                              int page_size, void* cache, void* a_out, int write_kv, int ntok, hipStream_t stream) {
  GS_REQUIRE(ntok >= 0 && q_rank > 0 && c > 0 && r >= 0 && r % 2 == 0, "latent_prep: bad sizes T=%d q_rank=%d c=%d r=%d",
             ntok, q_rank, c, r);
  GS_REQUIRE(q_off >= 0 && kv_off >= 0 && q_off + q_rank <= ld && (!write_kv || (kvw && kv_off + c + r <= ld)),
             "latent_prep: columns %d+%d, %d+%d+%d outside rows of %d", q_off, q_rank, kv_off, c, r, ld);
  GS_REQUIRE(page_size > 0 && max_blocks > 0, "latent_prep: bad page_size/max_blocks");
  if (ntok == 0) return 0;
  if (dtype == GS_F32)
    latent_prep_kernel<float><<<ntok, 256, 0, stream>>>((const float*)down, ld, q_off, q_rank, kv_off, c, r, qw, kvw, eps,
                                                        cos_t, sin_t, positions, seq_of_token, block_table, max_blocks,
                                                        page_size, (float*)cache, (float*)a_out, write_kv);
  else if (dtype == GS_BF16)
    latent_prep_kernel<bf16><<<ntok, 256, 0, stream>>>((const bf16*)down, ld, q_off, q_rank, kv_off, c, r, qw, kvw, eps,
                                                       cos_t, sin_t, positions, seq_of_token, block_table, max_blocks,
                                                       page_size, (bf16*)cache, (bf16*)a_out, write_kv);
  else
    GS_REQUIRE(false, "latent_prep: unknown dtype %d", dtype);
  GS_LAUNCH_CHECK("latent_prep");
  return 0;
}

// A pair of features turned.  (What is fused is written out: the compiler's choice differs between kernels, and their results with it.)
__device__ __forceinline__ void turn_pair(float u, float v, float cs, float sn, float& a, float& b) {
  a = fmaf(u, cs, -(v * sn));
  b = fmaf(u, sn, v * cs);
}

// q (T, ldq): head h at [h (n + r), ...), its last r columns rotated into qa (T, H (c + r)) at [h (c + r) + c, ...).
template <typename T>
__global__ void latent_q_rot_kernel(const T* __restrict__ q, int ldq, int H, int n, int r, int c,
                                    const float* __restrict__ cos_t, const float* __restrict__ sin_t,
                                    const int* __restrict__ positions, T* __restrict__ qa) {
  const int t = blockIdx.x, half = r / 2, pos = positions[t];
  const T* row = q + (size_t)t * ldq;
  T* dst = qa + (size_t)t * H * (c + r);
  for (int idx = threadIdx.x; idx < H * half; idx += blockDim.x) {
    const int h = idx / half, j = idx % half;
    const float u = to_f32(row[h * (n + r) + n + j]), v = to_f32(row[h * (n + r) + n + j + half]);
    const float cs = cos_t[(size_t)pos * half + j], sn = sin_t[(size_t)pos * half + j];
    float a, b;
    turn_pair(u, v, cs, sn, a, b);
    dst[h * (c + r) + c + j] = from_f32<T>(a);
    dst[h * (c + r) + c + j + half] = from_f32<T>(b);
  }
}

extern "C" int gs_latent_q_rot(const void* q, int dtype, int ldq, int H, int n, int r, int c, const float* cos_t,
                               const float* sin_t, const int* positions, void* qa, int ntok, hipStream_t stream) {
  GS_REQUIRE(ntok >= 0 && H > 0 && n >= 0 && r >= 0 && r % 2 == 0 && c > 0, "latent_q_rot: bad sizes");
  GS_REQUIRE(ldq >= H * (n + r), "latent_q_rot: rows of %d hold no %d heads of %d", ldq, H, n + r);
  if (ntok == 0 || r == 0) return 0;
  if (dtype == GS_F32)
    latent_q_rot_kernel<float><<<ntok, 128, 0, stream>>>((const float*)q, ldq, H, n, r, c, cos_t, sin_t, positions,
                                                         (float*)qa);
  else if (dtype == GS_BF16)
    latent_q_rot_kernel<bf16><<<ntok, 128, 0, stream>>>((const bf16*)q, ldq, H, n, r, c, cos_t, sin_t, positions,
                                                        (bf16*)qa);
  else
    GS_REQUIRE(false, "latent_q_rot: unknown dtype %d", dtype);
  GS_LAUNCH_CHECK("latent_q_rot");
  return 0;
}

// ---------------------------------------------------------------------------------------------------------------
// Y[m, h, :N] = W[h] (N, K) . X[m, h, :K], all heads in one launch: head h's rows of X start hx elements after head
// h - 1's, those of Y hy elements.  The summation order of an output is that of the plain tiled product (chunks of 64
// from zero in ascending k, then the chunks' sums), so a value depends neither on M nor on its neighbours.
#define HP_TM 64
#define HP_TN 64
#define HP_TK 16

template <typename TX, typename TW>
__global__ void heads_product_kernel(const TX* __restrict__ X, int ldx, int hx, const TW* __restrict__ W,
                                     TX* __restrict__ Y, int ldy, int hy, const TX* __restrict__ G, int ldg,
                                     int gate_each, int M, int N, int K) {
  __shared__ float xs[HP_TK][HP_TM + 4];
  __shared__ float ws[HP_TK][HP_TN + 4];
  const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
  const int h = blockIdx.z, m0 = blockIdx.y * HP_TM, n0 = blockIdx.x * HP_TN;
  X += (size_t)h * hx;
  Y += (size_t)h * hy;
  W += (size_t)h * N * K;
  float acc[4][4], tot[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = tot[i][j] = 0.f;
  for (int k0 = 0; k0 < K; k0 += HP_TK) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int idx = tid + e * 256, r = idx >> 4, kk = idx & 15;
      const int m = m0 + r, n = n0 + r, k = k0 + kk;
      xs[kk][r] = (m < M && k < K) ? to_f32(X[(size_t)m * ldx + k]) : 0.f;
      ws[kk][r] = (n < N && k < K) ? to_f32(W[(size_t)n * K + k]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < HP_TK; ++kk) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = xs[kk][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = ws[kk][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
    if (((k0 / HP_TK) & (GS_SUM_CHUNK / HP_TK - 1)) == GS_SUM_CHUNK / HP_TK - 1 || k0 + HP_TK >= K) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          tot[i][j] += acc[i][j];
          acc[i][j] = 0.f;
        }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty * 4 + i;
    if (m >= M) continue;
    float gate = 1.f;
    if (G && !gate_each) gate = 1.f / (1.f + expf(-to_f32(G[(size_t)m * ldg + h])));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n >= N) continue;
      if (G && gate_each) gate = 1.f / (1.f + expf(-to_f32(G[(size_t)m * ldg + (size_t)h * N + n])));
      Y[(size_t)m * ldy + n] = from_f32<TX>(tot[i][j] * gate);
    }
  }
}

// The same product on the matrix cores (bfloat16 rows and weights, float32 sums): v_mfma_f32_16x16x32_bf16 with both
// operands loaded straight from memory in operand order (lane l: row or weight row l % 16, eight consecutive k at
// 8 (l / 16)); a head's weight is small and stays in the caches, so nothing is staged.  A wavefront owns 16 MTW rows x
// 16 NTW columns of one head; the wavefronts of a block own such pieces of their own, and no barrier is needed.
//
// `rot` features that follow a head's K in X go, turned by the row's position, behind the head's N in Y: pieces beyond those of the
// products, a wavefront for 256 pairs of the same rows (latent attention's queries; a launch of its own took 4.4 us a layer of a step).
// (A wavefront for all pairs of its rows was slower than that launch where they are many beside the products: 16 heads of 128 x 64
// with 128 turned, 256 rows, two launches 8.3 us, so 10.3, these 5.7.)
struct HeadsRot {
  int rot;
  const float* cos_t;      // (positions, rot / 2)
  const float* sin_t;
  const int* positions;    // (M)
};
constexpr int HP_TURNS = 256;
__host__ __device__ constexpr int heads_turns(int rows, int half) { return (rows * half + HP_TURNS - 1) / HP_TURNS; }
typedef __attribute__((ext_vector_type(8))) __bf16 hp_bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float hp_f32x4_t;
typedef __attribute__((ext_vector_type(4))) unsigned hp_u32x4_t;

template <int NTW, int MTW, int DEPTH>
__global__ __launch_bounds__(256) void heads_product_mfma_kernel(const bf16* __restrict__ X, int ldx, int hx,
                                                                 const bf16* __restrict__ W, bf16* __restrict__ Y,
                                                                 int ldy, int hy, const bf16* __restrict__ G, int ldg,
                                                                 int gate_each, int M, int N, int K, HeadsRot hr) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r16 = lane & 15, g = lane >> 4;
  const int h = blockIdx.y;
  const int mtiles = (M + 16 * MTW - 1) / (16 * MTW), ngroups = (N + 16 * NTW - 1) / (16 * NTW);
  const int item = blockIdx.x * (blockDim.x >> 6) + wave;
  const int m0 = (item % mtiles) * 16 * MTW, n0 = (item / mtiles) * 16 * NTW;
  if (item >= mtiles * ngroups) {
    const int half = hr.rot / 2, part = item / mtiles - ngroups;
    if (part >= heads_turns(16 * MTW, half)) return;
    const int pairs = (M - m0 < 16 * MTW ? M - m0 : 16 * MTW) * half;
    float u[HP_TURNS / 64], v[HP_TURNS / 64], cs[HP_TURNS / 64], sn[HP_TURNS / 64];
    // (all asked for at once; what lies beyond the rows is loaded from the first pair and not stored)
#pragma unroll
    for (int t = 0; t < HP_TURNS / 64; ++t) {
      const int p = part * HP_TURNS + 64 * t + lane, q = p < pairs ? p : 0, m = m0 + q / half, j = q % half;
      const bf16* x = X + (size_t)m * ldx + (size_t)h * hx + K + j;
      const size_t at = (size_t)hr.positions[m] * half + j;
      u[t] = to_f32(x[0]);
      v[t] = to_f32(x[half]);
      cs[t] = hr.cos_t[at];
      sn[t] = hr.sin_t[at];
    }
#pragma unroll
    for (int t = 0; t < HP_TURNS / 64; ++t) {
      const int p = part * HP_TURNS + 64 * t + lane;
      if (p >= pairs) return;
      bf16* y = Y + (size_t)(m0 + p / half) * ldy + (size_t)h * hy + N + p % half;
      float a, b;
      turn_pair(u[t], v[t], cs[t], sn[t], a, b);
      y[0] = f32_to_bf16(a);
      y[half] = f32_to_bf16(b);
    }
    return;
  }
  const bf16* xp[MTW];
#pragma unroll
  for (int i = 0; i < MTW; ++i) {
    const int mrow = m0 + 16 * i + r16 < M ? m0 + 16 * i + r16 : M - 1;
    xp[i] = X + (size_t)mrow * ldx + (size_t)h * hx + 8 * g;
  }
  const bf16* wp[NTW];
#pragma unroll
  for (int j = 0; j < NTW; ++j) {
    const int n = n0 + 16 * j + r16 < N ? n0 + 16 * j + r16 : N - 1;
    wp[j] = W + ((size_t)h * N + n) * K + 8 * g;
  }
  hp_f32x4_t acc[MTW][NTW];
#pragma unroll
  for (int i = 0; i < MTW; ++i)
#pragma unroll
    for (int j = 0; j < NTW; ++j) acc[i][j] = hp_f32x4_t{0.f, 0.f, 0.f, 0.f};
  // the loads of DEPTH steps of 32 k are issued before the first is multiplied (a piece beyond K is read from the row's start
  // and counts as zeros: that is put in behind the loads, where a test between them would wait for each; one at a time the
  // compiler orders four steps as it likes)
#pragma unroll (DEPTH == 1 ? 4 : 1)
  for (int k0 = 0; k0 < K; k0 += 32 * DEPTH) {
    hp_u32x4_t a[DEPTH][MTW], b[DEPTH][NTW];
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      const int k = k0 + 32 * d, kk = k + 8 * g < K ? k : -8 * g;      // K in whole pieces of 8: a piece is inside or outside
#pragma unroll
      for (int i = 0; i < MTW; ++i) a[d][i] = *reinterpret_cast<const hp_u32x4_t*>(xp[i] + kk);
#pragma unroll
      for (int j = 0; j < NTW; ++j) b[d][j] = *reinterpret_cast<const hp_u32x4_t*>(wp[j] + kk);
    }
    if (DEPTH > 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      const bool in = k0 + 32 * d + 8 * g < K;
#pragma unroll
      for (int i = 0; i < MTW; ++i)
#pragma unroll
        for (int j = 0; j < NTW; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(hp_bf16x8_t, in ? a[d][i] : hp_u32x4_t{0u, 0u, 0u, 0u}),
              __builtin_bit_cast(hp_bf16x8_t, in ? b[d][j] : hp_u32x4_t{0u, 0u, 0u, 0u}), acc[i][j], 0, 0, 0);
    }
  }
#pragma unroll
  for (int i = 0; i < MTW; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int m = m0 + 16 * i + 4 * g + e;
      if (m >= M) continue;
      float gate = 1.f;
      if (G && !gate_each) gate = 1.f / (1.f + expf(-to_f32(G[(size_t)m * ldg + h])));
#pragma unroll
      for (int j = 0; j < NTW; ++j) {
        const int n = n0 + 16 * j + r16;
        if (n >= N) continue;
        if (G && gate_each) gate = 1.f / (1.f + expf(-to_f32(G[(size_t)m * ldg + (size_t)h * N + n])));
        Y[(size_t)m * ldy + (size_t)h * hy + n] = f32_to_bf16(acc[i][j][e] * gate);
      }
    }
}

static int heads_product(const void* X, int x_dtype, int ldx, int hx, const void* W, int w_dtype, void* Y, int ldy, int hy, const void* G,
                         int ldg, int gate_each, int M, int N, int K, int H, HeadsRot hr, hipStream_t stream) {
  GS_REQUIRE(M >= 0 && N > 0 && K > 0 && H > 0, "heads_product: bad sizes M=%d N=%d K=%d H=%d", M, N, K, H);
  GS_REQUIRE(H <= 65535 && gs_ceil_div(M, HP_TM) <= 65535, "heads_product: too many heads or rows for one launch");
  GS_REQUIRE((long)(H - 1) * hx + K <= ldx && (long)(H - 1) * hy + N <= ldy,
             "heads_product: heads reach past their rows (ldx=%d hx=%d K=%d, ldy=%d hy=%d N=%d)", ldx, hx, K, ldy, hy, N);
  GS_REQUIRE(G == nullptr || ldg >= (gate_each ? H * N : H), "heads_product: gate rows of %d hold no gates for %d heads", ldg, H);
  if (M == 0) return 0;
  if (x_dtype == GS_BF16 && w_dtype == GS_BF16 && K % 8 == 0 && ldx % 8 == 0 && hx % 8 == 0 && ((uintptr_t)X & 15) == 0 &&
      ((uintptr_t)W & 15) == 0) {
    // few rows: narrow pieces, so that a head's weight is spread over more wavefronts; many: 32 x 64 a wavefront
    const int ntw = M <= 64 ? 1 : 4, mtw = M <= 64 ? 1 : 2;
    const int mtiles = gs_ceil_div(M, 16 * mtw);
    const long products = (long)mtiles * gs_ceil_div(N, 16 * ntw), items = products + (long)mtiles * heads_turns(16 * mtw, hr.rot / 2);
    GS_REQUIRE(items + 1 < (1L << 31), "heads_product: too many tiles");
    // Up to 64 rows, all of K in flight up to 512, in forms of 2, 4 and 16 steps of 32 k (8 rows, 16 heads of 512 x 128 and 128 x 512
    // in a step: 4.7 us each in the mean, four steps at a time, each waiting for its own, 7.3).  Steps beyond K load the row's start
    // and multiply zeros: hidden while a piece has a compute unit of its own (8 rows, 8 heads of 64 x 136 on cold weights 3.4 us,
    // four steps at a time 4.7), not where they queue up (64 rows, 32 heads of 512 x 192: 17.0 us and 8.5; 16 of 512 x 384, a
    // quarter of the steps, 9.7 and 8.2; 17 rows, 512 pieces, 5.0 and 4.6; 33 rows, 16 of 128 x 384, 384 pieces, 0.86 of it).  So
    // more pieces than units go four steps at a time unless what the form adds is little.
    const int steps = gs_ceil_div(K, 32), depth = steps <= 2 ? 2 : steps <= 4 ? 4 : 16, added = gs_ceil_div(steps, depth) * depth - steps;
    const long pieces = products * H;
    const bool held = pieces <= 256 || pieces * added <= 170L * steps;
    // (few pieces: a wavefront a block, so that they spread over as many compute units)
    const int waves = ntw == 1 && held && pieces < 1024 ? 1 : 4;
    dim3 grid((unsigned)gs_ceil_div(items, waves), H);
#define HP_RUN(NTW, MTW, DEPTH)                                                                                              \
  heads_product_mfma_kernel<NTW, MTW, DEPTH><<<grid, 64 * waves, 0, stream>>>((const bf16*)X, ldx, hx, (const bf16*)W, (bf16*)Y, \
                                                                              ldy, hy, (const bf16*)G, ldg, gate_each, M, N, K, hr)
    // (many rows: two steps at a time, an odd number of them one at a time: 333 rows of 16 heads of 96 x 96 5.5 us, by twos 5.8)
    if (ntw == 4) { if (steps % 2) HP_RUN(4, 2, 1); else HP_RUN(4, 2, 2); }
    else if (!held) HP_RUN(1, 1, 1);
    else if (depth == 2) HP_RUN(1, 1, 2);
    else if (depth == 4) HP_RUN(1, 1, 4);
    else HP_RUN(1, 1, 16);
#undef HP_RUN
    GS_LAUNCH_CHECK("heads_product_mfma");
    return 0;
  }
  if (hr.rot) {
    // (a product of another kind: the turned features by their own kernel)
    const int rc = gs_latent_q_rot(X, x_dtype, ldx, H, K, hr.rot, N, hr.cos_t, hr.sin_t, hr.positions, Y, M, stream);
    if (rc) return rc;
  }
  dim3 grid(gs_ceil_div(N, HP_TN), gs_ceil_div(M, HP_TM), H);
  if (x_dtype == GS_F32 && w_dtype == GS_F32)
    heads_product_kernel<float, float><<<grid, 256, 0, stream>>>((const float*)X, ldx, hx, (const float*)W, (float*)Y,
                                                                 ldy, hy, (const float*)G, ldg, gate_each, M, N, K);
  else if (x_dtype == GS_BF16 && w_dtype == GS_BF16)
    heads_product_kernel<bf16, bf16><<<grid, 256, 0, stream>>>((const bf16*)X, ldx, hx, (const bf16*)W, (bf16*)Y, ldy,
                                                               hy, (const bf16*)G, ldg, gate_each, M, N, K);
  else if (x_dtype == GS_BF16 && w_dtype == GS_F32)
    heads_product_kernel<bf16, float><<<grid, 256, 0, stream>>>((const bf16*)X, ldx, hx, (const float*)W, (bf16*)Y, ldy,
                                                                hy, (const bf16*)G, ldg, gate_each, M, N, K);
  else
    GS_REQUIRE(false, "heads_product: unsupported types %d %d", x_dtype, w_dtype);
  GS_LAUNCH_CHECK("heads_product");
  return 0;
}

extern "C" int gs_heads_product(const void* X, int x_dtype, int ldx, int hx, const void* W, int w_dtype, void* Y,
                                int ldy, int hy, const void* G, int ldg, int gate_each, int M, int N, int K, int H,
                                hipStream_t stream) {
  return heads_product(X, x_dtype, ldx, hx, W, w_dtype, Y, ldy, hy, G, ldg, gate_each, M, N, K, H, HeadsRot{}, stream);
}

// The same without gates and, in the same launch for up to 512 rows where the matrix cores take it, gs_latent_q_rot: X's rows are H heads of K + rot
// features, Y's H heads of N + rot.
extern "C" int gs_heads_product_rot(const void* X, int x_dtype, int ldx, const void* W, int w_dtype, void* Y, int M, int N, int K, int H,
                                    int rot, const float* cos_t, const float* sin_t, const int* positions, hipStream_t stream) {
  GS_REQUIRE(rot > 0 && rot % 2 == 0 && cos_t && sin_t && positions, "heads_product_rot: %d features to turn, tables and positions", rot);
  GS_REQUIRE(H > 0 && (long)H * (K + rot) <= ldx, "heads_product_rot: rows of %d hold no %d heads of %d", ldx, H, K + rot);
  // Beyond 512 rows the pieces cost as much as the launch they save, or more: 16 heads of 512 x 128 with 64 turned, one launch and two,
  // 512 rows 11.1 us and 13.5, 1,000 rows 21.7 and 20.9, 2,048 rows 35.2 and 33.2.
  const bool apart = M > 512;
  if (apart) {
    const int rc = gs_latent_q_rot(X, x_dtype, ldx, H, K, rot, N, cos_t, sin_t, positions, Y, M, stream);
    if (rc) return rc;
  }
  return heads_product(X, x_dtype, ldx, K + rot, W, w_dtype, Y, H * (N + rot), N + rot, nullptr, 0, 0, M, N, K, H,
                       apart ? HeadsRot{} : HeadsRot{rot, cos_t, sin_t, positions}, stream);
}

// ---------------------------------------------------------------------------------------------------------------
// The general attention kernel over latent rows: one wavefront per (query token, head).  The query at position p of
// its sequence sees the rows lo..p, lo = 0 or p - window + 1, read through the block table (this step's own rows were
// written before).  Rows are walked in tiles of 64 from lo with a running maximum and sum, so a position's result
// does not depend on how its sequence was cut into steps.
//
//   s_u = (q~ . row_u) * scale over all D = c + r columns;  o = sum_u softmax(s)_u row_u[:c]
//
// With `sinks` (one float32 a head) the softmax's denominator has one more term, exp(sinks[h]), which has no row.
//
// qa (T, H D); out (T, H c); cache (pages, page_size, D).
#define LAT_MAX_C 2048

template <typename T>
__global__ void attention_latent_kernel(const T* __restrict__ qa, const T* __restrict__ cache,
                                        const int* __restrict__ positions, const int* __restrict__ seq_of_token,
                                        const int* __restrict__ block_table, int max_blocks, int page_size, int window,
                                        float scale, T* __restrict__ out, int H, int c, int D,
                                        const float* __restrict__ sinks) {
  extern __shared__ float qs[];      // D floats
  __shared__ float ps[64];
  __shared__ long rowoff[64];
  const int lane = threadIdx.x, t = blockIdx.x, h = blockIdx.y;
  const int pos = positions[t];
  const int* bt = block_table + (size_t)seq_of_token[t] * max_blocks;
  for (int j = lane; j < D; j += 64) qs[j] = to_f32(qa[((size_t)t * H + h) * D + j]);
  __syncthreads();
  const int lo = window > 0 ? (pos - window + 1 > 0 ? pos - window + 1 : 0) : 0;
  float m = sinks ? sinks[h] : -INFINITY, l = sinks ? 1.f : 0.f;      // the sink's own term: its score is stored as it counts
  float acc[LAT_MAX_C / 64];
#pragma unroll
  for (int i = 0; i < LAT_MAX_C / 64; ++i) acc[i] = 0.f;
  for (int base = lo; base <= pos; base += 64) {
    const int u = base + lane;
    float s = -INFINITY;
    long off = 0;
    if (u <= pos) {
      off = ((long)bt[u / page_size] * page_size + u % page_size) * D;
      const T* kr = cache + off;
      float dot = 0.f;
      for (int j = 0; j < D; ++j) dot += qs[j] * to_f32(kr[j]);
      s = dot * scale;
    }
    const float m_new = fmaxf(m, wave_max(s));
    const float p = u <= pos ? expf(s - m_new) : 0.f;
    const float alpha = expf(m - m_new);
    l = l * alpha + wave_sum(p);
    m = m_new;
    __syncthreads();
    ps[lane] = p;
    rowoff[lane] = off;
    __syncthreads();
    const int nk = pos - base + 1 < 64 ? pos - base + 1 : 64;
#pragma unroll
    for (int i = 0; i < LAT_MAX_C / 64; ++i) {
      const int j = lane + 64 * i;
      if (j < c) {
        float a = acc[i] * alpha;
        for (int k = 0; k < nk; ++k) a += ps[k] * to_f32(cache[rowoff[k] + j]);
        acc[i] = a;
      }
    }
  }
  const float inv = 1.0f / l;
#pragma unroll
  for (int i = 0; i < LAT_MAX_C / 64; ++i) {
    const int j = lane + 64 * i;
    if (j < c) out[((size_t)t * H + h) * c + j] = from_f32<T>(acc[i] * inv);
  }
}

extern "C" int gs_attention_latent(const void* qa, const void* cache, int dtype, const int* positions,
                                   const int* seq_of_token, const int* block_table, int max_blocks, int page_size,
                                   int window, float scale, void* out, int ntok, int H, int c, int r, const float* sinks,
                                   hipStream_t stream) {
  GS_REQUIRE(ntok >= 0 && H > 0 && c > 0 && r >= 0, "attention_latent: bad sizes T=%d H=%d c=%d r=%d", ntok, H, c, r);
  GS_REQUIRE(c <= LAT_MAX_C && c + r <= 12288, "attention_latent: latent rows of %d + %d above the kernel's limit", c, r);
  GS_REQUIRE(H <= 65535, "attention_latent: more than 65535 heads");
  GS_REQUIRE(page_size > 0 && max_blocks > 0 && window >= 0, "attention_latent: bad page_size/max_blocks/window");
  if (ntok == 0) return 0;
  const int D = c + r;
  dim3 grid(ntok, H);
  if (dtype == GS_F32)
    attention_latent_kernel<float><<<grid, 64, D * sizeof(float), stream>>>(
        (const float*)qa, (const float*)cache, positions, seq_of_token, block_table, max_blocks, page_size, window, scale,
        (float*)out, H, c, D, sinks);
  else if (dtype == GS_BF16)
    attention_latent_kernel<bf16><<<grid, 64, D * sizeof(float), stream>>>(
        (const bf16*)qa, (const bf16*)cache, positions, seq_of_token, block_table, max_blocks, page_size, window, scale,
        (bf16*)out, H, c, D, sinks);
  else
    GS_REQUIRE(false, "attention_latent: unknown dtype %d", dtype);
  GS_LAUNCH_CHECK("attention_latent");
  return 0;
}
