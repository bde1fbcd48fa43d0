// Linear attention through a fading matrix state, and the norm and gate of its output.
//
// Per sequence and head a state S (n x m, float32, in the request's slot) is advanced token by token:
//
//   S <- decay_h S + k_t v_t^T,   o_t = S^T q_t
//
// q_t, k_t (n values) and v_t (m values) are columns of a row buffer x (T, ld): q of head h at [oq + h n, ...), k at
// [ok + h n, ...), v at [ov + h m, ...).  On their way in they may be activated (silu), q and k may be turned by the
// token's position (the first rd features of a head, feature i with i + rd/2, cos and sin from tables made on the
// host), and k may be scaled, all in float32: what enters the state is never rounded to the activation type again.
//
// linear_attention_scan: one block per (sequence, head, tile of 64 value columns); the columns of S are independent
// of each other, so wide values share out over blocks.  Lane l of wavefront w holds the state's rows rg, rg + 4, ...
// (rg = l / 16) of column 16 w + l % 16 in registers, so that sixteen lanes move 64 contiguous bytes of a row (8 rows, 16
// heads of 128 x 128: 8.15 us; neighbouring lanes in neighbouring rows were 0.5 us slower); the four partial sums of a column's output lie
// sixteen lanes apart.  A step's tokens come through LDS eight at a time.  The sums run in one fixed order per output, whatever
// the step's cut: a sequence fed whole, in portions or token by token leaves the same state and outputs, bit for bit.
// A step of single tokens is the same kernel with one token a block.  With `below` > 0 only the sequences that bring
// fewer tokens than that are taken: the longer ones go to the kernel on the matrix cores (linear_attention_mfma.hip).
//
// gated_outnorm: the heads' outputs of a token, normed in float32 (all heads as one row with a weight, or each head by
// its own root mean square, no weight) and multiplied by sigmoid or silu of a gate row.
#include "common.h"

#define LA_TB 8          // tokens staged at once
#define LA_COLS 64       // value columns a block

__device__ __forceinline__ float la_act(float z, int act) { return act ? z / (1.0f + expf(-z)) : z; }

template <typename TI, int RMAX>
__global__ void __launch_bounds__(256)
linear_attention_scan_kernel(const TI* __restrict__ x, int ld, int oq, int ok, int ov, int act,
                             const float* __restrict__ cos_t, const float* __restrict__ sin_t, int rd, float key_scale,
                             const float* __restrict__ decay, float* __restrict__ state,
                             const int* __restrict__ q_start, const int* __restrict__ slots,
                             const int* __restrict__ positions, float* __restrict__ out, int H, int n, int m,
                             int below) {
  constexpr int NMAX = 4 * RMAX;
  __shared__ float qs[LA_TB][NMAX];
  __shared__ float ks[LA_TB][NMAX];
  __shared__ float vs[LA_TB][LA_COLS];
  const int seq = blockIdx.x, h = blockIdx.y, j0 = blockIdx.z * LA_COLS;
  const int tid = threadIdx.x, rg = (tid >> 4) & 3, jl = (tid >> 6) * 16 + (tid & 15), j = j0 + jl;
  const int t0 = q_start[seq], t1 = q_start[seq + 1];
  if (t1 <= t0 || (below > 0 && t1 - t0 >= below)) return;      // (longer sequences are another kernel's)
  const float d = decay[h];
  float* S = state + (((size_t)slots[seq] * H + h) * n) * m;
  // The first token's values are asked for before the state (loads return in order: behind it they would come last, and the
  // conversion and the barrier after all of it).  A thread's feature, its partner of the rotation and its value column; what it has
  // none of is read from the first.  (8 rows, 16 heads of 128 x 128 10.35 and 8.15 us, one row 9.05 and 6.65, turned heads of 64 x 128 6.9 and
  // 5.85.)
  const int half = rd >> 1;
  const bool ahead = n <= 256;
  const int mine = tid < n ? tid : 0, pair = mine < half ? mine + half : mine < rd ? mine - half : mine;
  const TI* first = x + (size_t)t0 * ld;
  const TI q1 = first[oq + h * n + mine], k1 = first[ok + h * n + mine], q2 = first[oq + h * n + pair], k2 = first[ok + h * n + pair];
  const TI v1 = first[ov + h * m + (tid < LA_COLS && j0 + tid < m ? j0 + tid : 0)];
  float c1 = 1.f, s1 = 0.f;
  if (rd > 0) {
    const size_t at = (size_t)positions[t0] * half + (mine < half ? mine : mine < rd ? mine - half : 0);
    c1 = cos_t[at];
    s1 = sin_t[at];
  }
  float s[RMAX];
#pragma unroll
  for (int r = 0; r < RMAX; ++r) {
    const int i = rg + 4 * r;
    s[r] = (i < n && j < m) ? S[(size_t)i * m + j] : 0.f;
  }
  for (int tb = t0; tb < t1; tb += LA_TB) {
    const int nb = t1 - tb < LA_TB ? t1 - tb : LA_TB;
    __syncthreads();                                   // the batch before has been read
    const int done = ahead && tb == t0 ? 1 : 0;        // tokens of this batch whose values are at hand
    if (done) {
      float qv = la_act(to_f32(q1), act), kv = la_act(to_f32(k1), act);
      if (mine < rd) {
        const float qo = la_act(to_f32(q2), act), ko = la_act(to_f32(k2), act);
        qv = mine < half ? qv * c1 - qo * s1 : qv * c1 + qo * s1;
        kv = mine < half ? kv * c1 - ko * s1 : kv * c1 + ko * s1;
      }
      if (tid < n) {
        qs[0][tid] = qv;
        ks[0][tid] = kv * key_scale;
      }
      if (tid < LA_COLS) vs[0][tid] = j0 + tid < m ? la_act(to_f32(v1), act) : 0.f;
    }
    for (int idx = tid + done * n; idx < nb * n; idx += 256) {
      const int tt = idx / n, i = idx - tt * n;
      const TI* row = x + (size_t)(tb + tt) * ld;
      float qv = la_act(to_f32(row[oq + h * n + i]), act);
      float kv = la_act(to_f32(row[ok + h * n + i]), act);
      if (i < rd) {
        const bool low = i < half;
        const int p = low ? i : i - half, other = low ? i + half : i - half;
        const size_t at = (size_t)positions[tb + tt] * half + p;
        const float c = cos_t[at], sn = sin_t[at];
        const float qo = la_act(to_f32(row[oq + h * n + other]), act);
        const float ko = la_act(to_f32(row[ok + h * n + other]), act);
        // (u, v) -> (u cos - v sin, v cos + u sin)
        qv = low ? qv * c - qo * sn : qv * c + qo * sn;
        kv = low ? kv * c - ko * sn : kv * c + ko * sn;
      }
      qs[tt][i] = qv;
      ks[tt][i] = kv * key_scale;
    }
    for (int idx = tid + done * LA_COLS; idx < nb * LA_COLS; idx += 256) {
      const int tt = idx / LA_COLS, c = idx - tt * LA_COLS;
      vs[tt][c] = j0 + c < m ? la_act(to_f32(x[(size_t)(tb + tt) * ld + ov + h * m + j0 + c]), act) : 0.f;
    }
    __syncthreads();
    for (int tt = 0; tt < nb; ++tt) {
      const float vj = vs[tt][jl];
      float part = 0.f;
#pragma unroll
      for (int r = 0; r < RMAX; ++r) {
        const int i = rg + 4 * r;
        if (i < n) {
          s[r] = fmaf(ks[tt][i], vj, d * s[r]);
          part = fmaf(s[r], qs[tt][i], part);
        }
      }
      part += __shfl_xor(part, 16, 64);
      part += __shfl_xor(part, 32, 64);
      if (rg == 0 && j < m) out[((size_t)(tb + tt) * H + h) * m + j] = part;
    }
  }
#pragma unroll
  for (int r = 0; r < RMAX; ++r) {
    const int i = rg + 4 * r;
    if (i < n && j < m) S[(size_t)i * m + j] = s[r];
  }
}

extern "C" int gs_linear_attention_scan(const void* x, int dtype, int ld, int oq, int ok, int ov, int act,
                                        const float* cos_t, const float* sin_t, int rd, int max_position,
                                        float key_scale, const float* decay, float* state, const int* q_start,
                                        const int* slots, const int* positions, float* out, int nseq, int H, int n,
                                        int m, int below, hipStream_t stream) {
  GS_REQUIRE(nseq >= 0 && H > 0 && n > 0 && m > 0, "linear_attention: bad sizes nseq=%d H=%d n=%d m=%d", nseq, H, n, m);
  GS_REQUIRE(n <= 512, "linear_attention: keys of %d features, the kernel holds up to 512", n);
  GS_REQUIRE(H <= 65535 && (m + LA_COLS - 1) / LA_COLS <= 65535, "linear_attention: too many heads or value columns");
  GS_REQUIRE(rd >= 0 && rd <= n && rd % 2 == 0, "linear_attention: %d turned features of %d", rd, n);
  GS_REQUIRE(rd == 0 || (cos_t && sin_t && max_position > 0), "linear_attention: rotation without a table");
  GS_REQUIRE(oq >= 0 && ok >= 0 && ov >= 0 && oq + H * n <= ld && ok + H * n <= ld && ov + H * m <= ld,
             "linear_attention: q, k or v lie outside the rows of %d", ld);
  GS_REQUIRE(act == 0 || act == 1, "linear_attention: unknown activation %d", act);
  if (nseq == 0) return 0;
  dim3 grid(nseq, H, (m + LA_COLS - 1) / LA_COLS);
#define LA_RUN(TI, R)                                                                                                \
  linear_attention_scan_kernel<TI, R><<<grid, 256, 0, stream>>>((const TI*)x, ld, oq, ok, ov, act, cos_t, sin_t, rd, \
                                                                key_scale, decay, state, q_start, slots, positions,  \
                                                                out, H, n, m, below)
#define LA_RUN_T(TI)                      \
  if (n <= 32) LA_RUN(TI, 8);             \
  else if (n <= 64) LA_RUN(TI, 16);       \
  else if (n <= 128) LA_RUN(TI, 32);      \
  else if (n <= 256) LA_RUN(TI, 64);      \
  else LA_RUN(TI, 128)
  if (dtype == GS_F32) {
    LA_RUN_T(float);
  } else if (dtype == GS_BF16) {
    LA_RUN_T(bf16);
  } else {
    GS_REQUIRE(false, "linear_attention: unknown dtype %d", dtype);
  }
#undef LA_RUN_T
#undef LA_RUN
  GS_LAUNCH_CHECK("linear_attention_scan");
  return 0;
}

// A joint row of up to 8 TURNS values a thread (see gated_outnorm_kernel).
template <int TURNS, bool EARLY, typename TI, typename TO>
__device__ __forceinline__ void gated_outnorm_held(const float* __restrict__ row, const TI* __restrict__ g,
                                                   const float* __restrict__ w, float eps, int gate_act, TO* __restrict__ dst,
                                                   int W, float* red) {
  float v[TURNS][8], z[TURNS][8], wv[TURNS][8];
  float ss = 0.f;
  auto load = [&](int u) __attribute__((always_inline)) {
    const int c = (u * blockDim.x + threadIdx.x) * 8, at = c < W ? c : 0;
    load8f(g + at, z[u]);
    if (w) load8f(w + at, wv[u]);
  };
#pragma unroll
  for (int u = 0; u < TURNS; ++u) {
    const int c = (u * blockDim.x + threadIdx.x) * 8;
    load8f(row + (c < W ? c : 0), v[u]);
    if (EARLY) load(u);
  }
#pragma unroll
  for (int u = 0; u < TURNS; ++u)
    if ((int)(u * blockDim.x + threadIdx.x) * 8 < W) {
#pragma unroll
      for (int i = 0; i < 8; ++i) ss = fmaf(v[u][i], v[u][i], ss);
    }
  ss = block_sum(ss, red);
  const float inv = norm_inverse(ss, (float)W, eps);
#pragma unroll
  for (int u = 0; u < TURNS; ++u) {
    const int c = (u * blockDim.x + threadIdx.x) * 8;
    if (c >= W) break;
    if (!EARLY) load(u);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float sg = 1.0f / (1.0f + expf(-z[u][i]));
      v[u][i] = v[u][i] * inv * (w ? wv[u][i] : 1.f) * (gate_act ? z[u][i] * sg : sg);
    }
    store8f(dst + c, v[u]);
  }
}

// One block per token.  o (T, H m) float32; gate rows in a buffer (T, ldg) at column og.
//   joint: y = o / sqrt(mean over all H m values + eps) * w;   else, per head: y = o / sqrt(mean over the head's m + eps)
//   out = y * g(gate),  g = sigmoid (gate_act 0) or silu (1)
// EARLY (few rows, which are bound by the chain of loads): a row or head is asked for with its gate and weight before its sum
// (8 rows of 2048, joint and by heads of 128: 5.2 us, gate and weight asked for after it 5.9).  Many rows hide the chain, and
// the registers would cost wavefronts in flight (2,048 rows of 16 heads of 128 in float32: 12.7 us, early 13.7).  The sums are the same.
template <bool EARLY, typename TI, typename TO>
__global__ void gated_outnorm_kernel(const float* __restrict__ o, const TI* __restrict__ gate, int ldg, int og,
                                     const float* __restrict__ w, float eps, int joint, int gate_act,
                                     TO* __restrict__ out, int H, int m) {
  __shared__ float red[17];
  const int t = blockIdx.x, W = H * m;
  const float* row = o + (size_t)t * W;
  const TI* g = gate + (size_t)t * ldg + og;
  TO* dst = out + (size_t)t * W;
  if (joint && (W & 7) == 0 && W <= 8 * 256 * 4 && aligned16(row) && aligned16(g) && aligned16(dst) && (!w || aligned16(w))) {
    // eight values a thread and turn, rows up to 8192 values
    if (W <= 8 * (int)blockDim.x) gated_outnorm_held<1, EARLY>(row, g, w, eps, gate_act, dst, W, red);
    else if (W <= 16 * (int)blockDim.x) gated_outnorm_held<2, EARLY>(row, g, w, eps, gate_act, dst, W, red);
    else gated_outnorm_held<4, EARLY>(row, g, w, eps, gate_act, dst, W, red);
    return;
  }
  if (joint) {
    float ss = 0.f;
    for (int c = threadIdx.x; c < W; c += blockDim.x) ss += row[c] * row[c];
    ss = block_sum(ss, red);
    const float inv = norm_inverse(ss, (float)W, eps);
    for (int c = threadIdx.x; c < W; c += blockDim.x) {
      const float z = to_f32(g[c]);
      const float sg = 1.0f / (1.0f + expf(-z));
      dst[c] = from_f32<TO>(row[c] * inv * (w ? w[c] : 1.f) * (gate_act ? z * sg : sg));
    }
    return;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if (EARLY && m <= 256) {
    // a head is at most four values a lane; the next head's too are asked for before its sum
    float v[2][4], z[2][4], wv[2][4];
    auto load = [&](int b, int h) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = h * m + (lane + 64 * i < m ? lane + 64 * i : 0);
        v[b][i] = row[c];
        z[b][i] = to_f32(g[c]);
        wv[b][i] = w ? w[c] : 1.f;
      }
    };
    auto head = [&](int b, int h) __attribute__((always_inline)) {
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) ss = lane + 64 * i < m ? fmaf(v[b][i], v[b][i], ss) : ss;
      const float inv = norm_inverse(wave_sum(ss), (float)m, eps);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float sg = 1.0f / (1.0f + expf(-z[b][i]));
        if (lane + 64 * i < m)
          dst[h * m + lane + 64 * i] = from_f32<TO>(v[b][i] * inv * wv[b][i] * (gate_act ? z[b][i] * sg : sg));
      }
    };
    load(0, wave < H ? wave : 0);
    for (int h = wave; h < H; h += 2 * nw) {
      load(1, h + nw < H ? h + nw : h);
      head(0, h);
      load(0, h + 2 * nw < H ? h + 2 * nw : h);
      if (h + nw < H) head(1, h + nw);
    }
    return;
  }
  for (int h = wave; h < H; h += nw) {
    float ss = 0.f;
    for (int c = lane; c < m; c += 64) ss = fmaf(row[h * m + c], row[h * m + c], ss);
    ss = wave_sum(ss);
    const float inv = norm_inverse(ss, (float)m, eps);
    for (int c = lane; c < m; c += 64) {
      const float z = to_f32(g[h * m + c]);
      const float sg = 1.0f / (1.0f + expf(-z));
      dst[h * m + c] = from_f32<TO>(row[h * m + c] * inv * (w ? w[h * m + c] : 1.f) * (gate_act ? z * sg : sg));
    }
  }
}

extern "C" int gs_gated_outnorm(const float* o, const void* gate, int gate_dtype, int ldg, int og, const float* w,
                                float eps, int joint, int gate_act, void* out, int out_dtype, int T, int H, int m,
                                hipStream_t stream) {
  GS_REQUIRE(T >= 0 && H > 0 && m > 0, "gated_outnorm: bad sizes T=%d H=%d m=%d", T, H, m);
  GS_REQUIRE(eps > 0.f, "gated_outnorm: eps must be positive");
  GS_REQUIRE(og >= 0 && og + H * m <= ldg, "gated_outnorm: the gate lies outside the rows of %d", ldg);
  GS_REQUIRE(gate_dtype == out_dtype || gate_dtype == GS_F32, "gated_outnorm: the gate is float32 or of the result's type");
  if (T == 0) return 0;
  // Early: heads of 128 and more (16 of 128, 512 rows: 5.5 us, late 6.2; 2,048 in float32 13.7 and 12.7; narrower ones leave lanes
  // idle: of 64, 384 rows 4.8 and 4.6), joint rows up to 1,024 of them (1,536 of 300 values 4.9 and 4.0) and wide ones in bfloat16
  // (2,048 of 4096: 13.8 and 15.2).
  const bool early = joint ? T <= 1024 || (out_dtype == GS_BF16 && H * m >= 2048) : m >= 128 && (T <= 1536 || out_dtype == GS_BF16);
#define GS_RUN(TI, TO)                                                                                                      \
  if (early)                                                                                                                \
    gated_outnorm_kernel<true, TI, TO><<<T, 256, 0, stream>>>(o, (const TI*)gate, ldg, og, w, eps, joint, gate_act,         \
                                                              (TO*)out, H, m);                                              \
  else                                                                                                                      \
    gated_outnorm_kernel<false, TI, TO><<<T, 256, 0, stream>>>(o, (const TI*)gate, ldg, og, w, eps, joint, gate_act,        \
                                                               (TO*)out, H, m)
  if (out_dtype == GS_F32) {
    GS_RUN(float, float);
  } else if (out_dtype == GS_BF16 && gate_dtype == GS_F32) {
    GS_RUN(float, bf16);
  } else if (out_dtype == GS_BF16) {
    GS_RUN(bf16, bf16);
  } else {
    GS_REQUIRE(false, "gated_outnorm: unknown dtype %d", out_dtype);
  }
#undef GS_RUN
  GS_LAUNCH_CHECK("gated_outnorm");
  return 0;
}
