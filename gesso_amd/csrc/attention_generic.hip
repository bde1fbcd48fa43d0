// Causal grouped-query attention over the paged cache: the generic kernel.
//
// Takes every head width up to 256, any number of heads and groups, any page size, an optional
// window, float32 or bfloat16 storage; all arithmetic is float32.  One wave per (query token,
// query head); a block of four where there are few in float32 (below).  The query at position p of sequence s sees keys lo..p of that sequence, lo = 0
// or p - window + 1; keys are read from the cache through the block table (this step's own
// keys were written there before).  Keys are walked in tiles of 64 starting at lo, with a running
// maximum and sum (online softmax), so the result for a position is the same however the
// sequence was cut into steps.
//
//   s_u = (q . k_u) * scale;  p_u = exp(s_u - max);  o = sum_u p_u v_u / sum_u p_u
//
// q (T, q_stride) with head h at columns [h d, (h+1) d); out (T, nh vd); key cache
// (num_pages, nkv, page_size, d), value cache (num_pages, nkv, page_size, vd).
//
// Further rules, each off unless asked for.  chunk > 0: positions are cut into runs of `chunk` from 0 on and a query
// sees only its own run, lo = max(lo, p - p % chunk).  sink: the denominator has one more term, exp(0 - max), which
// has no value: o = sum_u p_u v_u / (exp(-max) + sum_u p_u), the maximum taken over the scores and 0.  Value tables
// (max_position, vd/2): the cached values were turned by their own positions (rope_kv.hip), and the head's sum is
// turned back by the query's position, pair (a, b) -> (a cos + b sin, b cos - a sin), before it is stored.
// softcap > 0: s_u <- softcap tanh(s_u / softcap).  keep_first > 0 (with a window): the first keep_first positions of
// the sequence stay visible when the window has passed them; they are walked before the window's keys, at their own
// positions.  sinks (one float32 a head): the extra term of the denominator is exp(sinks[h] - max) instead of
// exp(0 - max); it is neither scaled nor capped.
#include "common.h"

#define GS_ATTN_MAX_D 256
#define GS_ATTN_ROWS 16

// PIECES > 0: key rows are whole pieces of 16 bytes, at addresses that are, PIECES of them in flight (4 where a row has no more:
// 8 requests of 5 keys, 4 heads of 8 in float32, 3.8 us, with 16 asked for 4.0).  A wavefront is bound by its chain of loads, so many are
// asked for before the first is used: LFM2-1.2B in float32, 6 requests, a portion of some 700 tokens and 16 decoded tokens over
// 150 keys each: 109 us a call on average with a number a load, 26 like this, the same bits.
template <typename T, int PIECES>
__global__ void attention_generic_kernel(const T* __restrict__ q, int q_stride, const T* __restrict__ kcache,
                                         const T* __restrict__ vcache, const int* __restrict__ positions,
                                         const int* __restrict__ seq_of_token, const int* __restrict__ block_table,
                                         int max_blocks, int page_size, int window, float scale, T* __restrict__ out,
                                         int nh, int nkv, int d, int vd, int chunk, int sink,
                                         const float* __restrict__ vcos, const float* __restrict__ vsin,
                                         int interleaved, float softcap, int keep_first,
                                         const float* __restrict__ sinks) {
  constexpr int E = 16 / sizeof(T);
  __shared__ float qs[GS_ATTN_MAX_D];
  __shared__ float ps[64];
  __shared__ long rowoff[64];
  int lane = threadIdx.x;
  int t = blockIdx.x, h = blockIdx.y;
  int kvh = h / (nh / nkv);
  int pos = positions[t];
  int seq = seq_of_token[t];
  const int* bt = block_table + (size_t)seq * max_blocks;
  for (int j = lane; j < d; j += 64) qs[j] = to_f32(q[(size_t)t * q_stride + (size_t)h * d + j]);
  __syncthreads();

  int lo = window > 0 ? (pos - window + 1 > 0 ? pos - window + 1 : 0) : 0;
  if (chunk > 0 && pos - pos % chunk > lo) lo = pos - pos % chunk;
  // the kept first positions that the window has passed: [lo0, hi0), walked before the window's keys
  int lo0 = chunk > 0 ? pos - pos % chunk : 0, hi0 = 0;
  if (window > 0 && keep_first > 0) hi0 = keep_first < pos - window + 1 ? keep_first : pos - window + 1;
  if (hi0 > lo) hi0 = lo;
  // with a sink the running maximum starts at the sink's score and the sum at its term
  float m = sinks ? sinks[h] : (sink ? 0.f : -INFINITY), l = (sink || sinks) ? 1.f : 0.f;
  float acc[GS_ATTN_MAX_D / 64];
#pragma unroll
  for (int i = 0; i < GS_ATTN_MAX_D / 64; ++i) acc[i] = 0.f;

  // two runs of keys: the kept first positions lo0 .. hi0 - 1 (where there are any), then lo .. pos
  for (int run = hi0 > lo0 ? 0 : 1; run < 2; ++run)
  for (int base = run ? lo : lo0, last = run ? pos : hi0 - 1; base <= last; base += 64) {
    int u = base + lane;
    float s = -INFINITY;
    long off = 0;
    if (u <= last) {
      int page = bt[u / page_size];
      off = ((long)page * nkv + kvh) * page_size + u % page_size;
      const T* kr = kcache + off * d;
      float dot = 0.f;
      if (PIECES > 0) {
        for (int j0 = 0; j0 < d; j0 += PIECES * E) {
          uint4 piece[PIECES > 0 ? PIECES : 1];
#pragma unroll
          for (int e = 0; e < PIECES; ++e)
            piece[e] = *reinterpret_cast<const uint4*>(kr + (j0 + e * E < d ? j0 + e * E : 0));
#pragma unroll
          for (int e = 0; e < PIECES; ++e)
            if (j0 + e * E < d) {
              T kv[E];
              __builtin_memcpy(kv, &piece[e], 16);
#pragma unroll
              for (int f = 0; f < E; ++f) dot = fmaf(qs[j0 + e * E + f], to_f32(kv[f]), dot);
            }
        }
      } else {
        for (int j = 0; j < d; ++j) dot = fmaf(qs[j], to_f32(kr[j]), dot);
      }
      s = dot * scale;
      if (softcap > 0.f) s = softcap * tanhf(s / softcap);
    }
    float m_new = fmaxf(m, wave_max(s));
    float p = u <= last ? expf(s - m_new) : 0.f;
    float alpha = expf(m - m_new);  // 0 on the first tile (m = -inf), since m_new is finite there
    l = l * alpha + wave_sum(p);
    m = m_new;
    __syncthreads();
    ps[lane] = p;
    rowoff[lane] = off;
    __syncthreads();
    int nk = last - base + 1 < 64 ? last - base + 1 : 64;
#pragma unroll
    for (int i = 0; i < GS_ATTN_MAX_D / 64; ++i) {
      int j = lane + 64 * i;
      if (j < vd) {
        float a = acc[i] * alpha;
        int k = 0;
        for (; k + GS_ATTN_ROWS <= nk; k += GS_ATTN_ROWS) {       // so many value rows in flight
          T v[GS_ATTN_ROWS];
#pragma unroll
          for (int e = 0; e < GS_ATTN_ROWS; ++e) v[e] = vcache[rowoff[k + e] * vd + j];
#pragma unroll
          for (int e = 0; e < GS_ATTN_ROWS; ++e) a = fmaf(ps[k + e], to_f32(v[e]), a);
        }
        for (; k < nk; ++k) a = fmaf(ps[k], to_f32(vcache[rowoff[k] * vd + j]), a);
        acc[i] = a;
      }
    }
  }
  float inv = 1.0f / l;
  if (vcos) {
    // the sum of turned values is turned back by the query's position
    __syncthreads();
#pragma unroll
    for (int i = 0; i < GS_ATTN_MAX_D / 64; ++i) {
      int j = lane + 64 * i;
      if (j < vd) qs[j] = acc[i] * inv;
    }
    __syncthreads();
    const int vh = vd >> 1;
    for (int i = lane; i < vh; i += 64) {
      const int ia = interleaved ? 2 * i : i, ib = interleaved ? 2 * i + 1 : i + vh;
      const float a = qs[ia], b = qs[ib];
      const float c = vcos[(size_t)pos * vh + i], sn = vsin[(size_t)pos * vh + i];
      out[((size_t)t * nh + h) * vd + ia] = from_f32<T>(a * c + b * sn);
      out[((size_t)t * nh + h) * vd + ib] = from_f32<T>(b * c - a * sn);
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < GS_ATTN_MAX_D / 64; ++i) {
    int j = lane + 64 * i;
    if (j < vd) out[((size_t)t * nh + h) * vd + j] = from_f32<T>(acc[i] * inv);
  }
}

#define GS_ATTN_FEW_WAVES 4

// Few queries (a decode step in float32) whose heads are at most 64 wide: a block of four wavefronts a (query token, query head), the
// same sums in the same order.  One wavefront alone waits for a tile's keys, then for its values, sixteen at a time, tile after tile; here
// each wavefront takes a tile of a round of four, asks for its keys and values at once, and leaves probabilities and values in LDS; the
// running maximum goes through the tiles' maxima in their order, and one wavefront adds up.  Keys beyond the last are the last one's row,
// loaded and not used.  D: the room of a row in LDS and the most a row is asked for in, the keys' or the values' width rounded up to 16, 32
// or 64.  (Microseconds by one wavefront and by four, 32 heads of 64 on 8, keys and values cold: 1 query of 20 keys 5.4 and 5.0, of 130
// 14.2 and 7.0, of 600 51.6 and 17.2, of 2,500 192 and 52; 8 queries 5.5 and 5.15, 14.9 and 7.35, 60 and 18.8, 225 and 57.  Heads of 32,
// 1 query of 5 keys 4.65 and 4.35, with room for 64 4.7; of 600 51 and 14.1, and 20 where the adding up read its values two at a time.  Heads
// of 8, 4 queries of 5 keys 4.1 and 3.9, with room for 64 4.5.)
template <int D>
__global__ __launch_bounds__(GS_ATTN_FEW_WAVES * 64) void attention_generic_few_kernel(
    const float* __restrict__ q, int q_stride, const float* __restrict__ kcache, const float* __restrict__ vcache,
    const int* __restrict__ positions, const int* __restrict__ seq_of_token, const int* __restrict__ block_table, int max_blocks,
    int page_size, int window, float scale, float* __restrict__ out, int nh, int nkv, int d, int vd, int chunk, int sink, float softcap,
    const float* __restrict__ sinks) {
  typedef __attribute__((ext_vector_type(4))) float f4;
  constexpr int NW = GS_ATTN_FEW_WAVES, PIECES = D / 4, TOGETHER = 64 / PIECES, LOADS = 64 / TOGETHER;   // rows of values a load, loads a tile
  extern __shared__ float values[];                      // (NW, 64, D)
  __shared__ float qs[D], ps[NW][64], tops[NW], sums[NW];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int t = blockIdx.x, h = blockIdx.y, kvh = h / (nh / nkv);
  const int pos = positions[t];
  const int* bt = block_table + (size_t)seq_of_token[t] * max_blocks;
  if (threadIdx.x < d) qs[threadIdx.x] = q[(size_t)t * q_stride + (size_t)h * d + threadIdx.x];
  int lo = window > 0 && pos - window + 1 > 0 ? pos - window + 1 : 0;
  if (chunk > 0 && pos - pos % chunk > lo) lo = pos - pos % chunk;
  float m = sinks ? sinks[h] : (sink ? 0.f : -INFINITY), l = (sink || sinks) ? 1.f : 0.f, acc = 0.f;
  const int piece = lane % PIECES, group = lane / PIECES;  // of a load of values: 16 bytes, of one of its rows
  float* mine = values + wave * 64 * D;
  for (int base = lo; base <= pos; base += 64 * NW) {
    const int u = base + 64 * wave + lane, there = u <= pos ? u : pos;
    const long off = ((long)bt[there / page_size] * nkv + kvh) * page_size + there % page_size;
    f4 kr[PIECES], vr[LOADS];
    const bool live = base + 64 * wave <= pos;           // (the same for the whole wavefront; a round's last tiles may hold no key)
    if (live) {
#pragma unroll
      for (int e = 0; e < PIECES; ++e) kr[e] = *reinterpret_cast<const f4*>(kcache + off * d + (4 * e < d ? 4 * e : 0));
#pragma unroll
      for (int e = 0; e < LOADS; ++e)
        vr[e] = *reinterpret_cast<const f4*>(vcache + __shfl(off, TOGETHER * e + group) * vd + (4 * piece < vd ? 4 * piece : 0));
    }
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();                                     // the queries are there, and the round before is added up
    float s = -INFINITY;
    if (live) {
      float dot = 0.f;
#pragma unroll
      for (int e = 0; e < PIECES; ++e)
        if (4 * e < d)
#pragma unroll
          for (int f = 0; f < 4; ++f) dot = fmaf(qs[4 * e + f], kr[e][f], dot);
      s = dot * scale;
      if (softcap > 0.f) s = softcap * tanhf(s / softcap);
      if (u > pos) s = -INFINITY;
#pragma unroll
      for (int e = 0; e < LOADS; ++e) *reinterpret_cast<f4*>(mine + (TOGETHER * e + group) * D + 4 * piece) = vr[e];
    }
    const float top = wave_max(s);
    if (lane == 0) tops[wave] = top;
    __syncthreads();
    float m_mine = m;
#pragma unroll
    for (int w = 0; w < NW; ++w)
      if (w <= wave) m_mine = fmaxf(m_mine, tops[w]);
    const float p = u <= pos ? expf(s - m_mine) : 0.f;
    const float sum = wave_sum(p);
    ps[wave][lane] = p;
    if (lane == 0) sums[wave] = sum;
    __syncthreads();
    for (int w = 0; w < NW && base + 64 * w <= pos; ++w) {
      const float m_new = fmaxf(m, tops[w]), alpha = expf(m - m_new);   // 0 on the first tile
      l = l * alpha + sums[w];
      m = m_new;
      if (wave == 0) {
        const int nk = pos - base - 64 * w + 1 < 64 ? pos - base - 64 * w + 1 : 64;
        const float* v = values + w * 64 * D + (lane < D ? lane : 0);
        float a = acc * alpha;
        int k = 0;
        for (; k + 16 <= nk; k += 16) {
          float x[16];
#pragma unroll
          for (int e = 0; e < 16; ++e) x[e] = v[(k + e) * D];
          __builtin_amdgcn_sched_barrier(0);               // (all sixteen asked for, not two at a time)
#pragma unroll
          for (int e = 0; e < 16; ++e) a = fmaf(ps[w][k + e], x[e], a);
        }
        for (; k < nk; ++k) a = fmaf(ps[w][k], v[k * D], a);
        acc = a;
      }
    }
  }
  if (wave == 0 && lane < vd) out[((size_t)t * nh + h) * vd + lane] = acc * (1.0f / l);
}

// Whether the four wavefronts pay: LDS has room for two such blocks a compute unit, 512 on the chip.  (One wavefront and four, 20, 160 and
// 600 keys: 16 queries of 32 heads 5.4, 16.4, 54 and 5.4, 9.2, 22 us; one query more 6.2, 19.5, 61 and 8.3, 15.2, 40; 32 queries 6.0, 20.2, 77
// and 9.2, 16.0, 46; 64 queries 6.9, 26, 97 and 16.6, 31, 88.  How many keys there are the host does not know: the
// first five of 16 queries are 5.25 and 5.5.)
static bool few_queries(int ntok, int nh, int d, int vd, const void* kcache, const void* vcache, const void* vcos, int window, int keep_first) {
  return (long)ntok * nh <= 512 && d <= 64 && vd <= 64 && d % 4 == 0 && vd % 4 == 0 && !vcos && !(window > 0 && keep_first > 0) &&
         (((uintptr_t)kcache | (uintptr_t)vcache) & 15) == 0;
}

extern "C" int gs_attention_generic(const void* q, int q_stride, const void* kcache, const void* vcache, int dtype,
                                    const int* positions, const int* seq_of_token, const int* block_table,
                                    int max_blocks, int page_size, int window, float scale, void* out, int ntok,
                                    int nh, int nkv, int d, int vd, int chunk, int sink, const float* vcos,
                                    const float* vsin, int interleaved, float softcap, int keep_first,
                                    const float* sinks, hipStream_t stream) {
  GS_REQUIRE(ntok >= 0 && nh > 0 && nkv > 0 && d > 0, "attention: bad sizes T=%d nh=%d nkv=%d d=%d", ntok, nh, nkv, d);
  GS_REQUIRE(nh % nkv == 0, "attention: %d query heads are no multiple of %d key heads", nh, nkv);
  GS_REQUIRE(d <= GS_ATTN_MAX_D, "attention: head width %d above the kernel's limit %d", d, GS_ATTN_MAX_D);
  GS_REQUIRE(nh <= 65535, "attention: more than 65535 heads");
  GS_REQUIRE(page_size > 0 && max_blocks > 0 && window >= 0, "attention: bad page_size/max_blocks/window");
  GS_REQUIRE(q_stride >= nh * d, "attention: q_stride %d below nh*d %d", q_stride, nh * d);
  GS_REQUIRE(vd > 0 && vd <= GS_ATTN_MAX_D, "attention: value width %d outside 1..%d", vd, GS_ATTN_MAX_D);
  GS_REQUIRE(chunk >= 0, "attention: bad chunk %d", chunk);
  GS_REQUIRE(softcap >= 0.f && keep_first >= 0, "attention: bad cap %f or kept positions %d", (double)softcap, keep_first);
  GS_REQUIRE(!(sink && sinks), "attention: the extra term is exp(0) or a head's own, not both");
  GS_REQUIRE((vcos == nullptr) == (vsin == nullptr) && (!vcos || vd % 2 == 0), "attention: value tables come together, for even widths");
  if (ntok == 0) return 0;
  dim3 grid(ntok, nh);
#define GS_RUN(T, PIECES)                                                                                              \
  attention_generic_kernel<T, PIECES><<<grid, 64, 0, stream>>>((const T*)q, q_stride, (const T*)kcache, (const T*)vcache, \
                                                            positions, seq_of_token, block_table, max_blocks, page_size, \
                                                            window, scale, (T*)out, nh, nkv, d, vd, chunk, sink, vcos,   \
                                                            vsin, interleaved, softcap, keep_first, sinks)
  const bool aligned = ((uintptr_t)kcache & 15) == 0;
  if (dtype == GS_F32 && few_queries(ntok, nh, d, vd, kcache, vcache, vcos, window, keep_first)) {
#define GS_FEW(D)                                                                                                              \
  do {                                                                                                                         \
    constexpr int lds = GS_ATTN_FEW_WAVES * 64 * D * sizeof(float);                                                            \
    if (D == 64) {                                                                                                             \
      /* with the rest more than the default limit of LDS: asked for once */                                                   \
      static const hipError_t asked = hipFuncSetAttribute(reinterpret_cast<const void*>(&attention_generic_few_kernel<D>),     \
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, lds);                    \
      (void)asked;                                                                                                             \
    }                                                                                                                          \
    attention_generic_few_kernel<D><<<grid, GS_ATTN_FEW_WAVES * 64, lds, stream>>>(                                            \
        (const float*)q, q_stride, (const float*)kcache, (const float*)vcache, positions, seq_of_token, block_table, max_blocks, page_size, \
        window, scale, (float*)out, nh, nkv, d, vd, chunk, sink, softcap, sinks);                                              \
  } while (0)
    const int wide = d > vd ? d : vd;
    if (wide <= 16) GS_FEW(16); else if (wide <= 32) GS_FEW(32); else GS_FEW(64);
#undef GS_FEW
  } else if (dtype == GS_F32) {
    if (aligned && d % 4 == 0) { if (d <= 16) GS_RUN(float, 4); else GS_RUN(float, 16); } else GS_RUN(float, 0);
  } else if (dtype == GS_BF16) {
    if (aligned && d % 8 == 0) { if (d <= 32) GS_RUN(bf16, 4); else GS_RUN(bf16, 16); } else GS_RUN(bf16, 0);
  } else {
    GS_REQUIRE(false, "attention: unknown dtype %d", dtype);
  }
#undef GS_RUN
  GS_LAUNCH_CHECK("attention_generic");
  return 0;
}
