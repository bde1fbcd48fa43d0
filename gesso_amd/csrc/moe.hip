// A mixture of small feed-forwards routed by a table over token ids: the token-by-token kernels.
//
// Token t with id v uses the experts table[v, 0 .. top-1], each with weight 1 / top; an expert is
// W_down act(W_up x), act(z) = relu(z)^2.  Expert weights lie stacked: up (E, F, H), down (E, H, F).
//
//   moe_table_up     a[t, k, :] = act(W_up[e_k] x_t)                       one block per (token, choice)
//   moe_table_down   y[t, :] = (1 / top) sum_k W_down[e_k] a[t, k, :]      one block per (token, 32 columns)
//                    (+ sigmoid(g_t) * s[t, :] when a shared expert's output s and its gate g are given)
//   relu_squared     act over the first F columns of rows (the shared expert's inner rows)
//
// A wavefront computes ROWS = 4 outputs (1 where few tokens leave the chip idle): its lanes walk the weight rows together (contiguous loads), each lane summing its
// columns in ascending order, then the lanes' sums are added in a fixed order; products and sums are float32.  What binds is
// the expert's weights (32 pairs of 704 x 2048: 92 MB, 61 MB of them different), so the loads of all rows are in flight
// before the first is used, and before the token's row, which comes through LDS, has arrived.  Blocks are numbered slice of
// outputs first, in multiples of eight, and blocks go to the eight XCDs in turn: tokens that share an expert find a slice's
// weights in one XCD's L2.  8 tokens, 4 of 32 experts each, 704 x 2048: up 15.9 us, down 17.0 (a wavefront an output at a time,
// token first: 25.4 and 33.2; all blocks resident at once counts for more than more loads a wavefront: down with four visits in
// flight, half of the blocks waiting, 28.3).  Only the chosen experts' weights are read, which is what a step of few tokens needs; steps of many
// tokens go through the grouped products of moe_group.hip, which read an expert's weights once for all of its tokens.
#include "common.h"

#define MOE_WAVES 4

// ROWS rows of n weights in pieces of eight a lane, P pieces of 512 columns from column j0 on; a piece beyond the row's end
// reads the row's beginning (and is not used).
template <int ROWS, int P, typename TW>
struct MoePieces {
  float4 raw[ROWS][P][sizeof(TW) / 2];
  __device__ __forceinline__ void load(const TW* __restrict__ row, const size_t* at, int j0, int n) {
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const int j = j0 + 512 * p < n ? j0 + 512 * p : 0;
#pragma unroll
        for (int q = 0; q < (int)sizeof(TW) / 2; ++q) raw[r][p][q] = *(reinterpret_cast<const float4*>(row + at[r] + j) + q);
      }
  }
  __device__ __forceinline__ void add(float* s, const float* __restrict__ x, int j0, int n) const {
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int j = j0 + 512 * p;
      if (j < n) {
        float xv[8];
        load8f(x + j, xv);
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
          float w8[8];
          load8f(reinterpret_cast<const TW*>(&raw[r][p][0]), w8);
#pragma unroll
          for (int i = 0; i < 8; ++i) s[r] = fmaf(w8[i], xv[i], s[r]);
        }
      }
    }
  }
};

// n numbers of a row as floats into LDS, by the whole block.
template <typename T>
__device__ __forceinline__ void moe_stage(const T* __restrict__ row, float* __restrict__ to, int n) {
  if ((n & 7) == 0 && aligned16(row)) {
    for (int j = 8 * threadIdx.x; j < n; j += 8 * MOE_WAVES * 64) {
      float v[8];
      load8f(row + j, v);
      store8f(to + j, v);
    }
  } else {
    for (int j = threadIdx.x; j < n; j += MOE_WAVES * 64) to[j] = to_f32(row[j]);
  }
}

template <int ROWS, typename T, typename TW>
__global__ __launch_bounds__(MOE_WAVES * 64) void moe_table_up_kernel(const T* __restrict__ x, int ldx,
                                                                      const int* __restrict__ ids,
                                                                      const int* __restrict__ table, int top,
                                                                      const TW* __restrict__ up, int F, int H,
                                                                      T* __restrict__ a, int pairs) {
  extern __shared__ float4 staged[];
  float* xs = reinterpret_cast<float*>(staged);      // H floats
  constexpr int P = 4 / (sizeof(TW) / 2);
  const int pair = blockIdx.y + blockIdx.z * gridDim.y;
  if (pair >= pairs || (int)blockIdx.x * (MOE_WAVES * ROWS) >= F) return;      // (the grid's last slices are there for their number)
  const int t = pair / top, k = pair % top;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int f0 = blockIdx.x * (MOE_WAVES * ROWS) + wave * ROWS;
  const int e = table[(size_t)ids[t] * top + k];
  const TW* w = up + (size_t)e * F * H;
  T* dst = a + ((size_t)t * top + k) * F;
  // rows of whole 16-byte pieces: eight weights a lane and load (the order of the sums depends on H alone)
  const bool vec = (H & 7) == 0 && aligned16(w);
  size_t at[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) at[r] = (size_t)(f0 + r < F ? f0 + r : F - 1) * H;
  MoePieces<ROWS, P, TW> b;
  if (vec) b.load(w, at, lane * 8, H);
  moe_stage(x + (size_t)t * ldx, xs, H);
  __syncthreads();
  if (f0 >= F) return;
  float s[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) s[r] = 0.f;
  if (vec) {
    for (int j = lane * 8; j - lane * 8 < H; j += 512 * P) {
      b.add(s, xs, j, H);
      if (j - lane * 8 + 512 * P < H) b.load(w, at, j + 512 * P, H);
    }
  } else {
    for (int j = lane; j < H; j += 64) {          // (a number of every row before the next of the first: four loads in flight)
      const float xj = xs[j];
#pragma unroll
      for (int r = 0; r < ROWS; ++r) s[r] = fmaf(to_f32(w[at[r] + j]), xj, s[r]);
    }
  }
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const float v = wave_sum_dpp(s[r]);
    if (lane == 0 && f0 + r < F) {
      // the product is stored in the activation type before the activation, as a product of its own would be
      float z = to_f32(from_f32<T>(v));
      z = z > 0.f ? z : 0.f;
      dst[f0 + r] = from_f32<T>(z * z);
    }
  }
}

template <int ROWS, typename T, typename TW>
__global__ __launch_bounds__(MOE_WAVES * 64) void moe_table_down_kernel(const T* __restrict__ a, const int* __restrict__ ids,
                                                                        const int* __restrict__ table, int top,
                                                                        const TW* __restrict__ down, int F, int H,
                                                                        const T* __restrict__ shared,
                                                                        const T* __restrict__ gate, int ldg,
                                                                        T* __restrict__ y, int ntok) {
  extern __shared__ float4 staged[];
  float* as = reinterpret_cast<float*>(staged);      // top * F floats
  constexpr int P = 2 / (sizeof(TW) / 2);            // pieces a visit: a row of up to 1024 is one visit
  constexpr int D = 2;                               // visits in flight (4: 173 registers, half of the blocks wait for the others)
  const int t = blockIdx.y + blockIdx.z * gridDim.y;
  if (t >= ntok || (int)blockIdx.x * (MOE_WAVES * ROWS) >= H) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i0 = blockIdx.x * (MOE_WAVES * ROWS) + wave * ROWS;
  const float share = 1.0f / (float)top;
  const int* mine = table + (size_t)ids[t] * top;
  const bool vec = (F & 7) == 0 && aligned16(down);
  size_t at[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) at[r] = (size_t)(i0 + r < H ? i0 + r : H - 1) * F;
  const int per = (F + 512 * P - 1) / (512 * P), visits = top * per;      // visit v: piece group v % per of choice v / per
  MoePieces<ROWS, P, TW> b[D];
  auto load = [&](MoePieces<ROWS, P, TW>& p, int v) __attribute__((always_inline)) {
    v = v < visits ? v : visits - 1;
    p.load(down + (size_t)mine[v / per] * H * F, at, lane * 8 + v % per * 512 * P, F);
  };
  if (vec) {
#pragma unroll
    for (int d = 0; d < D; ++d) load(b[d], d);
  }
  moe_stage(a + (size_t)t * top * F, as, top * F);
  float g = 0.f;
  if (shared) g = 1.f / (1.f + expf(-to_f32(gate[(size_t)t * ldg])));
  __syncthreads();
  if (i0 >= H) return;
  float s[ROWS], total[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) s[r] = total[r] = 0.f;
  auto finish = [&]() __attribute__((always_inline)) {                    // a choice's sums are complete
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      total[r] += wave_sum_dpp(s[r]) * share;
      s[r] = 0.f;
    }
  };
  if (vec) {
    for (int v0 = 0; v0 < visits; v0 += D)
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const int v = v0 + d;
        if (v < visits) {
          b[d].add(s, as + (size_t)(v / per) * F, lane * 8 + v % per * 512 * P, F);
          if (v0 + D < visits) load(b[d], v + D);
          if (v % per == per - 1) finish();
        }
      }
  } else {
    for (int k = 0; k < top; ++k) {
      const TW* w = down + (size_t)mine[k] * H * F;
      for (int j = lane; j < F; j += 64) {
        const float aj = as[k * F + j];
#pragma unroll
        for (int r = 0; r < ROWS; ++r) s[r] = fmaf(to_f32(w[at[r] + j]), aj, s[r]);
      }
      finish();
    }
  }
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
    if (lane == 0 && i0 + r < H) {
      if (shared) total[r] += g * to_f32(shared[(size_t)t * H + i0 + r]);
      y[(size_t)t * H + i0 + r] = from_f32<T>(total[r]);
    }
}

template <typename T>
__global__ void relu_squared_kernel(const T* __restrict__ x, int ldx, T* __restrict__ out, int F, long total) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const long t = i / F;
  const int f = (int)(i % F);
  float z = to_f32(x[t * ldx + f]);
  z = z > 0.f ? z : 0.f;
  out[i] = from_f32<T>(z * z);
}

// Outputs a wavefront: four, or one where that makes no more than half a block a compute unit (the same sums; one token, 2 of 16
// experts of 512 x 1024: 7.3 us up and down, four at a time 9.2; two tokens 8.4 and 9.5).
static int moe_rows(int outputs, long of) { return gs_ceil_div(outputs, MOE_WAVES * 4) * of <= 128 ? 1 : 4; }

// Slices of outputs by what they are of (a launch takes 65535 in y); where there are more than eight, in a multiple of the
// eight XCDs that blocks go to in turn.
static dim3 moe_grid(int outputs, long of) {
  const int y = of < 65535 ? (int)of : 65535, slices = gs_ceil_div(outputs, MOE_WAVES * moe_rows(outputs, of));
  return dim3(slices > 8 ? gs_ceil_div(slices, 8) * 8 : slices, y, gs_ceil_div(of, y));
}

extern "C" int gs_moe_table_up(const void* x, int dtype, int ldx, const int* ids, const int* table, int top,
                               const void* up, int w_dtype, int F, int H, void* a, int ntok, hipStream_t stream) {
  GS_REQUIRE(ntok >= 0 && top > 0 && F > 0 && H > 0 && ldx >= H, "moe_table_up: bad sizes T=%d top=%d F=%d H=%d", ntok, top, F, H);
  GS_REQUIRE(H * sizeof(float) <= 65536, "moe_table_up: rows of %d are wider than the kernel's staging", H);
  if (ntok == 0) return 0;
  const dim3 grid = moe_grid(F, (long)ntok * top);
  const size_t lds = H * sizeof(float);
#define GS_RUN(T, TW)                                                                                                        \
  if (moe_rows(F, (long)ntok * top) == 1)                                                                                    \
    moe_table_up_kernel<1, T, TW><<<grid, MOE_WAVES * 64, lds, stream>>>((const T*)x, ldx, ids, table, top, (const TW*)up,   \
                                                                         F, H, (T*)a, ntok * top);                           \
  else                                                                                                                       \
    moe_table_up_kernel<4, T, TW><<<grid, MOE_WAVES * 64, lds, stream>>>((const T*)x, ldx, ids, table, top, (const TW*)up,   \
                                                                         F, H, (T*)a, ntok * top)
  if (dtype == GS_F32 && w_dtype == GS_F32) {
    GS_RUN(float, float);
  } else if (dtype == GS_BF16 && w_dtype == GS_BF16) {
    GS_RUN(bf16, bf16);
  } else if (dtype == GS_BF16 && w_dtype == GS_F32) {
    GS_RUN(bf16, float);
  } else {
    GS_REQUIRE(false, "moe_table_up: unsupported types %d %d", dtype, w_dtype);
  }
#undef GS_RUN
  GS_LAUNCH_CHECK("moe_table_up");
  return 0;
}

extern "C" int gs_moe_table_down(const void* a, int dtype, const int* ids, const int* table, int top, const void* down,
                                 int w_dtype, int F, int H, const void* shared, const void* gate, int ldg, void* y,
                                 int ntok, hipStream_t stream) {
  GS_REQUIRE(ntok >= 0 && top > 0 && F > 0 && H > 0, "moe_table_down: bad sizes T=%d top=%d F=%d H=%d", ntok, top, F, H);
  GS_REQUIRE((long)top * F * sizeof(float) <= 65536, "moe_table_down: %d x %d inner values are more than the kernel stages", top, F);
  GS_REQUIRE((shared == nullptr) == (gate == nullptr), "moe_table_down: a shared expert's rows come with their gate");
  if (ntok == 0) return 0;
  const dim3 grid = moe_grid(H, ntok);
  const size_t lds = (size_t)top * F * sizeof(float);
#define GS_RUN(T, TW)                                                                                                       \
  if (moe_rows(H, ntok) == 1)                                                                                               \
    moe_table_down_kernel<1, T, TW><<<grid, MOE_WAVES * 64, lds, stream>>>((const T*)a, ids, table, top, (const TW*)down,   \
                                                                           F, H, (const T*)shared, (const T*)gate, ldg,     \
                                                                           (T*)y, ntok);                                    \
  else                                                                                                                      \
    moe_table_down_kernel<4, T, TW><<<grid, MOE_WAVES * 64, lds, stream>>>((const T*)a, ids, table, top, (const TW*)down,   \
                                                                           F, H, (const T*)shared, (const T*)gate, ldg,     \
                                                                           (T*)y, ntok)
  if (dtype == GS_F32 && w_dtype == GS_F32) {
    GS_RUN(float, float);
  } else if (dtype == GS_BF16 && w_dtype == GS_BF16) {
    GS_RUN(bf16, bf16);
  } else if (dtype == GS_BF16 && w_dtype == GS_F32) {
    GS_RUN(bf16, float);
  } else {
    GS_REQUIRE(false, "moe_table_down: unsupported types %d %d", dtype, w_dtype);
  }
#undef GS_RUN
  GS_LAUNCH_CHECK("moe_table_down");
  return 0;
}

extern "C" int gs_relu_squared(const void* x, int dtype, int ldx, void* out, int ntok, int F, hipStream_t stream) {
  GS_REQUIRE(ntok >= 0 && F > 0 && ldx >= F, "relu_squared: bad sizes T=%d F=%d ldx=%d", ntok, F, ldx);
  if (ntok == 0) return 0;
  const long total = (long)ntok * F;
  const int blocks = gs_ceil_div(total, 256);
  if (dtype == GS_F32)
    relu_squared_kernel<float><<<blocks, 256, 0, stream>>>((const float*)x, ldx, (float*)out, F, total);
  else if (dtype == GS_BF16)
    relu_squared_kernel<bf16><<<blocks, 256, 0, stream>>>((const bf16*)x, ldx, (bf16*)out, F, total);
  else
    GS_REQUIRE(false, "relu_squared: unknown dtype %d", dtype);
  GS_LAUNCH_CHECK("relu_squared");
  return 0;
}
