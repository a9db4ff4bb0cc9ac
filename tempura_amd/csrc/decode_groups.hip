// Products of decode steps (at most 16 bfloat16 rows) that come in groups: several products whose inputs differ in one
// launch, and the two products of a layer of routed experts.  Their time is the weights' stream from memory, so a launch per
// group pays its start and its end once for all, and the weights of experts that no row of the step has chosen are not read.
//
// Rows are k-blocked, [K / 8, M, 8], weights tiled, [N / 16][K / 32][64][8] (see gemm_mfma.hip): every load of a wave is
// one run of neighbouring bytes.  A block owns 16 result columns; its eight waves split K in runs of 128 (run r of a weight
// goes to wave r % 8, whatever else is skipped), and their sums meet through LDS in the order of the waves, so a row's
// result has the same bits whatever the other rows are.
#include <math.h>

#include "common.h"
#include "activations.h"
#include "moe_route.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

#define DG_WAVES 8
#define DG_MAX_GROUPS 8
#define DG_MAX_EXPERTS 512

__device__ inline f32x4_t dg_mfma(u32x4_t w, u32x4_t x, f32x4_t acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w), __builtin_bit_cast(bf16x8_t, x), acc, 0, 0, 0);
}

// acc += the wave's runs of one 16-row tile of a weight: wp this lane's first piece of the tile, xp of the rows; steps of 32 k.  DEPTH runs on their way at
// a time (see gemm_few_kernel in gemm_mfma.hip and dg_deep).  One run: a decode step of Zemarax at width 4,096 494 -> 473 us with both, Golavik's 701 -> 675, Makisun's 461 -> 444.
template <int DEPTH = 1>
__device__ inline f32x4_t dg_tile(const u32x4_t* wp, const u32x4_t* xp, int xstep, int steps, int wave, f32x4_t acc) {
  const int runs = steps / 4;      // (whole ones)
  u32x4_t a[DEPTH][4], b[DEPTH][4];
  auto request = [&](int d, int run) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; ++u) a[d][u] = __builtin_nontemporal_load(wp + (size_t)(run * 4 + u) * 64);
#pragma unroll
    for (int u = 0; u < 4; ++u) b[d][u] = xp[(size_t)(run * 4 + u) * xstep];
  };
  auto multiply = [&](int d) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; ++u) acc = dg_mfma(a[d][u], b[d][u], acc);
  };
  int run = wave;
  if constexpr (DEPTH == 2) {
    for (; run + DG_WAVES < runs; run += 2 * DG_WAVES) {
      request(0, run);
      request(1, run + DG_WAVES);
      __builtin_amdgcn_sched_barrier(0);
      multiply(0);
      multiply(1);
    }
  }
  for (; run < runs; run += DG_WAVES) {
    request(0, run);
    __builtin_amdgcn_sched_barrier(0);      // (all of a run's loads in front of its first product)
    multiply(0);
  }
  if (wave == runs % DG_WAVES)     // what is left of K, fewer than four steps
    for (int s = runs * 4; s < steps; ++s) acc = dg_mfma(__builtin_nontemporal_load(wp + (size_t)s * 64), xp[(size_t)s * xstep], acc);
  return acc;
}

// Whether the waves of a product have two runs on their way: one or two rows with a long K and more blocks than CUs.  These are bound by the weights alone, and a
// block that comes to its end leaves a CU with one run a wave (more rows' own loads fill that, and with up to one block a CU the second run's place costs
// more than it gives).  One run / two, one row and two, us: four copies' closing product 13,824 x 5,120 32.5 / 31.2 and 32.5 / 31.2, 14,336 x 8,192 40.6 / 39.4 and 40.4 / 39.3,
// 28,672 x 8,192 77.4 / 74.6 and 76.8 / 74.7 (four rows 74.9 / 74.8), but 14,336 x 4,096 21.7 / 21.9 and 21.5 / 21.9, 8,192 x 2,048 11.3 / 11.5; groups 14,336 x
// 8,192 39.3 / 38.5, 4,096 x 8,192 13.2 / 13.1, but 2,048 x 4,096 4.9 / 5.0; experts, choice of two of eight, width 4,096 with 3,584 38.2 / 37.9 and 63.5 / 62.7, 6,144
// with 16,384 205 / 200 and 390 / 381, 8,192 with 4,096 72.1 / 71.1 and 133.8 / 129.0, but width 2,048 with 1,408 (six of 64) 35.8 / 37.6 and 54.1 / 57.4.
static bool dg_deep(int M, int K, int blocks) { return M <= 2 && K >= 4096 && blocks > 256; }

// the waves' sums of element q (lane q / 4, register q % 4) in wave order
__device__ inline float dg_sum(const float (*red)[256], int q) {
  float v = 0.f;
#pragma unroll
  for (int i = 0; i < DG_WAVES; ++i) v += red[i][q];
  return v;
}

// ---- several products in one launch -------------------------------------------------------------
// Rows n of the stacked weight belong to the first group g with n < end[g] (multiples of 16) and multiply the rows x + g * M * K.
struct GroupEnds {
  int end[DG_MAX_GROUPS];
};

template <int DEPTH>
__global__ __launch_bounds__(DG_WAVES * 64) void group_linear_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                                      float* __restrict__ out, GroupEnds ends, int M, int N, int K) {
  __shared__ float red[DG_WAVES][256];
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int n0 = blockIdx.x * 16;
  int g = 0;
#pragma unroll
  for (int i = 0; i < DG_MAX_GROUPS - 1; ++i) g += n0 >= ends.end[i] ? 1 : 0;
  const u32x4_t* wp = (const u32x4_t*)(w + (size_t)n0 * K) + lane;
  const int row = min(lane & 15, M - 1);
  const u32x4_t* xp = (const u32x4_t*)(x + (size_t)g * M * K + ((size_t)(lane >> 4) * M + row) * 8);
  const f32x4_t acc = dg_tile<DEPTH>(wp, xp, 4 * M, K / 32, wave, (f32x4_t){0.f, 0.f, 0.f, 0.f});
#pragma unroll
  for (int r = 0; r < 4; ++r) red[wave][lane * 4 + r] = acc[r];
  __syncthreads();
  const int q = threadIdx.x;
  if (q >= 256) return;
  const int l = q / 4, m = l & 15;
  const float v = dg_sum(red, q);
  if (m < M) out[(size_t)m * N + n0 + (l >> 4) * 4 + q % 4] = v;
}

// x: bfloat16, groups times [K / 8, M, 8]; w: tiled [N, K]; ends: host array, ends[groups - 1] == N; out float32 [M, N]
extern "C" int tp_group_linear(const void* x, const void* w, float* out, const int* ends, int groups, int M, int N, int K, hipStream_t s) {
  TP_REQUIRE(M > 0 && M <= 16 && N > 0 && N % 16 == 0 && K > 0 && K % 64 == 0, "group_linear: sizes M %d N %d K %d", M, N, K);
  TP_REQUIRE(groups > 0 && groups <= DG_MAX_GROUPS && ends[groups - 1] == N, "group_linear: %d groups", groups);
  TP_REQUIRE((((uintptr_t)x | (uintptr_t)w) & 15) == 0, "group_linear: operands must be aligned to 16 bytes");
  GroupEnds e;
  for (int i = 0; i < DG_MAX_GROUPS; ++i) {
    e.end[i] = i < groups ? ends[i] : N;
    TP_REQUIRE(e.end[i] % 16 == 0 && e.end[i] <= N && e.end[i] > (i > 0 && i < groups ? e.end[i - 1] : 0), "group_linear: bad group borders");
  }
  hipLaunchKernelGGL(dg_deep(M, K, N / 16) ? group_linear_kernel<2> : group_linear_kernel<1>, dim3(N / 16), dim3(DG_WAVES * 64), 0, s, (const bf16_t*)x, (const bf16_t*)w, out, e, M, N, K);
  TP_CHECK_LAUNCH("group_linear");
  return 0;
}

// ---- a product of few column blocks --------------------------------------------------------------
// out [splits, M, N] float32: partial sums over equal parts of K, for the kernel that consumes the rows to add.  A block owns 16 columns:
// at 2,048 of them half the CUs have no block, and each block walks all of K.  With the norm behind it, a captured chain, whole / in parts: 2,048 x 8,192 one row 12.8 / 11.0 us, sixteen 16.1 / 12.5; 1,024 x 8,192
// (four parts) 11.9 / 8.5 and 15.4 / 9.8; 2,048 x 4,096 9.3 / 8.5 and 11.3 / 9.7.
__global__ __launch_bounds__(DG_WAVES * 64) void split_linear_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                                      float* __restrict__ out, int M, int N, int K) {
  __shared__ float red[DG_WAVES][256];
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int n0 = blockIdx.x * 16, steps = K / 32 / gridDim.y, s0 = blockIdx.y * steps;
  const int row = min(lane & 15, M - 1);
  const u32x4_t* wp = (const u32x4_t*)(w + (size_t)n0 * K) + lane + (size_t)s0 * 64;
  const u32x4_t* xp = (const u32x4_t*)(x + ((size_t)(lane >> 4) * M + row) * 8) + (size_t)s0 * 4 * M;
  const f32x4_t acc = dg_tile(wp, xp, 4 * M, steps, wave, (f32x4_t){0.f, 0.f, 0.f, 0.f});
#pragma unroll
  for (int r = 0; r < 4; ++r) red[wave][lane * 4 + r] = acc[r];
  __syncthreads();
  const int q = threadIdx.x;
  if (q >= 256) return;
  const int l = q / 4, m = l & 15;
  if (m < M) out[((size_t)blockIdx.y * M + m) * N + n0 + (l >> 4) * 4 + q % 4] = dg_sum(red, q);
}

// x: bfloat16 [K / 8, M, 8]; w: tiled [N, K]; K in `splits` equal parts of whole steps of 32
extern "C" int tp_split_linear(const void* x, const void* w, float* out, int M, int N, int K, int splits, hipStream_t s) {
  TP_REQUIRE(M > 0 && M <= 16 && N > 0 && N % 16 == 0 && K > 0 && K % 64 == 0 && splits >= 1 && splits <= 16 && K / 32 % splits == 0,
             "split_linear: sizes M %d N %d K %d in %d parts", M, N, K, splits);
  TP_REQUIRE((((uintptr_t)x | (uintptr_t)w) & 15) == 0, "split_linear: operands must be aligned to 16 bytes");
  hipLaunchKernelGGL(split_linear_kernel, dim3(N / 16, splits), dim3(DG_WAVES * 64), 0, s, (const bf16_t*)x, (const bf16_t*)w, out, M, N, K);
  TP_CHECK_LAUNCH("split_linear");
  return 0;
}

// ---- a product that closes a sublayer over several copies of the stream ---------------------------
// y = x w^T, then per row and column, in the order of hc_step_reg_kernel: h'[b] = sum_a mix[a, b] h[a] + outc[b] y, written back into
// h [M, S, N]; with norm_w also u = sum_a inc[a] h'[a], handed over as xg = bfloat16(u * norm_w), k-blocked [N / 8, M, 8], and ss
// [M, N / 16], each block's sums of u^2 per row, for the next product to finish the norm (RowScale in gemm_mfma.hip).  The copies mix
// column by column, so the block that has a column's sum has all it needs; what it reads besides is requested before the weights.
// Bound by the weights' stream, as the product alone.  Four copies, a captured chain, product and closing kernel / together, one row and
// eight: 4,096 x 4,096 11.4 / 8.4 and 12.8 / 8.9 us, 4,096 x 14,336 25.2 / 22.1 and 26.5 / 22.8, 2,048 x 7,168 13.7 / 11.5 and 15.2 / 12.2,
// 1,024 x 2,048 6.8 / 4.7 and 7.3 / 4.7; sixteen rows of 4,096 x 14,336 28.9 / 25.1.
struct StreamEnd {
  const float *mix, *outc, *inc, *norm_w;   // nullptr: identity, ones, ones, no norm behind
  bf16_t* xg;
  float* ss;
};

template <int DEPTH>
__global__ __launch_bounds__(DG_WAVES * 64) void stream_linear_kernel(const bf16_t* __restrict__ x, int blocked, const bf16_t* __restrict__ w,
                                                                       float* __restrict__ h, StreamEnd e, int M, int N, int K) {
  __shared__ float red[DG_WAVES][256];
  __shared__ float part[4][16];
  constexpr int S = 4;
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int n0 = blockIdx.x * 16;
  const int q = threadIdx.x, l = q / 4, m = l & 15, n = n0 + ((l >> 4) & 3) * 4 + q % 4;
  const bool mine = q < 256 && m < M;
  float v[S], wn = 0.f, mc[S * S], oc[S], ic[S];
  float* hp = h + (size_t)m * S * N + n;
  if (mine) {
#pragma unroll
    for (int a = 0; a < S; ++a) v[a] = hp[(size_t)a * N];
    if (e.norm_w != nullptr) wn = e.norm_w[n];
  }
#pragma unroll
  for (int a = 0; a < S; ++a) {
#pragma unroll
    for (int b = 0; b < S; ++b) mc[a * S + b] = e.mix ? e.mix[a * S + b] : (a == b ? 1.f : 0.f);
    oc[a] = e.outc ? e.outc[a] : 1.f;
    ic[a] = e.inc ? e.inc[a] : 1.f;
  }
  const u32x4_t* wp = (const u32x4_t*)(w + (size_t)n0 * K) + lane;
  const int row = min(lane & 15, M - 1);
  const u32x4_t* xp = blocked ? (const u32x4_t*)x + (size_t)(lane >> 4) * M + row : (const u32x4_t*)(x + (size_t)row * K) + (lane >> 4);
  const f32x4_t acc = dg_tile<DEPTH>(wp, xp, blocked ? 4 * M : 4, K / 32, wave, (f32x4_t){0.f, 0.f, 0.f, 0.f});
#pragma unroll
  for (int r = 0; r < 4; ++r) red[wave][lane * 4 + r] = acc[r];
  __syncthreads();
  if (q < 256) {
    float sq = 0.f;
    if (mine) {
      const float y = dg_sum(red, q);
      float u = 0.f;
#pragma unroll
      for (int b = 0; b < S; ++b) {
        float t = 0.f;
#pragma unroll
        for (int a = 0; a < S; ++a) t = fmaf(mc[a * S + b], v[a], t);
        t = fmaf(oc[b], y, t);
        hp[(size_t)b * N] = t;
        u = fmaf(ic[b], t, u);
      }
      if (e.norm_w != nullptr) e.xg[((size_t)(n >> 3) * M + m) * 8 + (n & 7)] = float_to_bf16(u * wn);
      sq = u * u;
    }
    sq += __shfl_xor(sq, 1, 64);      // the four columns of this lane's row
    sq += __shfl_xor(sq, 2, 64);
    if (q % 4 == 0) part[l >> 4][m] = sq;
  }
  if (e.norm_w == nullptr) return;   // (the same for every thread)
  __syncthreads();
  if ((int)threadIdx.x < M)
    e.ss[threadIdx.x * gridDim.x + blockIdx.x] = part[0][threadIdx.x] + part[1][threadIdx.x] + part[2][threadIdx.x] + part[3][threadIdx.x];
}

// x: bfloat16 [K / 8, M, 8] (blocked) or [M, K]; w: tiled [N, K]; h float32 [M, streams, N]; mix float32 [streams, streams], outc and inc
// [streams], norm_w [N] (each may be nullptr); xg bfloat16 [N / 8, M, 8] and ss [M, N / 16] with norm_w
extern "C" int tp_stream_linear(const void* x, int blocked, const void* w, float* h, int streams, const float* mix, const float* outc,
                                const float* inc, const float* norm_w, void* xg, float* ss, int M, int N, int K, hipStream_t s) {
  TP_REQUIRE(M > 0 && M <= 16 && N > 0 && N % 16 == 0 && K > 0 && K % 64 == 0, "stream_linear: sizes M %d N %d K %d", M, N, K);
  TP_REQUIRE((((uintptr_t)x | (uintptr_t)w) & 15) == 0, "stream_linear: operands must be aligned to 16 bytes");
  TP_REQUIRE(norm_w == nullptr || (xg != nullptr && ss != nullptr), "stream_linear: no room for the rows of the next norm");
  const StreamEnd e = {mix, outc, inc, norm_w, (bf16_t*)xg, ss};
  TP_REQUIRE(streams == 4, "stream_linear: %d copies of the stream (takes 4)", streams);
  hipLaunchKernelGGL(dg_deep(M, K, N / 16) ? stream_linear_kernel<2> : stream_linear_kernel<1>, dim3(N / 16), dim3(DG_WAVES * 64), 0, s, (const bf16_t*)x, blocked, (const bf16_t*)w, h, e, M, N, K);
  TP_CHECK_LAUNCH("stream_linear");
  return 0;
}

// ---- routed experts ---------------------------------------------------------------------------------
// Up: a[m][e * ff + c] = f(x_m . up_e[c]) * dense[m][e] as bfloat16, k-blocked over the columns of all experts; experts whose
// column of `dense` is zero for all rows are skipped (their columns stay unwritten).  GATED: the weight's rows alternate
// eight gate rows and eight up rows, and f is silu(gate) * up.
template <bool GATED, int DEPTH>
__global__ __launch_bounds__(DG_WAVES * 64) void moe_up_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                                const float* __restrict__ dense, bf16_t* __restrict__ a, int M, int experts,
                                                                int rows, int K, int kind) {
  __shared__ float red[DG_WAVES][256];
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int n0 = blockIdx.x * 16, e = n0 / rows;
  const float mine = lane < M ? dense[(size_t)lane * experts + e] : 0.f;
  if (__ballot(mine != 0.f) == 0ull) return;   // (the same for every wave of the block)
  const u32x4_t* wp = (const u32x4_t*)(w + (size_t)n0 * K) + lane;
  const int row = min(lane & 15, M - 1);
  const u32x4_t* xp = (const u32x4_t*)(x + ((size_t)(lane >> 4) * M + row) * 8);
  const f32x4_t acc = dg_tile<DEPTH>(wp, xp, 4 * M, K / 32, wave, (f32x4_t){0.f, 0.f, 0.f, 0.f});
#pragma unroll
  for (int r = 0; r < 4; ++r) red[wave][lane * 4 + r] = acc[r];
  __syncthreads();
  const int q = threadIdx.x;
  if (q >= (GATED ? 128 : 256)) return;
  const int l = q / 4, m = l & 15;
  if (m >= M) return;
  const float weight = dense[(size_t)m * experts + e];
  const float v = dg_sum(red, q);
  float y;
  if (GATED) {
    const float u = dg_sum(red, q + 128);   // (a gate row's up row is eight further on)
    y = act_f(v, 1) * u;
  } else {
    y = act_f(v, kind);
  }
  const int n = (GATED ? n0 / 2 : n0) + (l >> 4) * 4 + q % 4;
  a[((size_t)(n >> 3) * M + m) * 8 + (n & 7)] = float_to_bf16(weight == 0.f ? 0.f : y * weight);
}

// Opens a layer of routed experts: block 0 works out the router's logits and every row's choice, the others are the up product of
// an expert that every row uses (w tiled [rows >= size, K], activated; with `gated` its row `size` is a gate's, left raw in g [M]),
// which needs no choice and keeps the memory busy meanwhile.  The logits are formed in the order of the products of a few rows.
// Router product, choice, shared up product, its activation and its down product were launches of their own, 3 to 6 us each of which
// half is the chain: a layer of eight experts and a shared one at width 4,096, three rows, 79 -> 60 us of kernels (58 MB of them shared).
#define DG_OPEN_EXPERTS 64
__global__ __launch_bounds__(DG_WAVES * 64) void moe_open_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w_router, Route r,
                                                                  const bf16_t* __restrict__ w, bf16_t* __restrict__ a, float* __restrict__ g,
                                                                  int M, int K, int size, int kind, int gated) {
  __shared__ float red[DG_WAVES][256];
  __shared__ float logits[16][DG_OPEN_EXPERTS];
  __shared__ float route_lds[DG_WAVES][2 * DG_OPEN_EXPERTS];
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int row = min(lane & 15, M - 1);
  const u32x4_t* xp = (const u32x4_t*)(x + ((size_t)(lane >> 4) * M + row) * 8);
  const int q = threadIdx.x, l = q / 4, m = l & 15;
  if (blockIdx.x > 0) {
    const int n0 = (blockIdx.x - 1) * 16;
    const f32x4_t acc = dg_tile((const u32x4_t*)(w + (size_t)n0 * K) + lane, xp, 4 * M, K / 32, wave, (f32x4_t){0.f, 0.f, 0.f, 0.f});
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wave][lane * 4 + i] = acc[i];
    __syncthreads();
    if (q >= 256 || m >= M) return;
    const float v = dg_sum(red, q);
    const int n = n0 + (l >> 4) * 4 + q % 4;
    if (n < size) a[((size_t)(n >> 3) * M + m) * 8 + (n & 7)] = float_to_bf16(act_f(v, kind));
    else if (gated && n == size) g[m] = v;
    return;
  }
  for (int e0 = 0; e0 < r.experts; e0 += 16) {
    const u32x4_t* wp = (const u32x4_t*)(w_router + (size_t)e0 * K) + lane;
    // (rows of the tile past the last expert are not read)
    const bool mine = e0 + (lane & 15) < r.experts;
    f32x4_t acc = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    const int steps = K / 32;
    for (int s0 = wave * 4; s0 < steps; s0 += DG_WAVES * 8) {
      u32x4_t av[2][4], bv[2][4];
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int st = min(s0 + d * DG_WAVES * 4 + u, steps - 1);
          av[d][u] = (u32x4_t){0u, 0u, 0u, 0u};
          if (mine) av[d][u] = wp[(size_t)st * 64];
          bv[d][u] = xp[(size_t)st * 4 * M];
        }
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (s0 + d * DG_WAVES * 4 + u < steps) acc = dg_mfma(av[d][u], bv[d][u], acc);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wave][lane * 4 + i] = acc[i];
    __syncthreads();
    if (q < 256 && e0 + (l >> 4) * 4 + q % 4 < DG_OPEN_EXPERTS) logits[m][e0 + (l >> 4) * 4 + q % 4] = dg_sum(red, q);
    __syncthreads();
  }
  if (r.experts <= ROUTE_FEW) {
    if (wave < 4) route_few(r, logits[q / ROUTE_FEW], q / ROUTE_FEW, q / ROUTE_FEW < M);
    return;
  }
  for (int t0 = 0; t0 < M; t0 += DG_WAVES) {
    const int t = min(t0 + wave, M - 1);
    route_token<1>(r, logits[t], t, t0 + wave < M, route_lds[wave], route_lds[wave] + DG_OPEN_EXPERTS);
    __syncthreads();
  }
}

// x: bfloat16 [K / 8, M, 8]; w_router: tiled [experts rounded up to 16, K]; the outputs of tp_moe_route; w_shared: tiled [shared_rows, K]
// (nullptr: none), its first `size` rows activated into a_shared bfloat16 [size / 8, M, 8], row `size` with gate != nullptr into gate [M].
extern "C" int tp_moe_open(const void* x, const void* w_router, const float* correction, const float* logit_bias, int experts, int top, int groups,
                           int keep, float* dense, int* ids, float* weights, int M, int K, int score_kind, int group_best, int normalize,
                           float sum_eps, float scale, const void* w_shared, int shared_rows, int size, int kind, void* a_shared, float* gate,
                           hipStream_t s) {
  TP_REQUIRE(M > 0 && M <= 16 && K > 0 && K % 64 == 0, "moe_open: %d rows of %d", M, K);
  TP_REQUIRE(experts > 0 && experts <= DG_OPEN_EXPERTS && top > 0 && top <= experts && (groups <= 1 || (experts % groups == 0 && keep >= 1 && keep <= groups)) &&
                 (score_kind == 0 || score_kind == 1) && group_best >= 1,
             "moe_open: bad router");
  TP_REQUIRE(w_shared == nullptr || (shared_rows % 16 == 0 && size > 0 && size % 8 == 0 && size + (gate != nullptr ? 1 : 0) <= shared_rows && kind >= 0 &&
                                     kind <= 3 && a_shared),
             "moe_open: bad shared expert");
  TP_REQUIRE((((uintptr_t)x | (uintptr_t)w_router | (uintptr_t)w_shared | (uintptr_t)a_shared) & 15) == 0, "moe_open: operands must be aligned to 16 bytes");
  const Route r = {correction, logit_bias, experts, top, groups, keep, score_kind, group_best, normalize, sum_eps, scale, dense, ids, weights};
  hipLaunchKernelGGL(moe_open_kernel, dim3(1 + (w_shared != nullptr ? shared_rows / 16 : 0)), dim3(DG_WAVES * 64), 0, s, (const bf16_t*)x,
                     (const bf16_t*)w_router, r, (const bf16_t*)w_shared, (bf16_t*)a_shared, gate, M, K, size, kind, gate != nullptr ? 1 : 0);
  TP_CHECK_LAUNCH("moe_open");
  return 0;
}

// Down: y[m] (+)= sum_e a[m][e] . down_e, experts ascending; the same experts are skipped.  w: every expert's tiled [N, ff], one
// behind the other.  gridDim.y > 1: every expert's K in that many equal parts of whole runs, y [parts, M, N] (see split_linear_kernel).
// ws: then the shared expert's tiled [N, size] (nullptr: none) times a_shared, its sum added on its own, times
// sigmoid(gate[m]) where there is a gate.
template <int DEPTH>
__global__ __launch_bounds__(DG_WAVES * 64) void moe_down_kernel(const bf16_t* __restrict__ a, const bf16_t* __restrict__ w,
                                                                  const float* __restrict__ dense, float* __restrict__ y, int M, int experts,
                                                                  int ff, int N, int accumulate, const bf16_t* __restrict__ ws,
                                                                  const bf16_t* __restrict__ a_shared, const float* __restrict__ gate, int size) {
  __shared__ float red[DG_WAVES][256], red_s[DG_WAVES][256];
  __shared__ int list[DG_MAX_EXPERTS];
  __shared__ int counts[DG_WAVES];
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  // the experts in use, ascending
  bool used = false;
  if ((int)threadIdx.x < experts)
    for (int m = 0; m < M; ++m) used = used || dense[(size_t)m * experts + threadIdx.x] != 0.f;
  const unsigned long long mask = __ballot(used);
  if (lane == 0) counts[wave] = __popcll(mask);
  __syncthreads();
  int before = 0, total = 0;
#pragma unroll
  for (int i = 0; i < DG_WAVES; ++i) {
    if (i < wave) before += counts[i];
    total += counts[i];
  }
  if (used) list[before + __popcll(mask & ((1ull << lane) - 1ull))] = threadIdx.x;
  __syncthreads();

  const int n0 = blockIdx.x * 16, steps = ff / 32 / gridDim.y, runs = (steps + 3) / 4;
  const int row = min(lane & 15, M - 1);
  const int xstep = 4 * M;
  const size_t first = (size_t)blockIdx.y * steps;
  const u32x4_t* w_lane = (const u32x4_t*)(w + (size_t)n0 * ff) + lane + first * 64;
  const u32x4_t* x_lane = (const u32x4_t*)(a + ((size_t)(lane >> 4) * M + row) * 8) + first * xstep;
  const size_t w_expert = (size_t)N * ff / 8, x_expert = (size_t)(ff / 8) * M;   // in pieces of 16 bytes
  // run r of expert e goes to wave (e * runs + r) % 8: `per` turns an expert
  const int per = (runs + DG_WAVES - 1) / DG_WAVES;
  f32x4_t acc = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  int it = 0;
  if constexpr (DEPTH == 2) {      // (every expert's runs are whole and a multiple of the waves)
    for (; it + 1 < total * per; it += 2) {
      u32x4_t av[2][4], bv[2][4];
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        const int e = __builtin_amdgcn_readfirstlane(list[(it + d) / per]);
        const int run = (it + d) % per * DG_WAVES + ((wave - e * runs) & (DG_WAVES - 1));
        const u32x4_t* wp = w_lane + (size_t)e * w_expert + (size_t)run * 256;
        const u32x4_t* xp = x_lane + (size_t)e * x_expert + (size_t)run * 4 * xstep;
#pragma unroll
        for (int u = 0; u < 4; ++u) av[d][u] = __builtin_nontemporal_load(wp + u * 64);
#pragma unroll
        for (int u = 0; u < 4; ++u) bv[d][u] = xp[(size_t)u * xstep];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int u = 0; u < 4; ++u) acc = dg_mfma(av[d][u], bv[d][u], acc);
    }
  }
  for (; it < total * per; ++it) {
    const int e = __builtin_amdgcn_readfirstlane(list[it / per]);
    const int run = it % per * DG_WAVES + ((wave - e * runs) & (DG_WAVES - 1));
    if (run >= runs) continue;
    const u32x4_t* wp = w_lane + (size_t)e * w_expert + (size_t)run * 256;
    const u32x4_t* xp = x_lane + (size_t)e * x_expert + (size_t)run * 4 * xstep;
    const int left = steps - run * 4;
    if (left >= 4) {
      u32x4_t av[4], bv[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) av[u] = __builtin_nontemporal_load(wp + u * 64);
#pragma unroll
      for (int u = 0; u < 4; ++u) bv[u] = xp[(size_t)u * xstep];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 4; ++u) acc = dg_mfma(av[u], bv[u], acc);
    } else {
      for (int u = 0; u < left; ++u) acc = dg_mfma(__builtin_nontemporal_load(wp + u * 64), xp[(size_t)u * xstep], acc);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) red[wave][lane * 4 + r] = acc[r];
  if (ws != nullptr) {
    const int steps_s = size / 32 / gridDim.y;
    const size_t first_s = (size_t)blockIdx.y * steps_s;
    const f32x4_t sum = dg_tile((const u32x4_t*)(ws + (size_t)n0 * size) + lane + first_s * 64,
                                (const u32x4_t*)(a_shared + ((size_t)(lane >> 4) * M + row) * 8) + first_s * xstep, xstep, steps_s, wave,
                                (f32x4_t){0.f, 0.f, 0.f, 0.f});
#pragma unroll
    for (int r = 0; r < 4; ++r) red_s[wave][lane * 4 + r] = sum[r];
  }
  __syncthreads();
  const int q = threadIdx.x;
  if (q >= 256) return;
  const int l = q / 4, m = l & 15;
  if (m >= M) return;
  float* o = y + ((size_t)blockIdx.y * M + m) * N + n0 + (l >> 4) * 4 + q % 4;
  float v = dg_sum(red, q);
  if (accumulate) v = *o + v;
  if (ws != nullptr) {
    const float sv = dg_sum(red_s, q);
    v += gate != nullptr ? sv * (1.0f / (1.0f + expf(-gate[m]))) : sv;
  }
  *o = v;
}

// x: bfloat16 [K / 8, M, 8]; w_up: tiled [experts * rows, K], rows = ff, or 2 ff with gated (kind is then not read); w_down: experts
// tiled [N, ff]; dense float32 [M, experts]; a: bfloat16 scratch [experts * ff / 8, M, 8]; y float32 [M, N].  w_shared (nullptr: none):
// tiled [N, size], a_shared and gate (nullptr: none) as tp_moe_open leaves them.  parts > 1: y [parts, M, N], partial sums.
extern "C" int tp_moe_few(const void* x, const void* w_up, const void* w_down, const float* dense, void* a, float* y, int M, int experts,
                          int ff, int K, int N, int gated, int kind, int accumulate, const void* w_shared, const void* a_shared, const float* gate,
                          int size, int parts, hipStream_t s) {
  TP_REQUIRE(parts >= 1 && parts <= 16 && (parts == 1 || (!accumulate && ff / 32 % parts == 0 && (w_shared == nullptr || size / 32 % parts == 0))),
             "moe_few: K in %d parts", parts);
  TP_REQUIRE(w_shared == nullptr || (size > 0 && size % 64 == 0 && a_shared && (((uintptr_t)w_shared | (uintptr_t)a_shared) & 15) == 0),
             "moe_few: bad shared expert");
  TP_REQUIRE(M > 0 && M <= 16 && experts > 0 && experts <= DG_MAX_EXPERTS, "moe_few: %d rows, %d experts", M, experts);
  TP_REQUIRE(ff > 0 && ff % 64 == 0 && K > 0 && K % 64 == 0 && N > 0 && N % 16 == 0, "moe_few: sizes ff %d K %d N %d", ff, K, N);
  TP_REQUIRE(gated || (kind >= 0 && kind <= 3), "moe_few: unknown activation %d", kind);
  TP_REQUIRE((((uintptr_t)x | (uintptr_t)w_up | (uintptr_t)w_down | (uintptr_t)a) & 15) == 0, "moe_few: operands must be aligned to 16 bytes");
  const int rows = gated ? 2 * ff : ff;
  TP_REQUIRE((long)experts * rows < 0x7fffffffL, "moe_few: too many rows");
  const dim3 up(experts * rows / 16), block(DG_WAVES * 64);
  const bool deep = dg_deep(M, K, experts * rows / 16);
  if (gated)
    hipLaunchKernelGGL((deep ? moe_up_kernel<true, 2> : moe_up_kernel<true, 1>), up, block, 0, s, (const bf16_t*)x, (const bf16_t*)w_up, dense, (bf16_t*)a, M, experts, rows, K, 0);
  else
    hipLaunchKernelGGL((deep ? moe_up_kernel<false, 2> : moe_up_kernel<false, 1>), up, block, 0, s, (const bf16_t*)x, (const bf16_t*)w_up, dense, (bf16_t*)a, M, experts, rows, K, kind);
  const bool deep_down = dg_deep(M, ff / parts, N / 16 * parts) && ff / parts % (DG_WAVES * 128) == 0;
  hipLaunchKernelGGL(deep_down ? moe_down_kernel<2> : moe_down_kernel<1>, dim3(N / 16, parts), block, 0, s, (const bf16_t*)a, (const bf16_t*)w_down, dense, y, M, experts, ff, N, accumulate,
                     (const bf16_t*)w_shared, (const bf16_t*)a_shared, gate, size);
  TP_CHECK_LAUNCH("moe_few");
  return 0;
}

// bfloat16 rows [M, K] -> [K / 8, M, 8]
__global__ void block_rows_kernel(const u32x4_t* __restrict__ x, u32x4_t* __restrict__ out, int M, int pieces) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M * pieces) return;
  const int m = i / pieces, p = i % pieces;
  out[(size_t)p * M + m] = x[i];
}

extern "C" int tp_block_rows(const void* x, void* out, int M, int K, hipStream_t s) {
  TP_REQUIRE(M > 0 && K > 0 && K % 8 == 0 && (long)M * (K / 8) < 0x7fffffffL && (((uintptr_t)x | (uintptr_t)out) & 15) == 0, "block_rows: bad rows");
  const int total = M * (K / 8);
  hipLaunchKernelGGL(block_rows_kernel, dim3((total + 255) / 256), dim3(256), 0, s, (const u32x4_t*)x, (u32x4_t*)out, M, K / 8);
  TP_CHECK_LAUNCH("block_rows");
  return 0;
}
