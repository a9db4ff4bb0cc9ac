// Float32 products, out[M, N] (+)= x[M, K] * w[N, K]^T, every multiply-add in float32: 16-byte loads, K % 4 == 0.
//
// Up to 16 rows (gemm_f32_rows_kernel) the weight matrix is read once and bounds the product: a block of four waves owns a few
// weight rows and cuts K between its waves, a lane takes four neighbouring k of every weight row at a time (a wave's load is
// 1 KB of one row) and multiplies them with all rows of x; lanes and then waves are added in a fixed tree.  Two rows: 3,072 x 8,192 18.8 us (5.4 TB/s),
// 16,384 x 3,072 33 us (6.1), 128,256 x 3,072 234 us (6.7).  The general kernel, which stages x through LDS between barriers and has
// one weight element a lane in flight, takes 263, 124 (5,120 x 3,072; here 12.6) and 569 us.  At 16 rows the multiply-adds and the
// reads of x bound it (16,384 x 3,072: 56 us), still a quarter less than the blocks of 64 rows below.
//
// From 17 rows on (gemm_f32_mfma_kernel) the matrix cores take float32 operands at 157 TFLOP/s, twice the rate of the vector unit
// without packed instructions, and need one LDS read for four of them, so one pipeline of two LDS stages is enough.  611 rows:
// 3,072 x 3,072 119 us, 16,384 x 3,072 594 us (97 and 104 TFLOP/s; the general kernel 477 and 2,060 us); 2,048 rows of the latter 1,650 us (125).
#include "common.h"
#include "column_sum.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// ---- up to 16 rows --------------------------------------------------------------------------------------------------------------
#define FR_WAVES 4

// MC: rows of the block's registers (M <= MC), C: weight rows a block owns.
// NORM: x holds rows before their root-mean-square norm (weight norm_w): the block multiplies them with the norm's weight as it reads
// them, adds their squares beside the products (it sees every row whole) and scales its sums.
// GATE: N is the columns of each half of w [gate; up], and out is silu(gate) * up: the block owns C / 2 rows of each half.
// Decode steps of two rows are a chain of small kernels beside the products, each 5 us of launch and dependent reads, and this work
// costs the products, which wait for memory, little.  Two rows in a captured chain, separate kernels / here: 16,384 x 3,072 with norm
// and gate 36.3 / 34.1 us, 5,120 x 3,072 with the norm 15.4 / 13.5; 16 rows 73.9 / 63.2 and 35.3 / 27.3 (with eight weight rows a block,
// which halve what is read of x: without norm and gate 68.2 -> 56.3 and 28.9 -> 24.7; eight rows of x gain at 16,384 weight rows, 48 ->
// 40, and lose at 3,072 x 8,192, 24 -> 28: they stay at four).
template <int MC, int C, bool ACC, bool NORM, bool GATE>
__global__ __launch_bounds__(256) void gemm_f32_rows_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                            float* __restrict__ out, int M, int N, int K,
                                                            const float* __restrict__ norm_w, float eps) {
  constexpr int OWN = GATE ? C / 2 : C;                // columns of the result a block makes
  __shared__ float part[FR_WAVES][MC * C];
  __shared__ float squares[FR_WAVES][NORM ? MC : 1];
  const int lane = threadIdx.x % TP_WAVE, wave = threadIdx.x / TP_WAVE;
  const int n0 = blockIdx.x * OWN;
  // K in steps of 256 (a wave's load); the steps are dealt to the waves in runs
  const int steps = (K + 255) / 256, per = (steps + FR_WAVES - 1) / FR_WAVES;
  const int s0 = wave * per, s1 = min(steps, s0 + per);
  float acc[C * MC];
#pragma unroll
  for (int i = 0; i < C * MC; ++i) acc[i] = 0.f;
  const float* wr[C];
#pragma unroll
  for (int c = 0; c < C; ++c) wr[c] = w + ((size_t)min(n0 + c % OWN, N - 1) + (GATE && c >= OWN ? N : 0)) * K;
  float ss[NORM ? MC : 1];
#pragma unroll
  for (int m = 0; m < (NORM ? MC : 1); ++m) ss[m] = 0.f;
  f32x4 nw[C];
  auto fetch = [&](int s) {
    const int k = s * 256 + lane * 4;
    const bool in = s < s1 && k < K;
#pragma unroll
    for (int c = 0; c < C; ++c) nw[c] = in ? __builtin_nontemporal_load((const f32x4*)(wr[c] + k)) : (f32x4)(0.f);
  };
  fetch(s0);
  for (int s = s0; s < s1; ++s) {
    f32x4 cw[C];
#pragma unroll
    for (int c = 0; c < C; ++c) cw[c] = nw[c];
    fetch(s + 1);
    const int k = s * 256 + lane * 4;
    if (k < K) {
      f32x4 wn = (f32x4)(1.f);
      if constexpr (NORM) wn = *(const f32x4*)(norm_w + k);
#pragma unroll
      for (int m = 0; m < MC; ++m) {
        f32x4 xv = *(const f32x4*)(x + (size_t)min(m, M - 1) * K + k);
        if constexpr (NORM) {
#pragma unroll
          for (int j = 0; j < 4; ++j) ss[m] = fmaf(xv[j], xv[j], ss[m]);
          xv *= wn;
        }
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[c * MC + m] = fmaf(cw[c][j], xv[j], acc[c * MC + m]);
      }
    }
  }
  constexpr int NV = C * MC > 64 ? 64 : C * MC;
#pragma unroll
  for (int g = 0; g < C * MC / NV; ++g) {
    float v[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = acc[g * NV + i];
    const float t = lanes_transpose_sum<NV>(v, lane);
    if (lane % (TP_WAVE / NV) == 0) part[wave][g * NV + lane / (TP_WAVE / NV)] = t;
  }
  if constexpr (NORM) {
    const float t = lanes_transpose_sum<MC>(ss, lane);
    if (lane % (TP_WAVE / MC) == 0) squares[wave][lane / (TP_WAVE / MC)] = t;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < OWN * MC; i += 256) {
    const int c = i % OWN, m = i / OWN, n = n0 + c;
    if (m >= M || n >= N) continue;
    float rstd = 1.f;
    if constexpr (NORM) {
      float t = squares[0][m];
#pragma unroll
      for (int v = 1; v < FR_WAVES; ++v) t += squares[v][m];
      rstd = 1.0f / sqrtf(t / (float)K + eps);
    }
    auto sum_of = [&](int r) {
      float t = part[0][r * MC + m];
#pragma unroll
      for (int v = 1; v < FR_WAVES; ++v) t += part[v][r * MC + m];
      return NORM ? t * rstd : t;
    };
    float t = sum_of(c);
    if constexpr (GATE) t = t / (1.0f + expf(-t)) * sum_of(OWN + c);
    float* o = out + (size_t)m * N + n;
    *o = ACC ? *o + t : t;
  }
}

// ---- from 17 rows on --------------------------------------------------------------------------------------------------------------
#define FM_K 32           // K of a stage
#define FM_LD (FM_K + 4)  // floats of a row in LDS: rows four banks apart, so that eight lanes' 16-byte reads cover all banks

// A block of T x T results, four waves of T/2 x T/2.  v_mfma_f32_32x32x2_f32 takes k = 0 from lanes 0..31 and k = 1 from lanes
// 32..63; a lane reads four neighbouring k at once and feeds them to four instructions, so instruction j of a run of eight k
// multiplies k = j and k = 4 + j.
// splits > 1: blockIdx.y takes a run of K's stages and writes its sums to part [splits, M, N].
template <int T, bool ACC>
__global__ __launch_bounds__(256, 2) void gemm_f32_mfma_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                            float* __restrict__ out, float* __restrict__ part, int M, int N, int K,
                                                            int row_tiles, int tiles) {
  constexpr int W = T / 2, R = W / 32;                 // a wave's side, 32 x 32 tiles a side
  constexpr int LOADS = T * FM_K / 4 / 256;            // 16-byte loads a thread and operand
  __shared__ float xs[2][T * FM_LD], ws[2][T * FM_LD];
  // XCD j (blocks go to the XCDs in turn) takes the j-th eighth of the tiles, row tiles fastest: the blocks that share weight
  // rows then share an L2
  const int per = (tiles + 7) / 8;
  const int tile = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if ((int)(blockIdx.x / 8) >= per || tile >= tiles) return;
  const int m0 = tile % row_tiles * T, n0 = tile / row_tiles * T;
  const int tid = threadIdx.x, lane = tid % TP_WAVE, wave = tid / TP_WAVE;
  const int wm = wave / 2 * W, wn = wave % 2 * W;
  const int stages = (K + FM_K - 1) / FM_K, sper = (stages + gridDim.y - 1) / gridDim.y;
  const int s0 = blockIdx.y * sper, s1 = min(stages, s0 + sper);

  const int lr = tid / 8, lk = tid % 8 * 4;            // loader: 32 rows a pass, eight threads a row
  f32x4 gx[LOADS], gw[LOADS];
  auto fetch = [&](int s) {
    const int k = s * FM_K + lk;
    const bool in = k < K;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int r = lr + 32 * i;
      gx[i] = in ? *(const f32x4*)(x + (size_t)min(m0 + r, M - 1) * K + k) : (f32x4)(0.f);
      gw[i] = in ? *(const f32x4*)(w + (size_t)min(n0 + r, N - 1) * K + k) : (f32x4)(0.f);
    }
  };
  auto stage = [&](int b) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      *(f32x4*)&xs[b][(lr + 32 * i) * FM_LD + lk] = gx[i];
      *(f32x4*)&ws[b][(lr + 32 * i) * FM_LD + lk] = gw[i];
    }
  };
  // (two sums a result, over alternate runs of eight k: shorter chains of roundings than one sum in ascending order)
  f32x16 acc[2][R][R];
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int j = 0; j < R; ++j) acc[0][i][j] = acc[1][i][j] = (f32x16)(0.f);
  if (s0 < s1) {
    fetch(s0);
    stage(0);
  }
  __syncthreads();
  for (int s = s0; s < s1; ++s) {
    const int b = (s - s0) & 1;
    if (s + 1 < s1) fetch(s + 1);
#pragma unroll
    for (int kk = 0; kk < FM_K; kk += 8) {
      f32x4 a[R], c[R];
      const int k = kk + lane / 32 * 4;
#pragma unroll
      for (int i = 0; i < R; ++i) {
        a[i] = *(const f32x4*)&xs[b][(wm + i * 32 + lane % 32) * FM_LD + k];
        c[i] = *(const f32x4*)&ws[b][(wn + i * 32 + lane % 32) * FM_LD + k];
      }
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
          for (int j = 0; j < R; ++j)
            acc[kk / 8 % 2][i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][q], c[j][q], acc[kk / 8 % 2][i][j], 0, 0, 0);
    }
    if (s + 1 < s1) stage(b ^ 1);
    __syncthreads();
  }
  // a lane holds column lane % 32 and rows 8 (e / 4) + 4 (lane / 32) + e % 4 of a 32 x 32 tile
  const bool partial = gridDim.y > 1;
  float* o0 = partial ? part + (size_t)blockIdx.y * M * N : out;
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int n = n0 + wn + j * 32 + lane % 32;
      const f32x16 sum = acc[0][i][j] + acc[1][i][j];
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = m0 + wm + i * 32 + 8 * (e / 4) + 4 * (lane / 32) + e % 4;
        if (m < M && n < N) {
          float* o = o0 + (size_t)m * N + n;
          *o = ACC && !partial ? *o + sum[e] : sum[e];
        }
      }
    }
}

// out (+)= the parts in ascending order.
template <bool ACC>
__global__ __launch_bounds__(256) void gemm_f32_parts_kernel(const float* __restrict__ part, float* __restrict__ out, size_t count, int splits) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= count) return;
  float t = part[i];
  for (int s = 1; s < splits; ++s) t += part[(size_t)s * count + i];
  out[i] = ACC ? out[i] + t : t;
}

template <int MC, int C>
static void launch_rows(const float* x, const float* w, float* out, bool acc, int M, int N, int K, const float* norm_w, float eps, bool gate,
                        hipStream_t s) {
  const int own = gate ? C / 2 : C;
  const dim3 grid((N + own - 1) / own);
#define FR_LAUNCH(ACC_, NORM_, GATE_) \
  hipLaunchKernelGGL((gemm_f32_rows_kernel<MC, C, ACC_, NORM_, GATE_>), grid, dim3(256), 0, s, x, w, out, M, N, K, norm_w, eps)
  if (norm_w != nullptr && gate) FR_LAUNCH(false, true, true);
  else if (norm_w != nullptr) FR_LAUNCH(false, true, false);
  else if (gate) FR_LAUNCH(false, false, true);
  else if (acc) FR_LAUNCH(true, false, false);
  else FR_LAUNCH(false, false, false);
#undef FR_LAUNCH
}

static void launch_rows(const float* x, const float* w, float* out, bool acc, int M, int N, int K, const float* norm_w, float eps, bool gate,
                        hipStream_t s) {
  if (M == 1)
    launch_rows<1, 4>(x, w, out, acc, M, N, K, norm_w, eps, gate, s);
  else if (M == 2)
    launch_rows<2, 4>(x, w, out, acc, M, N, K, norm_w, eps, gate, s);
  else if (M <= 4)
    launch_rows<4, 4>(x, w, out, acc, M, N, K, norm_w, eps, gate, s);
  else if (M <= 8)
    launch_rows<8, 4>(x, w, out, acc, M, N, K, norm_w, eps, gate, s);
  else
    launch_rows<16, 8>(x, w, out, acc, M, N, K, norm_w, eps, gate, s);
}

template <int T>
static void launch_mfma(const float* x, const float* w, float* out, float* part, bool acc, int M, int N, int K, int splits, hipStream_t s) {
  const int row_tiles = (M + T - 1) / T, tiles = row_tiles * ((N + T - 1) / T);
  const dim3 grid((tiles + 7) / 8 * 8, splits);
  if (acc)
    hipLaunchKernelGGL((gemm_f32_mfma_kernel<T, true>), grid, dim3(256), 0, s, x, w, out, part, M, N, K, row_tiles, tiles);
  else
    hipLaunchKernelGGL((gemm_f32_mfma_kernel<T, false>), grid, dim3(256), 0, s, x, w, out, part, M, N, K, row_tiles, tiles);
}

// How the product of more than 16 rows is cut: blocks of 128 or 64 a side, K in up to eight parts.  The matrix cores bound it, so
// the time is the work of the fullest CU: rounds of 256 blocks times a block's results and its share of K; every part costs 3 % for
// writing and adding its sums and keeps 256 of K.  The parts, which a result's bits depend on, are chosen for rows counted in
// blocks of 128 (up to 64: 64), so that a step whose rows are padded to the next power of two, or multiple of 128, is cut alike;
// the block (which they do not depend on) for the rows there are.  3,072 x 3,072 at 64 rows in 1 / 4 / 5 parts: 41 / 25.7 / 23 us;
// 16,384 x 3,072 at 2,048 rows in blocks of 128 / 64: 1,650 / 1,790 us, 3,072 x 3,072 there 429 / 359 us (one and a half rounds of
// the large blocks).
static void f32_plan(int M, int N, int K, bool parts_ok, int* tile, int* splits) {
  const long rows = M <= 64 ? 64 : (long)(M + 127) / 128 * 128, cols = (N + 63) / 64;
  *splits = 1;
  double best = 1e30;
  for (int p = 1; p <= (parts_ok ? 8 : 1) && (p == 1 || K / p >= 256); ++p) {
    const double cost = (double)((rows / 64 * cols * p + 255) / 256) / p * (1.0 + 0.03 * (p - 1));
    if (cost < best) best = cost, *splits = p;
  }
  const long t128 = (long)(M + 127) / 128 * ((N + 127) / 128) * *splits, t64 = (long)(M + 63) / 64 * cols * *splits;
  *tile = 4.0 * ((t128 + 255) / 256) <= 1.08 * ((t64 + 255) / 256) ? 128 : 64;
}

// Floats of scratch that the product uses for parts of K (0: none).
extern "C" size_t tp_linear_f32_scratch(int M, int N, int K) {
  if (M <= 16 || N <= 0 || K <= 0) return 0;
  int tile, splits;
  f32_plan(M, N, K, true, &tile, &splits);
  return splits > 1 ? (size_t)splits * M * N : 0;
}

// The side of the blocks that the product takes with that scratch (0: it is one of few rows); for tests that mean a certain one.
extern "C" int tp_linear_f32_block(int M, int N, int K) {
  if (M <= 16 || N <= 0 || K <= 0) return 0;
  int tile, splits;
  f32_plan(M, N, K, true, &tile, &splits);
  return tile;
}

// Takes a product whose rows are whole 16-byte pieces (K % 4 == 0, aligned operands); -1: not its own, the general kernel runs.
int tp_linear_f32(const float* x, const float* w, float* out, int accumulate, int M, int N, int K, float* scratch,
                  size_t scratch_floats, hipStream_t s) {
  if (K % 4 != 0 || ((uintptr_t)x | (uintptr_t)w) % 16 != 0) return -1;
  const bool acc = accumulate != 0;
  if (M <= 16)
    launch_rows(x, w, out, acc, M, N, K, nullptr, 0.f, false, s);
  else {
    int tile, splits;
    f32_plan(M, N, K, true, &tile, &splits);
    if (splits > 1 && (scratch == nullptr || scratch_floats < (size_t)splits * M * N)) f32_plan(M, N, K, false, &tile, &splits);
    if (tile == 128)
      launch_mfma<128>(x, w, out, scratch, acc, M, N, K, splits, s);
    else
      launch_mfma<64>(x, w, out, scratch, acc, M, N, K, splits, s);
    if (splits > 1) {
      const size_t count = (size_t)M * N;
      const dim3 grid((unsigned)((count + 255) / 256));
      if (acc)
        hipLaunchKernelGGL((gemm_f32_parts_kernel<true>), grid, dim3(256), 0, s, scratch, out, count, splits);
      else
        hipLaunchKernelGGL((gemm_f32_parts_kernel<false>), grid, dim3(256), 0, s, scratch, out, count, splits);
    }
  }
  TP_CHECK_LAUNCH("linear (float32)");
  return 0;
}

// A product of at most 16 rows with what stands around it: x [M, K] before its norm (norm_w [K], eps; null: as it is); gate != 0: w [2 N, K] holds gate rows and then up rows, and out [M, N] is silu(gate) * up.
extern "C" int tp_linear_f32_rows(const float* x, const float* w, float* out, int M, int N, int K, const float* norm_w, float eps, int gate,
                                  hipStream_t s) {
  TP_REQUIRE(M >= 0 && M <= 16 && N > 0 && K > 0 && K % 4 == 0, "linear_f32_rows: bad sizes (%d x %d x %d)", M, N, K);
  TP_REQUIRE((((uintptr_t)x | (uintptr_t)w | (uintptr_t)norm_w) & 15) == 0, "linear_f32_rows: misaligned operand");
  if (M == 0) return 0;
  launch_rows(x, w, out, false, M, N, K, norm_w, eps, gate != 0, s);
  TP_CHECK_LAUNCH("linear_f32_rows");
  return 0;
}
