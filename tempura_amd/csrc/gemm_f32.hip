// Float32 products, out[M, N] (+)= x[M, K] * w[N, K]^T, every multiply-add in float32: 16-byte loads, K % 4 == 0.
//
// Up to 16 rows (gemm_f32_rows_kernel) the weight matrix is read once and bounds the product: a block of four waves owns a few
// weight rows and cuts K between its waves, a lane takes four neighbouring k of every weight row at a time (a wave's load is
// 1 KB of one row) and multiplies them with all rows of x; lanes and then waves are added in a fixed tree.  Two rows: 3,072 x 8,192 18.8 us (5.4 TB/s),
// 16,384 x 3,072 33 us (6.1), 128,256 x 3,072 234 us (6.7).  The general kernel, which stages x through LDS between barriers and has
// one weight element a lane in flight, takes 263, 124 (5,120 x 3,072; here 12.6) and 569 us.  At 16 rows the multiply-adds and the
// reads of x bound it (16,384 x 3,072: 56 us), still a quarter less than the blocks of 64 rows below.
//
// From 17 rows on the matrix cores multiply.  gemm_f32_split_kernel cuts the operands into bfloat16 pieces that hold all of their 24 bits and
// makes six bfloat16 products of every float32 one, at sixteen times the float32 rate: 611 rows by 3,072 x 3,072 126 -> 79 us, 16,384 x
// 3,072 573 -> 377 (104 -> 163 TFLOP/s), 3,072 x 8,192 321 -> 192; 2,048 rows by 16,384 x 3,072 1,649 -> 1,097.  The clock, 1.8 to 2.0 GHz while the
// matrix cores work, and the LDS reads and writes that share a phase with them bound it: 2,800 cycles a stage of a block for 1,536 of MFMAs.
// gemm_f32_mfma_kernel (operands as they are, 157 TFLOP/s; one LDS read for four of them, so one pipeline of two LDS stages is
// enough) takes few rows and short sums, where a block of 128 leaves CUs without work.
#include "common.h"
#include "column_sum.h"

#include <type_traits>

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

// ---- the same in bfloat16 pieces ------------------------------------------------------------------------------------------------
// x = h + m + l: h the upper half of x's bits, m what remains rounded to bfloat16, l the rest, which has no more than the eight bits that
// bfloat16 holds: nothing of an operand is lost.  Of the nine products of pieces the six largest are made; the three left out are below
// 2^-22 of x w together, and of either sign.  Products of two pieces are exact, sums are float32: against 64 bits, normal operands, K of 3,072,
// 2-norm of the error 1.1e-7 of the result's (gemm_f32_mfma_kernel 2.6e-7); operands over twelve orders of magnitude 0.9e-7 (1.7e-7), all positive
// 0.5e-7 (0.7e-7).
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

namespace {

// Eight neighbouring k of a row as the 16 bytes of each piece.  (The first piece is cut off rather than rounded, which takes no conversion; the
// second is rounded, so that the products left out have no common sign; what then remains is no more than eight bits.)
__device__ inline void split8(const f32x4 (&v)[2], u32x4 (&out)[3]) {
  float top = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) top = fmaxf(top, fabsf(v[i / 4][i % 4]));
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    const float x0 = v[i / 4][i % 4], x1 = v[i / 4][i % 4 + 1];
    const unsigned b0 = __float_as_uint(x0), b1 = __float_as_uint(x1);
    const f32x2 r = {x0 - __uint_as_float(b0 & 0xffff0000u), x1 - __uint_as_float(b1 & 0xffff0000u)};
    const unsigned mp = __builtin_bit_cast(unsigned, __builtin_convertvector(r, bf16x2));
    const float q0 = r[0] - __uint_as_float(mp << 16), q1 = r[1] - __uint_as_float(mp & 0xffff0000u);
    out[0][i / 2] = __builtin_amdgcn_perm(b1, b0, 0x07060302u);
    out[1][i / 2] = mp;
    out[2][i / 2] = __builtin_amdgcn_perm(__float_as_uint(q1), __float_as_uint(q0), 0x07060302u);
  }
  // Infinity in pieces: (1, 0, infinity), which a product with any finite pieces turns into what the whole value gives (an infinite first piece would
  // meet the zeros and the other signs among the other operand's pieces).  (A NaN's remainders are NaN as well.)
  if (top == __builtin_inff()) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float x = v[i / 4][i % 4];
      if (fabsf(x) != __builtin_inff()) continue;
      const unsigned piece[3] = {__float_as_uint(copysignf(1.f, x)), 0u, __float_as_uint(x)}, keep = i % 2 ? 0xffffu : 0xffff0000u;
#pragma unroll
      for (int q = 0; q < 3; ++q) out[q][i / 2] = (out[q][i / 2] & keep) | (i % 2 ? piece[q] : piece[q] >> 16);
    }
  }
}

}  // namespace

// A block of 128 x 128 results, eight waves: two groups of four (2 x 2, 64 x 64 each, tiles of 16 x 16) take K's stages in turn, each in
// LDS of its own.  While one group multiplies the other cuts its next stage into pieces and writes it, and at a barrier they change
// places: so the vector unit's share (six operations an element) runs beside the matrix cores'.
// v_mfma_f32_16x16x32_bf16 takes eight neighbouring k of row lane % 16 from lane / 16 * 8 on: a stage holds every 16 rows of a piece as
// those 64 x 16 bytes, the sixteen of each eight k turned by four places from the one before: the four threads that write a row's eight k then meet
// four different groups of banks (all in one: 3,200 cycles a stage instead of 2,800).
// splits > 1: blockIdx.y takes a run of K's stages and writes its sums to part [splits, M, N].
template <bool ACC>
__global__ __launch_bounds__(512) void gemm_f32_split_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                             float* __restrict__ out, float* __restrict__ part, int M, int N, int K,
                                                             int row_tiles, int tiles) {
  constexpr int T = 128, R = 4;
  __shared__ u32x4 lds[2][2][3][T / 16][64];           // group, operand, piece
  // XCD j (blocks go to the XCDs in turn) takes the j-th eighth of the tiles, row tiles fastest: the blocks that share weight
  // rows then share an L2
  const int per = (tiles + 7) / 8;
  const int tile = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if ((int)(blockIdx.x / 8) >= per || tile >= tiles) return;
  const int m0 = tile % row_tiles * T, n0 = tile / row_tiles * T;
  const int tid = threadIdx.x % 256, lane = tid % TP_WAVE, wave = __builtin_amdgcn_readfirstlane(tid / TP_WAVE);
  const int group = __builtin_amdgcn_readfirstlane(threadIdx.x / 256);
  const int wm = wave / 2 * R, wn = wave % 2 * R;      // the wave's first tile
  const int place = lane / 16 * 16 + (lane + lane / 16 * 4) % 16;
  const int stages = (K + FM_K - 1) / FM_K, sper = (stages + gridDim.y - 1) / gridDim.y;
  const int s0 = blockIdx.y * sper, s1 = min(stages, s0 + sper), turns = (s1 - s0 + 1) / 2;

  const int lr = tid / 4, lk = tid % 4 * 8;            // loader: 64 rows a pass, four threads a row
  f32x4 gx[2][2], gw[2][2];
  // (buffers that begin at the block's first rows: 32-bit offsets, and what lies outside, as k past the last is made to, reads as zero)
  const auto xb = __builtin_amdgcn_make_buffer_rsrc((void*)(x + (size_t)m0 * K), 0, 0x7ffffff0, 0x00020000);
  const auto wb = __builtin_amdgcn_make_buffer_rsrc((void*)(w + (size_t)n0 * K), 0, 0x7ffffff0, 0x00020000);
  unsigned ox[2], ow[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    ox[i] = (unsigned)min(lr + 64 * i, M - 1 - m0) * (unsigned)K * 4u + lk * 4;
    ow[i] = (unsigned)min(lr + 64 * i, N - 1 - n0) * (unsigned)K * 4u + lk * 4;
  }
  auto fetch = [&](int s) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const bool in = s < s1 && s * FM_K + lk + 4 * j < K;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        gx[i][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(xb, in ? ox[i] + s * (FM_K * 4) + 16 * j : 0xffffff00u, 0, 0));
        gw[i][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(wb, in ? ow[i] + s * (FM_K * 4) + 16 * j : 0xffffff00u, 0, 0));
      }
    }
  };
  auto stage = [&]() {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = lr + 64 * i, at = lk * 2 + (r + lk / 2) % 16;
      u32x4 p[3];
      split8(gx[i], p);
#pragma unroll
      for (int q = 0; q < 3; ++q) lds[group][0][q][r / 16][at] = p[q];
      split8(gw[i], p);
#pragma unroll
      for (int q = 0; q < 3; ++q) lds[group][1][q][r / 16][at] = p[q];
    }
  };
  // (this wave's LDS accesses done, and no access moved across by the compiler; its loads from memory may still be on their way)
  auto meet = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  f32x4 acc[R][R];
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int j = 0; j < R; ++j) acc[i][j] = (f32x4)(0.f);
  fetch(s0 + group);
  if (group == 1) meet();
  for (int t = 0; t < turns; ++t) {
    stage();
    meet();
    fetch(s0 + 2 * (t + 1) + group);
    // A stage's six products of a tile are summed from zero, the smallest first, and the sum is added to the tile's by the vector unit,
    // rounded to nearest (the matrix cores cut a sum's last bits off).  Two rows of tiles at a time.
    u32x4 c[3][R];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      u32x4 a[3][2];
#pragma unroll
      for (int z = 0; z < 3; ++z) {
        constexpr int QA[3] = {2, 0, 1}, QC[3] = {0, 2, 1};
#pragma unroll
        for (int i = 0; i < 2; ++i) a[QA[z]][i] = lds[group][0][QA[z]][wm + half * 2 + i][place];
        if (half == 0)
#pragma unroll
          for (int j = 0; j < R; ++j) c[QC[z]][j] = lds[group][1][QC[z]][wn + j][place];
      }
      f32x4 t[2][R];
#pragma unroll
      for (int p = 0; p < 6; ++p) {
        constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PC[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < R; ++j)
            t[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[PA[p]][i]), __builtin_bit_cast(bf16x8, c[PC[p]][j]),
                                                              p == 0 ? (f32x4)(0.f) : t[i][j], 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < R; ++j) acc[half * 2 + i][j] += t[i][j];
    }
    // The order of the instructions: the LDS reads of the first two products, then the others one by one between MFMAs.
    __builtin_amdgcn_sched_group_barrier(0x100, 12, 0);
#pragma unroll
    for (int z = 0; z < 12; ++z) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 84, 0);
    meet();
  }
  if (group == 0) meet();
  // each group gives half of its rows of tiles to the other and adds the other's sums to its own half
  f32x4* given = (f32x4*)lds + wave * (2 * 2 * R * 64);
  auto close = [&](auto mine_) {
    constexpr int mine = decltype(mine_)::value, other = 2 - mine;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < R; ++j) given[((other + i) * R + j) * 64 + lane] = acc[other + i][j];
    meet();
    // a lane holds column lane % 16 and rows lane / 16 * 4 + e of a 16 x 16 tile
    const bool partial = gridDim.y > 1;
    float* o0 = partial ? part + (size_t)blockIdx.y * M * N : out;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const int n = n0 + (wn + j) * 16 + lane % 16;
        const f32x4 sum = acc[mine + i][j] + given[((mine + i) * R + j) * 64 + lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int m = m0 + (wm + mine + i) * 16 + lane / 16 * 4 + e;
          if (m < M && n < N) {
            float* o = o0 + (size_t)m * N + n;
            *o = ACC && !partial ? *o + sum[e] : sum[e];
          }
        }
      }
  };
  if (group == 0) close(std::integral_constant<int, 0>{}); else close(std::integral_constant<int, 2>{});
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

static void launch_split(const float* x, const float* w, float* out, float* part, bool acc, int M, int N, int K, int splits, hipStream_t s) {
  const int row_tiles = (M + 127) / 128, tiles = row_tiles * ((N + 127) / 128);
  const dim3 grid((tiles + 7) / 8 * 8, splits);
  if (acc)
    hipLaunchKernelGGL((gemm_f32_split_kernel<true>), grid, dim3(512), 0, s, x, w, out, part, M, N, K, row_tiles, tiles);
  else
    hipLaunchKernelGGL((gemm_f32_split_kernel<false>), grid, dim3(512), 0, s, x, w, out, part, M, N, K, row_tiles, tiles);
}

// How the product of more than 16 rows is cut: K in up to eight parts of at least 256, and the block's side.  The parts, which a result's
// bits depend on, and the kernel are chosen for rows counted in blocks of 128 (up to 64: 64), so that a step whose rows are padded to the
// next power of two, or multiple of 128, is cut alike.
struct F32Plan {
  bool split;       // gemm_f32_split_kernel, blocks of 128
  int tile, splits;
};

static F32Plan f32_plan(int M, int N, int K, bool parts_ok) {
  F32Plan p = {false, 64, 1};
  const long rows = M <= 64 ? 64 : (long)(M + 127) / 128 * 128, cols = (N + 63) / 64;
  const int most = parts_ok ? 8 : 1;
  double best = 1e30;
  // In pieces, from 65 rows on, a K of 1,536 and 49,152 steps of K over all blocks (float32 blocks / pieces: 128 rows 2,048 x 2,048 19.7 / 19.4 us,
  // 2,048 x 3,072 26.5 / 25.8, 8,192 x 3,072 89 / 50; 300 rows 512 x 3,072 23.0 / 25.2, 1,024 rows of it 44.6 / 29.4; 64 rows, half a block, lose
  // everywhere: 16,384 x 3,072 89 / 117.  A shorter K gains from 100,000 steps on, 1.2 to 1.5 times, and is left: no configuration here has one).
  // The time is rounds of 256 blocks at 1.3 us a stage of a block, and the parts written, read and added at 3 TB/s and 5 us (611 rows in 1 / 2 /
  // 4 parts: 5,120 x 3,072 126 / 142 / 152 us, 3,072 x 3,072 125 / 79 / 84, 16,384 x 3,072 387 / 377 / 400, 3,072 x 8,192 315 / 192 / 191).
  const long blocks = (rows + 127) / 128 * ((N + 127) / 128);
  if (rows > 64 && K >= 1536 && blocks * K >= 49152 && (size_t)K * 512 < ((size_t)1 << 31)) {
    p.split = true;
    p.tile = 128;
    for (int q = 1; q <= most && (q == 1 || K / q >= 256); ++q) {
      const double cost = (double)((blocks * q + 255) / 256) / q * (K / 32.0) * 1.3 + (q > 1 ? 5.0 + (q + 2.0) * rows * N * 4.0 / 3e6 : 0.0);
      if (cost < best) best = cost, p.splits = q;
    }
    return p;
  }
  // In float32: the matrix cores bound it, so the time is the work of the fullest CU: rounds of 256 blocks times a block's results and its
  // share of K; every part costs 3 % for writing and adding its sums.  The block (which a result's bits do not depend on) is chosen for the
  // rows there are.  3,072 x 3,072 at 64 rows in 1 / 4 / 5 parts: 41 / 25.7 / 23 us.
  for (int q = 1; q <= most && (q == 1 || K / q >= 256); ++q) {
    const double cost = (double)((rows / 64 * cols * q + 255) / 256) / q * (1.0 + 0.03 * (q - 1));
    if (cost < best) best = cost, p.splits = q;
  }
  const long t128 = (long)(M + 127) / 128 * ((N + 127) / 128) * p.splits, t64 = (long)(M + 63) / 64 * cols * p.splits;
  if (4.0 * ((t128 + 255) / 256) <= 1.08 * ((t64 + 255) / 256)) p.tile = 128;
  return p;
}

// Floats of scratch that the product uses for parts of K (0: none).
extern "C" size_t tp_linear_f32_scratch(int M, int N, int K) {
  if (M <= 16 || N <= 0 || K <= 0) return 0;
  const F32Plan p = f32_plan(M, N, K, true);
  return p.splits > 1 ? (size_t)p.splits * M * N : 0;
}

// The side of the blocks that the product takes with that scratch (0: it is one of few rows); for tests that mean a certain one.
extern "C" int tp_linear_f32_block(int M, int N, int K) {
  if (M <= 16 || N <= 0 || K <= 0) return 0;
  return f32_plan(M, N, K, true).tile;
}

// Takes a product whose rows are whole 16-byte pieces (K % 4 == 0, aligned operands); -1: not its own, the general kernel runs.
int tp_linear_f32(const float* x, const float* w, float* out, int accumulate, int M, int N, int K, float* scratch,
                  size_t scratch_floats, hipStream_t s) {
  if (K % 4 != 0 || ((uintptr_t)x | (uintptr_t)w) % 16 != 0) return -1;
  const bool acc = accumulate != 0;
  if (M <= 16)
    launch_rows(x, w, out, acc, M, N, K, nullptr, 0.f, false, s);
  else {
    F32Plan p = f32_plan(M, N, K, true);
    if (p.splits > 1 && (scratch == nullptr || scratch_floats < (size_t)p.splits * M * N)) p = f32_plan(M, N, K, false);
    if (p.split)
      launch_split(x, w, out, scratch, acc, M, N, K, p.splits, s);
    else if (p.tile == 128)
      launch_mfma<128>(x, w, out, scratch, acc, M, N, K, p.splits, s);
    else
      launch_mfma<64>(x, w, out, scratch, acc, M, N, K, p.splits, s);
    if (p.splits > 1) {
      const size_t count = (size_t)M * N;
      const dim3 grid((unsigned)((count + 255) / 256));
      if (acc)
        hipLaunchKernelGGL((gemm_f32_parts_kernel<true>), grid, dim3(256), 0, s, scratch, out, count, p.splits);
      else
        hipLaunchKernelGGL((gemm_f32_parts_kernel<false>), grid, dim3(256), 0, s, scratch, out, count, p.splits);
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
