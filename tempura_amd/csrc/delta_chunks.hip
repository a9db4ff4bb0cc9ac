// The gated delta rule over long runs, 16 tokens at a time on the matrix cores (v_mfma_f32_16x16x4_f32), for key sizes of 64 and 128 and
// value sizes of a multiple of 16; delta.hip has the recurrence, and the chain of single tokens that short runs and other sizes take.
//
// Within 16 tokens, with G_t the product of the decays up to token t and S the state before them, the rule is a small linear system:
//   A[t, s] = sum_c k_t k_s (G_t / G_s)  (s < t),  B[t, s] the same with q_t (s <= t),  T = (I + diag(beta) A)^-1 diag(beta)
//   U = T (V - K~ S)  with K~_t = G_t k_t;   o = Q~ S + B U  with Q~_t = G_t q_t;   S <- G_16 S + K^T U  with K^_s = (G_16 / G_s) k_s
// Everything but the products with S and U is independent of the state: delta_chunk_prep_kernel works it out for all groups of 16 side by
// side, a wave each, and leaves K~, Q~, K^, T and B in scratch; the ratios of decays are running products, never quotients, so
// nothing overflows.  delta_chunk_scan_kernel is the chain over the groups: a block of four waves owns 16 value columns of a head, a wave
// a quarter of the key channels in accumulators, which lie as the next product's operand wants them; the waves' parts of K~ S and Q~ S meet
// in LDS once a group.
//
// The rounding is held to that of the chain of single tokens: the products of decays that act on the state (G, K~, Q~, K^) run in float64,
// the sums A and B over the channels are added in float64 from the second level of their tree on, and a group's tokens lie so that every
// matrix-core product adds them in ascending order (DC_PLACE): the tokens nearest to a result, which strong decays leave as most of it,
// are added last, where a sum's roundings are few.  Root mean square error against float64 over that of the chain, runs of 112, 300 and
// 1,000 tokens: decays of 0 to 1 a token 0.91 (states 0.99), 0.5 to 1 0.93 (0.97), 0.8 to 1 0.96 (0.95), 0.9 to 1 0.94 (0.92), 0.99 to 1
// 0.82 (0.81).  (In float32 throughout, tokens in the order of the rows and U = T V - (T K~) S it was 1.03, 1.06, 1.08, 1.06 and 0.94;
// one run of 2,048 tokens then took 201 us, now 198, four of 451 tokens 92 and 93, with 32 heads eight of 256 160 and 177.)
//
// Runs of fewer than 64 tokens (DC_SHORT) go by the chain (delta_chain.h) in further blocks of the same two launches, so that a step's
// long and short runs take the time of the longer way and not of both.
//
// The chain of single tokens is bound by what a wave issues and waits for a token, 0.25 to 0.55 us; here a group of 16 takes 1.3 us (its
// products, a meeting in LDS and the update, each waiting for the one before).  16 heads of 128 x 128, all by single tokens / as here: one
// run of 128 tokens 37 / 28 us, 2,048 486 / 198; four runs of 451 tokens 162 / 93 (a third of it the first kernel); runs of 82, 327, 573 and
// 821 tokens 262 / 118; 700 tokens beside 31 single ones 1,327 / 85, 1,800 beside 63 3,412 / 190, beside 247 1,316 / 324; 200 beside ten of
// 63 105 / 87.  What loses is a run of hardly more than 64 tokens beside many that stay with the chain: 64 beside seven of 63 56 / 63, beside
// 100 single ones 70 / 88.
#include <math.h>

#include "common.h"
#include "column_sum.h"
#include "delta_chain.h"

typedef float f32x4_d __attribute__((ext_vector_type(4)));

#define DC_T 16      // tokens of a group
// Runs of up to this many tokens go by the chain of single tokens, whatever runs stand beside them: a request's bits do not depend on its
// neighbours.  (Alone the two ways meet at 64 tokens, several runs sooner.  16 heads of 128 x 128, single tokens / groups: one run of 48
// tokens 18 / 20 us, 64 22 / 21, 96 29 / 24; three of 48 22 / 24, 64 28 / 27; eight of 32 29 / 27, 64 49 / 36.  Eight heads of 64 x 64: one
// of 48 16 / 17, 64 19 / 18; 24 of 48 22 / 25, 64 28 / 28.)
#define DC_SHORT 63
#define DC_HEADS 4    // key heads a wave makes unit vectors of, for those runs

struct DeltaChunkArgs {
  DeltaArgs in;           // (its q and k as they come: a group makes unit vectors of its own)
  float* scratch;
  int requests;
  int first, groups;      // the groups that this launch takes, among those of all long runs one behind the other
  int blocks;             // that many blocks take groups; those behind them the runs of up to DC_SHORT tokens (all in the first launch)
};

// Where a token of the group lies among the rows and columns of the operands: instruction i of a product over the tokens takes element i
// of each lane, from lanes quad = 0 .. 3, so with token 4 i + quad at place 4 quad + i the instructions run through the tokens in order.
// (Its own inverse.)
#define DC_PLACE(t) (4 * ((t) % 4) + (t) / 4)

// floats of scratch for one group of one head: K~, Q~ [16, dim], K^ [dim, 16], G_16 [dim], T [16, 16], B [16, 16] without its diagonal,
// that [16]; tokens at their places
__host__ __device__ inline size_t dc_item_floats(int dim) { return (size_t)49 * dim + 528; }

// places of the sums: for s B(s, s), then A(t, s), B(t, s) of t = s + 1 .. 15
#define DC_B(t, s) (32 * (s) - (s) * (s) + 2 * ((t) - (s)))
#define DC_A(t, s) (DC_B(t, s) - 1)

// The groups of all long runs are numbered one behind the other, so that scratch and launches are sized by the step's tokens and not by
// its requests times their longest run; where a run's groups begin is read from the runs' bounds here, 64 of them at a time.
__device__ inline int dc_run_groups(const int* cu_seqlens, int r, int requests) {
  const int len = r < requests ? cu_seqlens[r + 1] - cu_seqlens[r] : 0;
  return len > DC_SHORT ? (len + DC_T - 1) / DC_T : 0;
}

__device__ inline int dc_first_group(const int* cu_seqlens, int r, int lane) {
  int sum = 0;
  for (int r0 = 0; r0 < r; r0 += TP_WAVE) {
    int v = dc_run_groups(cu_seqlens, r0 + lane, r);
#pragma unroll
    for (int d = TP_WAVE / 2; d > 0; d /= 2) v += __shfl_xor(v, d, TP_WAVE);
    sum += v;
  }
  return __builtin_amdgcn_readfirstlane(sum);
}

// The run that group i belongs to, and its number there; false: there are fewer groups.
__device__ inline bool dc_find_group(const int* cu_seqlens, int requests, int i, int lane, int& run, int& number) {
  for (int r0 = 0; r0 < requests; r0 += TP_WAVE) {
    const int own = dc_run_groups(cu_seqlens, r0 + lane, requests);
    int upto = own;
#pragma unroll
    for (int d = 1; d < TP_WAVE; d *= 2) {
      const int below = __shfl_up(upto, d, TP_WAVE);
      if (lane >= d) upto += below;
    }
    const unsigned long long behind = __ballot(upto > i);
    if (behind != 0) {
      const int at = __ffsll(behind) - 1;
      run = __builtin_amdgcn_readfirstlane(r0 + at);
      number = __builtin_amdgcn_readfirstlane(i - __shfl(upto - own, at, TP_WAVE));
      return true;
    }
    i -= __shfl(upto, TP_WAVE - 1, TP_WAVE);
  }
  return false;
}

// Whether token t belongs to a run that goes by groups (the same in every lane).
__device__ inline bool dc_in_long_run(const int* cu_seqlens, int requests, int t, int lane) {
  for (int r0 = 0; r0 < requests; r0 += TP_WAVE) {
    const int r = r0 + lane, a = r < requests ? cu_seqlens[r] : 0, b = r < requests ? cu_seqlens[r + 1] : 0;
    if (__any(a <= t && t < b)) return __any(a <= t && t < b && b - a > DC_SHORT);
  }
  return false;
}

// The sums over the lanes of a wave of 64 values, lane i the i-th's: lanes_transpose_sum's tree (distance 32 down to 1), in float64 behind
// its first level.  The two widest levels are the instructions that swap halves or odd rows with even ones.
__device__ inline float dc_sum64(const float (&v)[64], int lane) {
  double d[32];
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[i]), __float_as_uint(v[i + 32]), false, false);
    d[i] = (double)(__uint_as_float(r[0]) + __uint_as_float(r[1]));
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(d[i]), __double2loint(d[i + 16]), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(d[i]), __double2hiint(d[i + 16]), false, false);
    d[i] = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
  }
#pragma unroll
  for (int w = 8; w > 0; w /= 2) {
    const bool up = lane & w;
#pragma unroll
    for (int i = 0; i < w; ++i) {
      const double keep = up ? d[i + w] : d[i], send = up ? d[i] : d[i + w];
      d[i] = keep + __shfl_xor(send, w, TP_WAVE);
    }
  }
  return (float)d[0];
}

// (a recursion: every place of v is then known to the compiler, which keeps v in registers)
template <int S, int PER>
__device__ inline void dc_dots(const float (&q)[DC_T][PER], const float (&k)[DC_T][PER], const float (&gd)[DC_T][PER], float (&v)[64],
                               float* dots, int lane) {
  float w[PER];
#pragma unroll
  for (int p = 0; p < PER; ++p) w[p] = k[S][p];
#pragma unroll
  for (int t = S; t < DC_T; ++t) {
    float da = 0.f, db = 0.f;
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      if (t > S) w[p] *= gd[t][p];
      da = fmaf(w[p], k[t][p], da);
      db = fmaf(w[p], q[t][p], db);
    }
    if (t > S) {
      v[DC_A(t, S) % 64] = da;
      if (DC_A(t, S) % 64 == 63) dots[DC_A(t, S) - 63 + lane] = dc_sum64(v, lane);
    }
    v[DC_B(t, S) % 64] = db;
    if (DC_B(t, S) % 64 == 63) dots[DC_B(t, S) - 63 + lane] = dc_sum64(v, lane);
  }
  if constexpr (S + 1 < DC_T) dc_dots<S + 1, PER>(q, k, gd, v, dots, lane);
}

template <int PER>
__global__ __launch_bounds__(64) void delta_chunk_prep_kernel(DeltaChunkArgs c) {
  constexpr int K = 64 * PER;
  __shared__ float dots[256];
  __shared__ float bs[DC_T];
  const int lane = threadIdx.x;
  const DeltaArgs& a = c.in;
  if ((int)blockIdx.x >= c.blocks) {      // unit vectors of the chain's tokens, DC_HEADS key heads a wave
    const int parts = (a.kv_heads + DC_HEADS - 1) / DC_HEADS, i = blockIdx.x - c.blocks, t = i / parts, g0 = i % parts * DC_HEADS;
    if (dc_in_long_run(a.cu_seqlens, c.requests, t, lane)) return;
    for (int g = g0; g < min(g0 + DC_HEADS, a.kv_heads); ++g) delta_unit_rows(a, t, g, lane);
    return;
  }
  const int h = blockIdx.x % a.heads, at = blockIdx.x / a.heads;
  int r, number;
  if (!dc_find_group(a.cu_seqlens, c.requests, c.first + at, lane, r, number)) return;
  const int run0 = a.cu_seqlens[r], t0 = number * DC_T, len = min(DC_T, a.cu_seqlens[r + 1] - run0 - t0);
  const size_t row0 = (size_t)(run0 + t0);
  const int g = h / (a.heads / a.kv_heads);
  const float* qp = a.qkv + row0 * a.row_stride + (size_t)g * K;
  const float* kp = qp + (size_t)a.kv_heads * K;
  const float* gp = a.decay + (row0 * a.heads + h) * K;
  float q[DC_T][PER], k[DC_T][PER], gd[DC_T][PER];      // (channels lane + 64 p)
#pragma unroll
  for (int t = 0; t < DC_T; ++t)
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int ch = lane + 64 * p;
      const bool in = t < len;
      q[t][p] = in ? qp[(size_t)t * a.row_stride + ch] : 0.f;
      k[t][p] = in ? kp[(size_t)t * a.row_stride + ch] : 0.f;
      gd[t][p] = in ? gp[(size_t)t * a.heads * K + ch] : 1.f;
    }
  if (lane < DC_T) bs[lane] = lane < len ? 1.0f / (1.0f + expf(-a.proj[(row0 + lane) * a.proj_stride + a.beta_col0 + h])) : 0.f;
  // unit vectors: the 16 sums of squares of q and of k at once, lane 2 i the i-th
  {
    float sq[2 * DC_T];
#pragma unroll
    for (int t = 0; t < DC_T; ++t) {
      float x = 0.f, y = 0.f;
#pragma unroll
      for (int p = 0; p < PER; ++p) {
        x = fmaf(q[t][p], q[t][p], x);
        y = fmaf(k[t][p], k[t][p], y);
      }
      sq[t] = x;
      sq[DC_T + t] = y;
    }
    const float total = lanes_transpose_sum<2 * DC_T>(sq, lane);
    const float unit = (lane < 32 ? a.q_scale : 1.0f) / sqrtf(total + a.unit_eps);
#pragma unroll
    for (int t = 0; t < DC_T; ++t) {
      const float rq = __shfl(unit, 2 * t, TP_WAVE), rk = __shfl(unit, 2 * (DC_T + t), TP_WAVE);
#pragma unroll
      for (int p = 0; p < PER; ++p) {
        q[t][p] *= rq;
        k[t][p] *= rk;
      }
    }
  }
  // A and B, 64 of their sums over the channels at a time
  {
    float v[64];
    dc_dots<0, PER>(q, k, gd, v, dots, lane);
  }
  float* item = c.scratch + ((size_t)at * a.heads + h) * dc_item_floats(K);
  float *Kt = item, *Q = Kt + DC_T * K, *KT = Q + DC_T * K, *G = KT + DC_T * K, *T = G + K, *B = T + 256, *diag = B + 256;
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int ch = lane + 64 * p;
    double tail = 1.0;
    float kt[DC_T];
#pragma unroll
    for (int s = DC_T - 1; s >= 0; --s) {
      kt[DC_PLACE(s)] = (float)((double)k[s][p] * tail);
      tail *= (double)gd[s][p];
    }
    G[ch] = (float)tail;
#pragma unroll
    for (int s = 0; s < DC_T; s += 4) *(f32x4_d*)(KT + (size_t)ch * DC_T + s) = (f32x4_d){kt[s], kt[s + 1], kt[s + 2], kt[s + 3]};
    double head = 1.0;
#pragma unroll
    for (int t = 0; t < DC_T; ++t) {
      head *= (double)gd[t][p];
      Q[DC_PLACE(t) * K + ch] = (float)((double)q[t][p] * head);
      Kt[DC_PLACE(t) * K + ch] = (float)((double)k[t][p] * head);
    }
  }
  __syncthreads();
  // lane j: column j of T
  if (lane < DC_T) {
    float col[DC_T];
#pragma unroll
    for (int t = 0; t < DC_T; ++t) {
      float sum = 0.f;
#pragma unroll
      for (int s = 0; s < t; ++s) sum = fmaf(dots[DC_A(t, s)], col[s], sum);
      col[t] = t == lane ? bs[t] : t > lane ? -bs[t] * sum : 0.f;
      T[DC_PLACE(t) * DC_T + DC_PLACE(lane)] = col[t];
    }
    diag[DC_PLACE(lane)] = dots[DC_B(lane, lane)];
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = lane + 64 * i, t = DC_PLACE(e / DC_T), s = DC_PLACE(e % DC_T);
    B[e] = s < t ? dots[DC_B(t, s)] : 0.f;
  }
}

// sum over s of M[token, s] x_s for this lane's four tokens (place 4 quad + i) and its column, one product after the other, M [16, 16] in
// scratch; s <= t, or s < t.  For values that are not finite: a matrix-core product multiplies them with zeros as well.
template <bool OWN>
__device__ inline f32x4_d dc_lower(const float* M, const f32x4_d& x, f32x4_d sum, int col, int quad) {
#pragma unroll
  for (int s = 0; s < DC_T; ++s) {
    const float xs = __shfl(x[s / 4], (s % 4) * 16 + col, TP_WAVE);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (OWN ? s <= 4 * i + quad : s < 4 * i + quad) sum[i] = fmaf(M[(4 * quad + i) * DC_T + DC_PLACE(s)], xs, sum[i]);
  }
  return sum;
}

__device__ inline bool dc_finite(const f32x4_d& x) {
  float odd = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) odd = fmaf(x[i], 0.f, odd);
  return !__any(!(odd == 0.f));
}

// CT: tiles of 16 value columns a block.
template <int KT, int CT>
__global__ __launch_bounds__(256) void delta_chunk_scan_kernel(DeltaChunkArgs x) {
  constexpr int K = 16 * KT, TILES = KT / 4;      // 16-channel tiles of a wave
  const DeltaArgs& a = x.in;
  if ((int)blockIdx.x >= x.blocks) {      // the chain: as many lanes a column as in delta.hip's kernel of this key size
    constexpr int KS = K / 8, CB = 4 * TP_WAVE / KS;
    const int i = blockIdx.x - x.blocks, strips = (a.vdim + CB - 1) / CB, r = i / (a.heads * strips);
    if (a.cu_seqlens[r + 1] - a.cu_seqlens[r] <= DC_SHORT) delta_chain<8, KS>(a, r, i / strips % a.heads, i % strips);
    return;
  }
  __shared__ f32x4_d part[2][4][2 * CT][TP_WAVE];
  const int lane = threadIdx.x % TP_WAVE, wave = threadIdx.x / TP_WAVE, col = lane % 16, quad = lane / 16;
  // The blocks of a head read the same W, Q~ and K^: they go side by side to one XCD and its L2, and the heads to the XCDs in turn.
  const int strips = a.vdim / (16 * CT), pairs = x.requests * a.heads;
  const int rest = blockIdx.x >> 3, pair = rest / strips * 8 + (blockIdx.x & 7), strip = rest % strips;
  if (pair >= pairs) return;
  const int h = pair % a.heads, r = pair / a.heads;
  const int run = a.cu_seqlens[r + 1] - a.cu_seqlens[r];
  if (run <= DC_SHORT) return;
  // this run's groups that the launch holds: from its c0-th on, where `begin` is the launch's first for this run
  const int begin = dc_first_group(a.cu_seqlens, r, lane) - x.first, c0 = max(0, -begin);
  const int groups = min(x.groups - begin, (run + DC_T - 1) / DC_T) - c0;
  if (groups <= 0) return;
  const int run0 = a.cu_seqlens[r] + c0 * DC_T, left = run - c0 * DC_T;      // (the run from there on)
  const int j0 = strip * 16 * CT + col, i0 = wave * TILES * 16;      // (this lane's columns: j0 + 16 n)
  const size_t size = dc_item_floats(K);
  const float* vcol = a.qkv + (size_t)run0 * a.row_stride + 2 * (size_t)a.kv_heads * K + (size_t)h * a.vdim + j0;
  const float* item = x.scratch + ((size_t)(begin + c0) * a.heads + h) * size;
  float* Sm = a.state + (size_t)a.state_slots[r] * a.state_stride + a.state_off + ((size_t)h * a.vdim + j0) * K;
  f32x4_d S[CT][TILES];
#pragma unroll
  for (int n = 0; n < CT; ++n)
#pragma unroll
    for (int m = 0; m < TILES; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) S[n][m][i] = Sm[(size_t)16 * n * K + i0 + 16 * m + 4 * quad + i];
  struct Group {
    f32x4_d w[TILES], q[TILES], k[TILES], g[TILES], t, b, d, v[CT];
  };
  auto fetch = [&](Group& x, int c) {
    const float* p = item + (size_t)c * a.heads * size;
#pragma unroll
    for (int m = 0; m < TILES; ++m) {
      x.w[m] = *(const f32x4_d*)(p + (size_t)col * K + i0 + 16 * m + 4 * quad);
      x.q[m] = *(const f32x4_d*)(p + (size_t)(DC_T + col) * K + i0 + 16 * m + 4 * quad);
      x.k[m] = *(const f32x4_d*)(p + (size_t)2 * DC_T * K + (size_t)(i0 + 16 * m + col) * DC_T + 4 * quad);
      x.g[m] = *(const f32x4_d*)(p + (size_t)3 * DC_T * K + i0 + 16 * m + 4 * quad);
    }
    x.t = *(const f32x4_d*)(p + (size_t)49 * K + col * DC_T + 4 * quad);
    x.b = *(const f32x4_d*)(p + (size_t)49 * K + 256 + col * DC_T + 4 * quad);
    x.d = *(const f32x4_d*)(p + (size_t)49 * K + 512 + 4 * quad);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = c * DC_T + 4 * i + quad;
#pragma unroll
      for (int n = 0; n < CT; ++n) x.v[n][i] = t < left ? vcol[(size_t)t * a.row_stride + 16 * n] : 0.f;
    }
  };
  auto step = [&](const Group& x, int c) {
    f32x4_d(*buf)[2 * CT][TP_WAVE] = part[c & 1];
#pragma unroll
    for (int n = 0; n < CT; ++n) {
      f32x4_d ws[2], qs[2];
#pragma unroll
      for (int m = 0; m < TILES; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const bool first = m == 0 && i < 2;
          ws[i % 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w[m][i], S[n][m][i], first ? (f32x4_d)(0.f) : ws[i % 2], 0, 0, 0);
          qs[i % 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.q[m][i], S[n][m][i], first ? (f32x4_d)(0.f) : qs[i % 2], 0, 0, 0);
        }
      buf[wave][2 * n][lane] = ws[0] + ws[1];
      buf[wave][2 * n + 1][lane] = qs[0] + qs[1];
    }
#pragma unroll
    for (int n = 0; n < CT; ++n)
#pragma unroll
      for (int m = 0; m < TILES; ++m) S[n][m] *= x.g[m];
    __syncthreads();      // (the buffer of the group before is free again behind this one)
#pragma unroll
    for (int n = 0; n < CT; ++n) {
      const f32x4_d e = x.v[n] - ((buf[0][2 * n][lane] + buf[1][2 * n][lane]) + (buf[2][2 * n][lane] + buf[3][2 * n][lane]));
      const float* M = item + (size_t)c * a.heads * size + (size_t)49 * K;
      f32x4_d u = (f32x4_d)(0.f);
#pragma unroll
      for (int i = 0; i < 4; ++i) u = __builtin_amdgcn_mfma_f32_16x16x4f32(x.t[i], e[i], u, 0, 0, 0);
      if (!dc_finite(e)) u = dc_lower<true>(M, e, (f32x4_d)(0.f), col, quad);      // (looked at while the products run)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int m = 0; m < TILES; ++m) S[n][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[m][i], u[i], S[n][m], 0, 0, 0);
      if (wave == ((c + n) & 3)) {      // (the waves write the rows in turn)
        const int q0 = 2 * n + 1;
        f32x4_d o = (buf[0][q0][lane] + buf[1][q0][lane]) + (buf[2][q0][lane] + buf[3][q0][lane]);
        if (dc_finite(u)) {
          f32x4_d bu = (f32x4_d)(0.f);
#pragma unroll
          for (int i = 0; i < 4; ++i) bu = __builtin_amdgcn_mfma_f32_16x16x4f32(x.b[i], u[i], bu, 0, 0, 0);
          o += bu;
        } else {
          o = dc_lower<false>(M + 256, u, o, col, quad);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int t = c * DC_T + 4 * i + quad;
          // (a token's own part, most of the sum where decays are strong, is added last: one rounding at its size)
          if (t < left) a.y[((size_t)(run0 + t) * a.heads + h) * a.vdim + j0 + 16 * n] = fmaf(u[i], x.d[i], o[i]);
        }
      }
    }
  };
  Group even, odd;
  fetch(even, 0);
  for (int c = 0; c < groups; c += 2) {
    if (c + 1 < groups) fetch(odd, c + 1);
    step(even, c);
    if (c + 1 < groups) {
      if (c + 2 < groups) fetch(even, c + 2);
      step(odd, c + 1);
    }
  }
#pragma unroll
  for (int n = 0; n < CT; ++n)
#pragma unroll
    for (int m = 0; m < TILES; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) Sm[(size_t)16 * n * K + i0 + 16 * m + 4 * quad + i] = S[n][m][i];
}

// Groups that one pair of launches takes, 0: the runs are not these kernels'; *all: groups of the step, at most (a long run has more than
// DC_SHORT tokens, and one group that is not full).  The scratch is held to a quarter of a GB: longer steps take several pairs, each from
// the states that the one before left.  A pair then writes and reads that much, beside which its launches and the states are little.
static int dc_groups(int n, int n_req, int max_run, int heads, int dim, int vdim, int* all) {
  *all = 0;
  if (max_run <= DC_SHORT || (dim != 64 && dim != 128) || vdim % 16 != 0) return 0;
  const size_t fit = ((size_t)64 << 20) / ((size_t)heads * dc_item_floats(dim));
  if (fit < 1 || ((long)n_req * heads + 8) * (vdim / 16) >= 0x7fffffffL) return 0;
  const int runs = n / (DC_SHORT + 1);
  *all = n / DC_T + (runs < n_req ? runs : n_req);
  return (size_t)*all < fit ? *all : (int)fit;
}

// Floats of scratch for n tokens in n_req runs of up to max_run (0: all go token by token).
extern "C" size_t tp_delta_scan_scratch(int n, int n_req, int max_run, int heads, int dim, int vdim) {
  if (n <= 0 || n_req <= 0 || heads <= 0 || dim <= 0 || vdim <= 0) return 0;
  int all;
  return (size_t)dc_groups(n, n_req, max_run, heads, dim, vdim, &all) * heads * dc_item_floats(dim);
}

// Returns 0 when it took the step's runs, -1 when none of them is a long one of its own, DC_SHORT when it took those alone that are longer.
int tp_delta_chunks(const DeltaArgs& in, int n, int n_req, int max_run, float* scratch, size_t scratch_floats, hipStream_t s) {
  const int heads = in.heads, dim = in.dim, vdim = in.vdim;
  int all;
  const int groups = dc_groups(n, n_req, max_run, heads, dim, vdim, &all);
  if (groups == 0 || scratch == nullptr || ((uintptr_t)scratch & 15) || scratch_floats < (size_t)groups * heads * dc_item_floats(dim)) return -1;
  // (32 columns a block read K~, Q~ and K^ half as often, which bounds the chain once there are more blocks of 16 columns than the two
  // a CU that run at a time: 16 heads of 128 x 128, four runs of 451 tokens, 512 blocks of 16 columns or half as many of 32: 94 / 102 us;
  // 32 heads, eight runs of 256, 2,048 blocks: 202 / 174 when the rule was made.  Blocks of short runs end at once and do not count.)
  const long others = max_run < n ? (n - max_run) / (DC_SHORT + 1) : 0, long_runs = 1 + (others < n_req - 1 ? others : n_req - 1);
  const bool wide = vdim % 32 == 0 && long_runs * heads * (vdim / 16) > 512;
  // Short runs go beside the long ones, in blocks behind theirs (one behind the other the two kinds would add their chains), unless the
  // shortest run that such a step can have is a long one.
  const bool short_runs = (long)n - (long)(n_req - 1) * max_run <= DC_SHORT;
  const int column_block = dim == 128 ? 16 : 32;
  // (Where their blocks are many beside a long run that ends soon, they are left to delta.hip's kernels, which hold five blocks a CU where
  // the registers of the groups' kernel hold two.  128 x 128, in the same launches / apart: 16 heads, 64 tokens beside 100 single ones 101 /
  // 88 us, 128 beside 127 123 / 103, 128 beside 31 47 / 52, 700 beside 127 145 / 156; 32 heads, 300 beside 100 213 / 188, 1,800 beside 247
  // 601 / 705.)
  const bool apart = short_runs && (long)n_req * heads * ((vdim + column_block - 1) / column_block) > 40L * max_run;
  const long unit_blocks = short_runs && !apart ? (long)n * ((in.kv_heads + DC_HEADS - 1) / DC_HEADS) : 0;
  const long chain_blocks = short_runs && !apart ? (long)n_req * heads * ((vdim + column_block - 1) / column_block) : 0;
  const long scan_blocks = ((long)n_req * heads + 7) / 8 * 8 * (vdim / (wide ? 32 : 16));
  if ((long)groups * heads + unit_blocks >= 0x7fffffffL || scan_blocks + chain_blocks >= 0x7fffffffL) return -1;
  DeltaChunkArgs a{in, scratch, n_req, 0, groups, 0};
  for (; a.first < all; a.first += groups) {
    const long prep_blocks = (long)(groups < all - a.first ? groups : all - a.first) * heads;
    const dim3 prep((unsigned)(prep_blocks + (a.first == 0 ? unit_blocks : 0))), scan((unsigned)(scan_blocks + (a.first == 0 ? chain_blocks : 0)));
    a.blocks = (int)prep_blocks;
    if (dim == 128) hipLaunchKernelGGL(delta_chunk_prep_kernel<2>, prep, dim3(64), 0, s, a);
    else hipLaunchKernelGGL(delta_chunk_prep_kernel<1>, prep, dim3(64), 0, s, a);
    a.blocks = (int)scan_blocks;
#define DC_SCAN(KT_)                                                                                                 \
  do {                                                                                                               \
    if (wide) hipLaunchKernelGGL((delta_chunk_scan_kernel<KT_, 2>), scan, dim3(256), 0, s, a);                       \
    else hipLaunchKernelGGL((delta_chunk_scan_kernel<KT_, 1>), scan, dim3(256), 0, s, a);                            \
  } while (0)
    if (dim == 128) DC_SCAN(8);
    else DC_SCAN(4);
#undef DC_SCAN
  }
  return apart ? DC_SHORT : 0;
}
