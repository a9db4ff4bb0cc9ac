// A selective state-space mixer (state-space duality form) over a batch of requests that each bring a run of
// tokens: short causal convolution with carried inputs, the recurrence over a per-request state, and the gated
// grouped norm behind it.  All arithmetic is float32; the state lives in float32 rows of a per-request state tensor
// (row = request slot): first the convolution's last taps - 1 inputs, [taps - 1, channels], oldest first, then
// the recurrent state, [heads, state, head_dim].
//
// A request r of the batch owns tokens cu_seqlens[r] .. cu_seqlens[r + 1] - 1 and the state row state_slots[r];
// everything is read from device memory, so the same launches serve prompt portions, single decoded tokens and
// captured steps.  How a prompt was cut changes rounding only.
#include <math.h>

#include "common.h"

__device__ inline float silu_f(float v) { return v / (1.0f + expf(-v)); }
// ln(1 + e^v) without overflow: max(v, 0) + ln(1 + e^-|v|)
__device__ inline float softplus_f(float v) { return fmaxf(v, 0.f) + log1pf(expf(-fabsf(v))); }

// ---- causal convolution per channel (+ SiLU) --------------------------------------------------
// in: rows [n, in_stride] float32, the channels at column col0; w [taps, channels] (tap-major, so that the lanes of
// a wave read neighbouring weights; the last tap is the current token's), b [channels] or none.  The inputs before
// a run's first token come from the request's state row, from element state_off on (zeros for a fresh request).
// out [n, channels] = silu(conv + b), or conv + b itself when `act` is 0.
__global__ void causal_conv_kernel(const float* __restrict__ in, int in_stride, int col0, const float* __restrict__ w,
                                   const float* __restrict__ b, const float* __restrict__ state, size_t state_stride,
                                   const int* __restrict__ cu_seqlens, const int* __restrict__ token_req,
                                   const int* __restrict__ state_slots, float* __restrict__ out, int channels, int taps,
                                   int channel_blocks, size_t state_off, int act) {
  // (neighbouring blocks take neighbouring channels of one token: they read one row of the input after the other)
  const int t = blockIdx.x / channel_blocks;
  const int c = (blockIdx.x % channel_blocks) * blockDim.x + threadIdx.x;
  if (c >= channels) return;
  const int r = token_req[t];
  const int start = cu_seqlens[r];
  const int i = t - start;
  const float* st = state + (size_t)state_slots[r] * state_stride + state_off;
  float acc = b != nullptr ? b[c] : 0.f;
  for (int k = 0; k < taps; ++k) {
    const int src = i - (taps - 1 - k);
    const float v = src >= 0 ? in[(size_t)(start + src) * in_stride + col0 + c] : st[(size_t)(taps - 1 + src) * channels + c];
    acc = fmaf(w[(size_t)k * channels + c], v, acc);
  }
  out[(size_t)t * channels + c] = act ? silu_f(acc) : acc;
}

// The state after a run: the last taps - 1 inputs of (carried inputs, then the run's).  In place, ascending: entry j
// takes entry j + len of the old state or an input of the run, and entries below j are never read again.
__global__ void conv_state_kernel(const float* __restrict__ in, int in_stride, int col0, float* __restrict__ state,
                                  size_t state_stride, const int* __restrict__ cu_seqlens,
                                  const int* __restrict__ state_slots, int channels, int taps, size_t state_off) {
  const int r = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= channels) return;
  const int start = cu_seqlens[r], len = cu_seqlens[r + 1] - start;
  if (len <= 0) return;
  float* st = state + (size_t)state_slots[r] * state_stride + state_off;
  for (int j = 0; j < taps - 1; ++j) {
    const int src = len - (taps - 1) + j;
    const float v = src >= 0 ? in[(size_t)(start + src) * in_stride + col0 + c] : st[(size_t)(j + len) * channels + c];
    st[(size_t)j * channels + c] = v;
  }
}

// The same, four neighbouring channels and a run of CONV_RUN tokens a thread (16-byte places, at most CONV_TAPS taps): a row is
// read once by the thread that needs it for all taps, where a thread a token reads every row once a tap, and all rows of a run are
// in flight together.  A channel's sum is formed in the order of the kernel above: the same bits.  10,240 channels, four taps,
// 2,048 tokens (168 MB): 102 -> 44 us.
#define CONV_RUN 8
#define CONV_TAPS 4
__global__ __launch_bounds__(256) void causal_conv_run_kernel(const float* __restrict__ in, int in_stride, int col0,
                                                              const float* __restrict__ w, const float* __restrict__ b,
                                                              const float* __restrict__ state, size_t state_stride,
                                                              const int* __restrict__ cu_seqlens, const int* __restrict__ token_req,
                                                              const int* __restrict__ state_slots, float* __restrict__ out, int n,
                                                              int channels, int taps, int channel_blocks, size_t state_off, int act) {
  const int t0 = blockIdx.x / channel_blocks * CONV_RUN;
  const int c = ((blockIdx.x % channel_blocks) * 256 + threadIdx.x) * 4;
  if (c >= channels) return;
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  float4 wv[CONV_TAPS];   // the last CONV_TAPS places of the window; a shorter filter leaves the first ones zero
#pragma unroll
  for (int k = 0; k < CONV_TAPS; ++k) {
    const int j = k - (CONV_TAPS - taps);
    wv[k] = j >= 0 ? *(const float4*)(w + (size_t)j * channels + c) : zero;
  }
  const float4 bias = b != nullptr ? *(const float4*)(b + c) : zero;
  float4 row[CONV_RUN];
#pragma unroll
  for (int i = 0; i < CONV_RUN; ++i)
    row[i] = t0 + i < n ? *(const float4*)(in + (size_t)(t0 + i) * in_stride + col0 + c) : zero;
  float4 win[CONV_TAPS - 1];   // the inputs before the token, oldest first
  int run_end = t0;            // (the first token below opens a run or joins one)
#pragma unroll
  for (int i = 0; i < CONV_RUN; ++i) {
    const int t = t0 + i;
    if (t >= n) break;
    if (t == run_end) {        // uniform over the block
      const int r = token_req[t], start = cu_seqlens[r];
      run_end = cu_seqlens[r + 1];
      const float* st = state + (size_t)state_slots[r] * state_stride + state_off + c;
#pragma unroll
      for (int k = 0; k < CONV_TAPS - 1; ++k) {
        const int src = t - start - (CONV_TAPS - 1) + k, j = taps - 1 + src;
        if (src >= 0)
          win[k] = *(const float4*)(in + (size_t)(start + src) * in_stride + col0 + c);
        else if (j >= 0)       // (the carried rows' place need not be aligned)
          win[k] = make_float4(st[(size_t)j * channels], st[(size_t)j * channels + 1], st[(size_t)j * channels + 2], st[(size_t)j * channels + 3]);
        else
          win[k] = zero;
      }
    }
    float4 acc = bias;
#pragma unroll
    for (int k = 0; k < CONV_TAPS; ++k) {
      if (k < CONV_TAPS - taps) continue;
      const float4 v = k < CONV_TAPS - 1 ? win[k] : row[i];
      acc.x = fmaf(wv[k].x, v.x, acc.x);
      acc.y = fmaf(wv[k].y, v.y, acc.y);
      acc.z = fmaf(wv[k].z, v.z, acc.z);
      acc.w = fmaf(wv[k].w, v.w, acc.w);
    }
#pragma unroll
    for (int k = 0; k < CONV_TAPS - 2; ++k) win[k] = win[k + 1];
    win[CONV_TAPS - 2] = row[i];
    if (act) acc = make_float4(silu_f(acc.x), silu_f(acc.y), silu_f(acc.z), silu_f(acc.w));
    *(float4*)(out + (size_t)t * channels + c) = acc;
  }
}

// Every request brings one token: the convolution and the state after it in one launch (a thread is the only reader of its
// channel's carried inputs).  Same sums as above.
__global__ void causal_conv_single_kernel(const float* __restrict__ in, int in_stride, int col0, const float* __restrict__ w,
                                          const float* __restrict__ b, float* __restrict__ state, size_t state_stride,
                                          const int* __restrict__ token_req, const int* __restrict__ state_slots,
                                          float* __restrict__ out, int channels, int taps, int channel_blocks, size_t state_off, int act) {
  const int t = blockIdx.x / channel_blocks;
  const int c = (blockIdx.x % channel_blocks) * blockDim.x + threadIdx.x;
  if (c >= channels) return;
  const float cur = in[(size_t)t * in_stride + col0 + c];
  float* st = state + (size_t)state_slots[token_req[t]] * state_stride + state_off + c;
  float acc = b != nullptr ? b[c] : 0.f;
  for (int k = 0; k < taps; ++k) {
    const float v = k < taps - 1 ? st[(size_t)k * channels] : cur;
    if (k > 0) st[(size_t)(k - 1) * channels] = v;
    acc = fmaf(w[(size_t)k * channels + c], v, acc);
  }
  out[(size_t)t * channels + c] = act ? silu_f(acc) : acc;
}

extern "C" int tp_causal_conv(const float* in, int in_stride, int col0, const float* w, const float* b, float* state,
                              size_t state_stride, size_t state_off, const int* cu_seqlens, const int* token_req,
                              const int* state_slots, float* out, int n, int n_req, int channels, int taps, int act,
                              int max_run, hipStream_t s) {
  // (max_run: the longest run of the step, 0: not known)
  TP_REQUIRE(n >= 0 && n_req >= 0 && channels > 0 && taps >= 1, "causal_conv: bad sizes");
  TP_REQUIRE(in_stride >= col0 + channels && state_stride >= state_off + (size_t)(taps - 1) * channels, "causal_conv: rows too short");
  if (n == 0) return 0;
  const int threads = channels >= 256 ? 256 : 64;
  const int cb = (channels + threads - 1) / threads;
  TP_REQUIRE(cb <= 65535 && (long)n * cb < 0x7fffffffL, "causal_conv: too many channels or tokens");
  if (max_run == 1) {
    hipLaunchKernelGGL(causal_conv_single_kernel, dim3((unsigned)((long)n * cb)), dim3(threads), 0, s, in, in_stride, col0, w, b, state,
                       state_stride, token_req, state_slots, out, channels, taps, cb, state_off, act);
    TP_CHECK_LAUNCH("causal_conv");
    return 0;
  }
  const bool four = taps >= 2 && taps <= CONV_TAPS && channels % 4 == 0 && in_stride % 4 == 0 && col0 % 4 == 0 &&
                    (((uintptr_t)in | (uintptr_t)w | (uintptr_t)b | (uintptr_t)out) & 15) == 0;
  // (a thread's run is a chain of three dependent trips to memory, 9 us whatever the step: the grid of single tokens is faster until it
  // reads some megabytes four times over.  Four taps, single tokens / runs: 64 tokens of 10,240 channels 6.9 / 9.3 us, 130 9.9 / 9.7, 500
  // 26 / 17; 300 of 3,072 8.2 / 9.3, 500 10.7 / 9.7; 700 of 2,048 10.2 / 9.6; 2,000 of 512 8.8 / 9.0; two
  // taps, 500 of 3,072 8.9 / 9.1, 700 11.3 / 10.6)
  if (four && (long)n * channels >= (taps > 2 ? 1300000 : 1600000)) {
    const int qb = (channels / 4 + 255) / 256;
    hipLaunchKernelGGL(causal_conv_run_kernel, dim3((unsigned)((n + CONV_RUN - 1) / CONV_RUN * qb)), dim3(256), 0, s, in, in_stride, col0,
                       w, b, state, state_stride, cu_seqlens, token_req, state_slots, out, n, channels, taps, qb, state_off, act);
  } else {
    hipLaunchKernelGGL(causal_conv_kernel, dim3((unsigned)((long)n * cb)), dim3(threads), 0, s, in, in_stride, col0, w, b, state,
                       state_stride, cu_seqlens, token_req, state_slots, out, channels, taps, cb, state_off, act);
  }
  if (taps > 1 && n_req > 0)
    hipLaunchKernelGGL(conv_state_kernel, dim3(n_req, cb), dim3(threads), 0, s, in, in_stride, col0, state,
                       state_stride, cu_seqlens, state_slots, channels, taps, state_off);
  TP_CHECK_LAUNCH("causal_conv");
  return 0;
}

// ---- the recurrence ---------------------------------------------------------------------------
// Per head h (its inputs B and C are those of group h / (heads / groups)), with dt = softplus(dt_raw + dt_bias[h])
// and a = exp(-exp(a_log[h]) * dt):
//   S <- a S + dt * B x^T        (S is [state, head_dim], float32)
//   y  = S^T C + d_skip[h] * x
// xbc [n, channels] float32 holds, per token, x [heads * head_dim] | B [groups * state] | C [groups * state] (after
// the convolution); dt_raw is column dt_col0 + h of the projection's rows.
//
// A block owns one request, one head and PC = (256 / R) * TP value columns; a thread holds TN consecutive state
// entries of TP neighbouring columns in registers, and the R lanes (a power of two, neighbours in a wave) that share
// those columns split the state index among them.
// Tokens are taken TC at a time: their B, C, x, dt and decay are staged in LDS by all threads (rows padded with
// zeros to R * TN entries, so the run itself needs no bounds), then the run over the chunk is register
// arithmetic, 16-byte LDS reads that most lanes share, and one reduction over the R lanes per token (row
// permutes up to 16 lanes, which cost an instruction each and no trip through LDS).
//
// Long runs are cut into pieces of `piece` tokens that run side by side (a recurrence is a chain, and a prompt of
// thousands of tokens on a chain leaves most of the chip idle).  Three launches:
//   SCAN_LOCAL   every piece from a zero state: its end state and its total decay, to scratch;
//   the carry    per state entry, piece by piece (ssm_carry_kernel): the state a piece starts from is
//                decay(previous piece) * (state the previous piece started from) + (its end state from zero);
//                the state after the last piece is the request's new state;
//   SCAN_OUTPUT  every piece again from the state it starts from, now writing y.
// Where the sizes fit, the first and the last of them are products on the matrix cores (ssm_chunk_kernel).
// Short runs take SCAN_DIRECT: one launch, from the request's state to its new state; single tokens a kernel of their own.
// How a run is cut changes rounding only.
enum { SCAN_DIRECT = 0, SCAN_LOCAL = 1, SCAN_OUTPUT = 2 };

struct ScanArgs {
  const float* xbc;
  const float* proj;
  int proj_stride, dt_col0;
  const float* dt_bias;
  const float* a_log;
  const float* d_skip;
  float* state;
  size_t state_stride, state_off;
  const int* cu_seqlens;
  const int* state_slots;
  float* y;
  int heads, head_dim, n_state, groups, channels;
  int R, TC;
  int mode, piece, max_pieces;
  int unit;             // heads that share B and C and run side by side (ssm_chunk_kernel)
  float* piece_state;   // [request, head, piece, n_state, head_dim]
  float* piece_decay;   // [request, head, piece]
};

// sum over the R lanes (R a power of two, the lanes neighbours from a multiple of R on); every lane gets it
__device__ inline float lanes_sum(float v, int R) {
#define DPP_ADD(ctrl) v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, 0xf, 0xf, false))
  if (R >= 2) DPP_ADD(0xB1);    // quad_perm [1, 0, 3, 2]
  if (R >= 4) DPP_ADD(0x4E);    // quad_perm [2, 3, 0, 1]
  if (R >= 8) DPP_ADD(0x141);   // row_half_mirror: lane i of eight reads lane 7 - i
  if (R >= 16) DPP_ADD(0x140);  // row_mirror: lane i of sixteen reads lane 15 - i
#undef DPP_ADD
  if (R >= 32) v += __shfl_xor(v, 16, TP_WAVE);
  if (R >= 64) v += __shfl_xor(v, 32, TP_WAVE);
  return v;
}

template <int TN, int TP>
__global__ __launch_bounds__(256) void ssm_scan_kernel(ScanArgs a) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int N = a.n_state, P = a.head_dim, R = a.R, CG = 256 / a.R, PC = CG * TP, TC = a.TC;
  const int NS = R * TN;           // padded row of B and C
  float* Bs = lds;                 // [TC, NS]
  float* Cs = Bs + (size_t)TC * NS;
  float* xs = Cs + (size_t)TC * NS; // [TC, PC]
  float* dts = xs + (size_t)TC * PC;
  float* das = dts + TC;
  const int r = blockIdx.x, h = blockIdx.y;
  const int slices = (P + PC - 1) / PC;
  const int slice = blockIdx.z % slices, pc = blockIdx.z / slices;
  const int cg = threadIdx.x / R, rr = threadIdx.x % R;
  const int p0 = slice * PC + cg * TP;      // this thread's first value column
  const int g = h / (a.heads / a.groups);
  const int run0 = a.cu_seqlens[r], run_len = a.cu_seqlens[r + 1] - run0;
  if (run_len <= 0) return;
  const int inner = a.heads * P;
  const int n0 = rr * TN;
  float* S = a.state + (size_t)a.state_slots[r] * a.state_stride + a.state_off + (size_t)h * N * P;
  const int pieces = a.mode == SCAN_DIRECT ? 1 : (run_len + a.piece - 1) / a.piece;
  float* PS = a.piece_state + ((size_t)(r * a.heads + h) * a.max_pieces) * N * P;
  float* PD = a.piece_decay + (size_t)(r * a.heads + h) * a.max_pieces;
#define SCAN_HAS(i, j) (n0 + (i) < N && p0 + (j) < P)
#define SCAN_AT(i, j) ((size_t)(n0 + (i)) * P + p0 + (j))

  if (pc >= pieces) return;
  const int start = a.mode == SCAN_DIRECT ? run0 : run0 + pc * a.piece;
  const int len = a.mode == SCAN_DIRECT ? run_len : min(a.piece, run_len - pc * a.piece);
  const float* init = a.mode == SCAN_DIRECT ? S : (a.mode == SCAN_OUTPUT ? PS + (size_t)pc * N * P : nullptr);
  float st[TN][TP];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TP; ++j) st[i][j] = (init != nullptr && SCAN_HAS(i, j)) ? init[SCAN_AT(i, j)] : 0.f;
  const float A = -expf(a.a_log[h]);
  const float dtb = a.dt_bias[h], Dh = a.d_skip[h];
  const bool write_y = a.mode != SCAN_LOCAL;
  float dt_sum = 0.f;
  for (int t0 = 0; t0 < len; t0 += TC) {
    const int nt = min(TC, len - t0);
    __syncthreads();
    // (a wave stages every fourth token, its lanes the entries of a row: no division in the loop)
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int tt = wave; tt < nt; tt += 4) {
      const float* row = a.xbc + (size_t)(start + t0 + tt) * a.channels;
      for (int n = lane; n < NS; n += 64) {
        float bv = 0.f, cv = 0.f;
        if (n < N) {
          bv = row[inner + g * N + n];
          cv = row[inner + (a.groups + g) * N + n];
        }
        Bs[tt * NS + n] = bv;
        Cs[tt * NS + n] = cv;
      }
      for (int c = lane; c < PC; c += 64) {
        const int pp = slice * PC + c;
        xs[tt * PC + c] = pp < P ? row[h * P + pp] : 0.f;
      }
    }
    for (int idx = threadIdx.x; idx < nt; idx += 256) {
      const float dt = softplus_f(a.proj[(size_t)(start + t0 + idx) * a.proj_stride + a.dt_col0 + h] + dtb);
      dts[idx] = dt;
      das[idx] = expf(A * dt);
    }
    __syncthreads();
    for (int tt = 0; tt < nt; ++tt) {
      const float dt = dts[tt], da = das[tt];
      float xv[TP], dx[TP], acc[TP];
#pragma unroll
      for (int j = 0; j < TP; ++j) {
        xv[j] = xs[tt * PC + cg * TP + j];
        dx[j] = dt * xv[j];
        acc[j] = 0.f;
      }
      const float* Bt = Bs + (size_t)tt * NS + n0;
      const float* Ct = Cs + (size_t)tt * NS + n0;
      float bv[TN], cv[TN];
      if constexpr (TN % 4 == 0) {
#pragma unroll
        for (int i = 0; i < TN; i += 4) {
          const float4 b4 = *(const float4*)(Bt + i), c4 = *(const float4*)(Ct + i);
          bv[i] = b4.x; bv[i + 1] = b4.y; bv[i + 2] = b4.z; bv[i + 3] = b4.w;
          cv[i] = c4.x; cv[i + 1] = c4.y; cv[i + 2] = c4.z; cv[i + 3] = c4.w;
        }
      } else {
#pragma unroll
        for (int i = 0; i < TN; ++i) {
          bv[i] = Bt[i];
          cv[i] = Ct[i];
        }
      }
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TP; ++j) {
          st[i][j] = fmaf(da, st[i][j], dx[j] * bv[i]);
          acc[j] = fmaf(st[i][j], cv[i], acc[j]);
        }
      dt_sum += dt;
      if (write_y) {
#pragma unroll
        for (int j = 0; j < TP; ++j) {
          const float total = lanes_sum(acc[j], R);
          if (rr == 0 && p0 + j < P) a.y[(size_t)(start + t0 + tt) * inner + h * P + p0 + j] = fmaf(Dh, xv[j], total);
        }
      }
    }
  }
  if (a.mode == SCAN_OUTPUT) return;
  float* dst = a.mode == SCAN_DIRECT ? S : PS + (size_t)pc * N * P;
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TP; ++j)
      if (SCAN_HAS(i, j)) dst[SCAN_AT(i, j)] = st[i][j];
  if (a.mode == SCAN_LOCAL && slice == 0 && threadIdx.x == 0) PD[pc] = expf(A * dt_sum);
#undef SCAN_HAS
#undef SCAN_AT
}

// ---- one token a request ----------------------------------------------------------------------------
// The recurrence for runs of one token (a run of none is left alone): the threads, their entries and the order of every sum are those of
// ssm_scan_kernel, so the bits are the same, but nothing passes through LDS and nothing waits behind a barrier.  Bound by two dependent
// trips to memory (where the request's token and state are; the state and the token's inputs, all requested at once) and, for many
// requests, by the state, read and written.  128 heads of 64 with a state of 128, one request: 10 us in
// the loop over chunks, 6.8 here; four 13.5 / 12.2 us, sixteen 43 / 37; 64 heads with a state of 64, four requests 7.2 / 4.8.
template <int TN, int TP>
__global__ __launch_bounds__(256) void ssm_step_kernel(ScanArgs a) {
  const int N = a.n_state, P = a.head_dim, R = a.R, PC = 256 / R * TP;
  const int r = blockIdx.x, h = blockIdx.y, slice = blockIdx.z;
  const int cg = threadIdx.x / R, rr = threadIdx.x % R;
  const int p0 = slice * PC + cg * TP, n0 = rr * TN;
  const int g = h / (a.heads / a.groups), inner = a.heads * P;
  const int t = a.cu_seqlens[r], len = a.cu_seqlens[r + 1] - t, slot = a.state_slots[r];
  const float A = -expf(a.a_log[h]), dtb = a.dt_bias[h], Dh = a.d_skip[h];
  if (len <= 0) return;
  float* S = a.state + (size_t)slot * a.state_stride + a.state_off + (size_t)h * N * P + (size_t)n0 * P + p0;
  const float* row = a.xbc + (size_t)t * a.channels;
  const float* Bp = row + inner + g * N + n0;
  const float* Cp = row + inner + (a.groups + g) * N + n0;
  const bool pairs = TP == 2 && P % 2 == 0 && ((uintptr_t)S & 7) == 0;
  const bool quads = TN % 4 == 0 && (((uintptr_t)Bp | (uintptr_t)Cp) & 15) == 0 && n0 + TN <= N;
  float st[TN][TP], bv[TN], cv[TN], xv[TP];
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    if (pairs && n0 + i < N && p0 + 1 < P) {
      const float2 v = *(const float2*)(S + (size_t)i * P);
      st[i][0] = v.x;
      st[i][TP - 1] = v.y;
    } else {
#pragma unroll
      for (int j = 0; j < TP; ++j) st[i][j] = (n0 + i < N && p0 + j < P) ? S[(size_t)i * P + j] : 0.f;
    }
  }
  if (quads) {
#pragma unroll
    for (int i = 0; i < TN; i += 4) {
      const float4 b4 = *(const float4*)(Bp + i), c4 = *(const float4*)(Cp + i);
      const float b[4] = {b4.x, b4.y, b4.z, b4.w}, c[4] = {c4.x, c4.y, c4.z, c4.w};
#pragma unroll
      for (int d = 0; d < 4 && i + d < TN; ++d) bv[i + d] = b[d], cv[i + d] = c[d];
    }
  } else {
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      bv[i] = n0 + i < N ? Bp[i] : 0.f;
      cv[i] = n0 + i < N ? Cp[i] : 0.f;
    }
  }
#pragma unroll
  for (int j = 0; j < TP; ++j) xv[j] = p0 + j < P ? row[h * P + p0 + j] : 0.f;
  const float dt = softplus_f(a.proj[(size_t)t * a.proj_stride + a.dt_col0 + h] + dtb), da = expf(A * dt);
  float acc[TP];
#pragma unroll
  for (int j = 0; j < TP; ++j) acc[j] = 0.f;
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TP; ++j) {
      st[i][j] = fmaf(da, st[i][j], dt * xv[j] * bv[i]);
      acc[j] = fmaf(st[i][j], cv[i], acc[j]);
    }
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    if (pairs && n0 + i < N && p0 + 1 < P) {
      *(float2*)(S + (size_t)i * P) = make_float2(st[i][0], st[i][TP - 1]);
    } else {
#pragma unroll
      for (int j = 0; j < TP; ++j)
        if (n0 + i < N && p0 + j < P) S[(size_t)i * P + j] = st[i][j];
    }
  }
#pragma unroll
  for (int j = 0; j < TP; ++j) {
    const float total = lanes_sum(acc[j], R);
    if (rr == 0 && p0 + j < P) a.y[(size_t)t * inner + h * P + p0 + j] = fmaf(Dh, xv[j], total);
  }
}

// ---- pieces of a long run on the matrix cores -----------------------------------------------------
// The same two passes over a piece (SCAN_LOCAL, SCAN_OUTPUT) for states of 16 x NT entries, 32 tokens at a time as four products with
// v_mfma_f32_16x16x4_f32.  With c_t the sum of dt up to token t of the 32 and S the state before them:
//   y_t = exp(A c_t) S^T C_t + sum over s <= t of (C_t . B_s) exp(A (c_t - c_s)) dt_s x_s + d_skip x_t
//   S  <- exp(A c_31) S + sum over s of exp(A (c_31 - c_s)) dt_s B_s x_s^T
// The sums c are float64 and every exponent is at most zero, so a decay over many tokens is one exponential of a difference: its error
// does not grow with the distance, as that of a product of steps does.
// A block owns one request, head, piece and 64 value columns; a wave keeps the state of 16 columns in accumulators, which lie as the
// next product's operand wants them (a lane holds four entries of one column), so the state never leaves the registers.  C_t . B_s is
// worked out once a block (one 16 x 16 tile a wave) and passed through LDS with its weights; the tile above the diagonal is left out.
// Sums over the state are added in runs of eight products (C . B: four): longer chains of roundings would lose to the walk's, which adds
// 16 a lane and then the lanes in a tree.  Tokens lie in LDS so that every product over them adds them in ascending order (SC_PLACE), and
// a token's own part is added behind it: with strong decays the tokens nearest to a result are most of it, and what is added last is
// rounded least often.  Root mean square error against float64 over the walk's, decays near one / strong / strong with small steps: states
// of 16 0.84 / 0.93 / 0.95, 32 0.91 / 0.95 / 0.99, 64 0.84 / 0.93 / 0.96, 128 0.82 / 0.87 / 0.89.  (In the order of the rows, a token's own
// part among the others', 32 entries 0.94 / 1.05 / 1.02 and 128 0.84 / 0.94 / 0.94; the order costs 2 to 4 % of the time.)
// Up to 16 heads that share B and C of a piece are a unit and go to one XCD and its L2, the units to the XCDs in turn.
//
// Bound by the matrix cores: 2,048 tokens of 128 heads of 64 with a state of 128 are 14.5 GFLOP in both passes, 100 us at the float32
// rate; with the carry 225 us, token by token 653 (257 tokens 62 / 206 us; 32 heads of 64 with a state of 16, 2,048 tokens, 36 / 125).
// (Two blocks a CU for a state of 128: held to three the last pass spills, 248 us.)
#define SC_T 32     // tokens at a time
#define SC_P 64     // value columns a block
// the row in LDS of token t of the 32: instruction i of a product over 16 tokens takes element i of each lane, from lanes quad = 0 .. 3,
// so with token 4 i + quad in row 4 quad + i the instructions run through them in order (its own inverse)
#define SC_PLACE(t) (((t) & 16) + 4 * ((t) & 3) + (((t) & 15) >> 2))
typedef float f32x4_s __attribute__((ext_vector_type(4)));

template <int NT, bool OUT>
__global__ __launch_bounds__(256, OUT && NT == 8 ? 2 : 3) void ssm_chunk_kernel(ScanArgs a, int requests) {
  constexpr int N = 16 * NT, LD = N + 4, NV = (SC_T * N / 4 + 255) / 256;
  __shared__ __attribute__((aligned(16))) float Bs[SC_T][LD];
  __shared__ __attribute__((aligned(16))) float Cs[OUT ? SC_T : 1][LD];
  __shared__ __attribute__((aligned(16))) float xs[SC_T][SC_P + 4];
  __shared__ __attribute__((aligned(16))) float Gs[OUT ? SC_T : 1][SC_T + 4];
  __shared__ double cs[SC_T];
  __shared__ __attribute__((aligned(16))) float dts[SC_T], from_start[SC_T], to_end[SC_T], diag[OUT ? SC_T : 4];
  const int P = a.head_dim, slices = (P + SC_P - 1) / SC_P;
  long item = (long)(blockIdx.x >> 3) / a.unit * 8 + (blockIdx.x & 7);      // (units go to the XCDs in turn)
  const int units = a.heads / a.unit;
  const int h = (int)(item % units) * a.unit + (int)(blockIdx.x >> 3) % a.unit;
  item /= units;
  const int slice = (int)(item % slices);
  item /= slices;
  const int pc = (int)(item % a.max_pieces), r = (int)(item / a.max_pieces);
  if (r >= requests) return;
  const int run0 = a.cu_seqlens[r], run_len = a.cu_seqlens[r + 1] - run0;
  const int start = run0 + pc * a.piece, len = min(a.piece, run_len - pc * a.piece);
  if (len <= 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, col = lane & 15, quad = lane >> 4;
  const int g = h / (a.heads / a.groups), inner = a.heads * P;
  const int p = slice * SC_P + wave * 16 + col;      // this lane's value column
  const bool live = p < P;                           // (P is a multiple of 16: a wave's columns are all there or none is)
  float* state = a.piece_state + (((size_t)r * a.heads + h) * a.max_pieces + pc) * N * P;
  const float A = -expf(a.a_log[h]), dtb = a.dt_bias[h], Dh = a.d_skip[h];
  f32x4_s S[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) S[j][i] = (OUT && live) ? state[(size_t)(16 * j + 4 * quad + i) * P + p] : 0.f;

  f32x4_s br[NV], cr[OUT ? NV : 1], xr[2];
  float dt_raw = 0.f;
  auto fetch = [&](int t0) {     // the next tokens on their way (rows past the piece's last: zeros)
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int idx = tid + 256 * v, t = idx / (N / 4), n = idx % (N / 4) * 4;
      const bool ok = t < SC_T && t0 + t < len;
      const float* row = a.xbc + (size_t)(start + (ok ? t0 + t : 0)) * a.channels + inner;
      br[v] = ok ? *(const f32x4_s*)(row + g * N + n) : (f32x4_s)(0.f);
      if constexpr (OUT) cr[v] = ok ? *(const f32x4_s*)(row + (a.groups + g) * N + n) : (f32x4_s)(0.f);
    }
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      const int t = (tid >> 4) + 16 * v, c = slice * SC_P + (tid & 15) * 4;
      xr[v] = (t0 + t < len && c < P) ? *(const f32x4_s*)(a.xbc + (size_t)(start + t0 + t) * a.channels + (size_t)h * P + c) : (f32x4_s)(0.f);
    }
    if (wave == 0 && lane < SC_T && t0 + lane < len) dt_raw = a.proj[(size_t)(start + t0 + lane) * a.proj_stride + a.dt_col0 + h];
  };
  double dt_sum = 0.0;
  fetch(0);
  for (int t0 = 0; t0 < len; t0 += SC_T) {
    __syncthreads();
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int idx = tid + 256 * v, t = idx / (N / 4), n = idx % (N / 4) * 4;
      if (t < SC_T) {
        *(f32x4_s*)&Bs[SC_PLACE(t)][n] = br[v];
        if constexpr (OUT) *(f32x4_s*)&Cs[SC_PLACE(t)][n] = cr[v];
      }
    }
#pragma unroll
    for (int v = 0; v < 2; ++v) *(f32x4_s*)&xs[SC_PLACE((tid >> 4) + 16 * v)][(tid & 15) * 4] = xr[v];
    if (wave == 0) {
      const float dt = (lane < SC_T && t0 + lane < len) ? softplus_f(dt_raw + dtb) : 0.f;
      double c = dt;
#pragma unroll
      for (int d = 1; d < SC_T; d *= 2) {
        const double below = __shfl_up(c, d, SC_T);
        if ((lane & (SC_T - 1)) >= d) c += below;
      }
      const double all = __shfl(c, SC_T - 1, TP_WAVE);
      dt_sum += all;
      if (lane < SC_T) {
        // (a difference of zero is a decay of one, whatever A is)
        const int row = SC_PLACE(lane);
        cs[row] = c;
        dts[row] = dt;
        from_start[row] = c == 0.0 ? 1.f : expf((float)(A * c));
        to_end[row] = all == c ? 1.f : expf((float)(A * (all - c)));
      }
    }
    __syncthreads();
    if (t0 + SC_T < len) fetch(t0 + SC_T);

    if constexpr (OUT) {
      // C_t . B_s with its weight, rows t of 16 and columns s of 16 a wave: (0, 0), (16, 0), (16, 16); a token's own beside them
      if (wave < 3) {
        const int tt = wave > 0 ? 16 : 0, ss = wave > 1 ? 16 : 0, row = tt + col, t = SC_PLACE(row);
        f32x4_s cb = (f32x4_s)(0.f);
#pragma unroll
        for (int j0 = 0; j0 < NT; j0 += 2) {
          f32x4_s part[2];
#pragma unroll
          for (int j = j0; j < j0 + 2 && j < NT; ++j) {
            f32x4_s sum[4];
            const f32x4_s b4 = *(const f32x4_s*)&Bs[ss + col][16 * j + 4 * quad], c4 = *(const f32x4_s*)&Cs[row][16 * j + 4 * quad];
#pragma unroll
            for (int i = 0; i < 4; ++i) sum[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(b4[i], c4[i], (f32x4_s)(0.f), 0, 0, 0);
            part[j - j0] = (sum[0] + sum[1]) + (sum[2] + sum[3]);
          }
          cb += NT > 1 ? part[0] + part[1] : part[0];
        }
        const double ct = cs[row];
        f32x4_s w;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int at = ss + 4 * quad + i, s = ss + 4 * i + quad;
          const double d = ct - cs[at];
          const float decay = d == 0.0 ? 1.f : expf((float)(A * d));
          w[i] = s < t ? cb[i] * decay * dts[at] : 0.f;
          if (s == t) diag[row] = cb[i] * dts[at];
        }
        *(f32x4_s*)&Gs[row][ss + 4 * quad] = w;
      }
    }
    // this lane's x: tokens 16 k + 4 i + quad of its column, rows 16 k + 4 quad + i
    f32x4_s xv[2];
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i) xv[k][i] = xs[16 * k + 4 * quad + i][wave * 16 + col];
    if constexpr (OUT) {
      f32x4_s y[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        y[k] = (f32x4_s)(0.f);
#pragma unroll
        for (int j0 = 0; j0 < NT; j0 += 2) {
          f32x4_s sum[4];
#pragma unroll
          for (int j = j0; j < j0 + 2 && j < NT; ++j) {
            const f32x4_s c4 = *(const f32x4_s*)&Cs[16 * k + col][16 * j + 4 * quad];
#pragma unroll
            for (int i = 0; i < 4; ++i) sum[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(c4[i], S[j][i], j == j0 ? (f32x4_s)(0.f) : sum[i], 0, 0, 0);
          }
          y[k] += (sum[0] + sum[1]) + (sum[2] + sum[3]);
        }
      }
      __syncthreads();
      // A zero of the weights times an x that is not finite would reach tokens before it: those columns are added one by one.
      float odd = 0.f;
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int i = 0; i < 4; ++i) odd = fmaf(xv[k][i], 0.f, odd);
      if (__any(!(odd == 0.f))) {
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int row = 16 * k + 4 * quad + i, t = SC_PLACE(row);
            y[k][i] *= from_start[row];
            for (int s = 0; s < t; ++s) y[k][i] = fmaf(Gs[row][SC_PLACE(s)], xs[SC_PLACE(s)][wave * 16 + col], y[k][i]);
          }
      } else {
        f32x4_s z[3];
#pragma unroll
        for (int u = 0; u < 3; ++u) {      // (tokens 0..15 of themselves; tokens 16..31 of these and of themselves)
          f32x4_s sum[2];
          const f32x4_s g4 = *(const f32x4_s*)&Gs[u > 0 ? 16 + col : col][u > 1 ? 16 + 4 * quad : 4 * quad];
#pragma unroll
          for (int i = 0; i < 4; ++i) sum[i % 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(g4[i], xv[u > 1][i], i < 2 ? (f32x4_s)(0.f) : sum[i % 2], 0, 0, 0);
          z[u] = sum[0] + sum[1];
        }
        z[1] += z[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const f32x4_s e = *(const f32x4_s*)&from_start[16 * k + 4 * quad];
#pragma unroll
          for (int i = 0; i < 4; ++i) y[k][i] = fmaf(y[k][i], e[i], z[k][i]);
        }
      }
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const f32x4_s own = *(const f32x4_s*)&diag[16 * k + 4 * quad];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int t = 16 * k + 4 * i + quad;
          const float v = fmaf(own[i], xv[k][i], y[k][i]);
          if (live && t0 + t < len) a.y[(size_t)(start + t0 + t) * inner + (size_t)h * P + p] = fmaf(Dh, xv[k][i], v);
        }
      }
    }
    if (!OUT || t0 + SC_T < len) {
      const float decay = from_start[SC_T - 1];
#pragma unroll
      for (int j = 0; j < NT; ++j) S[j] *= decay;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int s = 16 * k + 4 * quad + i;      // (its row)
          const float w = xv[k][i] * (to_end[s] * dts[s]);
#pragma unroll
          for (int j = 0; j < NT; ++j) S[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(Bs[s][16 * j + col], w, S[j], 0, 0, 0);
        }
      }
    }
  }
  if constexpr (!OUT) {
    if (live)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) state[(size_t)(16 * j + 4 * quad + i) * P + p] = S[j][i];
    if (slice == 0 && tid == 0) a.piece_decay[((size_t)r * a.heads + h) * a.max_pieces + pc] = dt_sum == 0.0 ? 1.f : expf((float)(A * dt_sum));
  }
}

// The carry between the passes: a thread owns one entry of a head's state and walks the pieces, four of them on their way at a time.
// Bound by memory (each piece's state is read and written once).
__global__ __launch_bounds__(256) void ssm_carry_kernel(ScanArgs a) {
  const size_t size = (size_t)a.n_state * a.head_dim;
  const int blocks = (int)((size + 255) / 256), r = blockIdx.x / blocks, h = blockIdx.y;
  const int run_len = a.cu_seqlens[r + 1] - a.cu_seqlens[r];
  const size_t e = (size_t)(blockIdx.x % blocks) * 256 + threadIdx.x;
  if (run_len <= 0 || e >= size) return;
  const int pieces = (run_len + a.piece - 1) / a.piece;
  float* S = a.state + (size_t)a.state_slots[r] * a.state_stride + a.state_off + (size_t)h * size + e;
  float* PS = a.piece_state + ((size_t)r * a.heads + h) * a.max_pieces * size + e;
  const float* PD = a.piece_decay + ((size_t)r * a.heads + h) * a.max_pieces;
  float cur = *S;
  for (int c0 = 0; c0 < pieces; c0 += 4) {
    float local[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) local[i] = c0 + i < pieces ? PS[(size_t)(c0 + i) * size] : 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (c0 + i < pieces) {
        PS[(size_t)(c0 + i) * size] = cur;
        cur = fmaf(PD[c0 + i], cur, local[i]);
      }
  }
  *S = cur;
}

// scratch floats a scan of n_req requests whose longest run has max_run tokens needs (0: it runs in one launch)
extern "C" size_t tp_ssm_scan_scratch(int n_req, int max_run, int heads, int head_dim, int n_state, int* piece_out) {
  int piece = 0;
  if (max_run > 256) {
    piece = 128;
    while ((max_run + piece - 1) / piece > 32) piece *= 2;    // at most 32 pieces a run
  }
  if (piece_out) *piece_out = piece;
  if (piece == 0) return 0;
  const size_t pieces = (size_t)((max_run + piece - 1) / piece);
  return (size_t)n_req * heads * pieces * ((size_t)n_state * head_dim + 1);
}

extern "C" int tp_ssm_scan(const float* xbc, const float* proj, int proj_stride, int dt_col0, const float* dt_bias,
                           const float* a_log, const float* d_skip, float* state, size_t state_stride, size_t state_off,
                           const int* cu_seqlens, const int* state_slots, float* y, int n_req, int heads, int head_dim,
                           int n_state, int groups, int max_run, float* scratch, size_t scratch_floats, hipStream_t s) {
  TP_REQUIRE(n_req >= 0 && heads > 0 && head_dim > 0 && n_state > 0 && groups > 0 && heads % groups == 0, "ssm_scan: bad sizes");
  TP_REQUIRE(n_state <= 2048, "ssm_scan: state size %d exceeds 2048", n_state);
  TP_REQUIRE(state_stride >= state_off + (size_t)heads * n_state * head_dim, "ssm_scan: state rows too short");
  TP_REQUIRE(heads <= 65535 && max_run >= 0, "ssm_scan: too many heads");
  if (n_req == 0) return 0;
  ScanArgs a;
  a.xbc = xbc; a.proj = proj; a.proj_stride = proj_stride; a.dt_col0 = dt_col0;
  a.dt_bias = dt_bias; a.a_log = a_log; a.d_skip = d_skip;
  a.state = state; a.state_stride = state_stride; a.state_off = state_off;
  a.cu_seqlens = cu_seqlens; a.state_slots = state_slots; a.y = y;
  a.heads = heads; a.head_dim = head_dim; a.n_state = n_state; a.groups = groups;
  a.channels = heads * head_dim + 2 * groups * n_state;
  // A thread holds TN state entries of TP value columns; the R lanes that share those columns split the state index.
  // Two columns a thread halve what a token's B and C cost in LDS reads for each update of the state; sixteen
  // entries a lane keep most of a wave's instructions the recurrence's own.  No more columns a block than the head has.
  const int TP = (head_dim >= 2 && n_state <= 1024) ? 2 : 1;
  const int cap = TP == 2 ? 16 : 32;
  int R = 1;
  while (R < 64 && R * cap < n_state) R *= 2;
  int pc_pow2 = 1;
  while (pc_pow2 < head_dim) pc_pow2 *= 2;
  while (R < 64 && (256 / R) * TP > pc_pow2) R *= 2;
  const int per_lane = (n_state + R - 1) / R;
  int tn = 1;
  while (tn < per_lane) tn *= 2;
  TP_REQUIRE(tn <= cap, "ssm_scan: state size %d does not fit a block", n_state);
  a.R = R;
  const int PC = (256 / R) * TP;
  const int per_token = 2 * R * tn + PC + 2;
  int TC = (32 * 1024 / 4) / per_token;
  TC = TC < 1 ? 1 : (TC > 64 ? 64 : TC);
  a.TC = TC;
  const size_t shmem = (size_t)TC * per_token * sizeof(float);
  const int slices = (head_dim + PC - 1) / PC;
  int piece = 0;
  const size_t need = tp_ssm_scan_scratch(n_req, max_run, heads, head_dim, n_state, &piece);
  a.piece = piece;
  a.max_pieces = piece ? (max_run + piece - 1) / piece : 1;
  a.piece_state = scratch;
  a.piece_decay = scratch ? scratch + (size_t)n_req * heads * a.max_pieces * n_state * head_dim : nullptr;
  TP_REQUIRE(piece == 0 || (scratch != nullptr && scratch_floats >= need), "ssm_scan: scratch of %zu floats needed", need);
  TP_REQUIRE((long)slices * a.max_pieces <= 65535, "ssm_scan: too many pieces");
#define SCAN_LAUNCH(TN_, TP_, GRID)                                                                     \
  do {                                                                                                  \
    if (max_run == 1) hipLaunchKernelGGL((ssm_step_kernel<TN_, TP_>), GRID, dim3(256), 0, s, a);        \
    else hipLaunchKernelGGL((ssm_scan_kernel<TN_, TP_>), GRID, dim3(256), shmem, s, a);                 \
  } while (0)
#define SCAN_DISPATCH(GRID)                                \
  do {                                                     \
    if (TP == 2) {                                         \
      if (tn == 1) SCAN_LAUNCH(1, 2, GRID);                \
      else if (tn == 2) SCAN_LAUNCH(2, 2, GRID);           \
      else if (tn == 4) SCAN_LAUNCH(4, 2, GRID);           \
      else if (tn == 8) SCAN_LAUNCH(8, 2, GRID);           \
      else SCAN_LAUNCH(16, 2, GRID);                       \
    } else {                                               \
      if (tn == 1) SCAN_LAUNCH(1, 1, GRID);                \
      else if (tn == 2) SCAN_LAUNCH(2, 1, GRID);           \
      else if (tn == 4) SCAN_LAUNCH(4, 1, GRID);           \
      else if (tn == 8) SCAN_LAUNCH(8, 1, GRID);           \
      else if (tn == 16) SCAN_LAUNCH(16, 1, GRID);         \
      else SCAN_LAUNCH(32, 1, GRID);                       \
    }                                                      \
  } while (0)
  if (piece == 0) {
    a.mode = SCAN_DIRECT;
    SCAN_DISPATCH(dim3(n_req, heads, slices));
  } else {
    // The matrix cores' form reads x, B and C in 16-byte pieces and has whole tiles of 16 columns and 16, 32, 64 or 128 state entries.
    const bool chunked = head_dim % 16 == 0 && (n_state == 16 || n_state == 32 || n_state == 64 || n_state == 128) &&
                         ((uintptr_t)xbc & 15) == 0;      // (then every column offset and the rows' stride are multiples of 16 floats)
    const size_t entries = (size_t)n_state * head_dim;
    const size_t carry_blocks = (entries + 255) / 256 * n_req;
    TP_REQUIRE(carry_blocks < 0x7fffffffUL, "ssm_scan: too many requests");
    a.unit = heads / groups;
    while (a.unit > 16 && a.unit % 2 == 0) a.unit /= 2;
    const long items = ((long)n_req * (heads / a.unit) * ((head_dim + SC_P - 1) / SC_P) * a.max_pieces + 7) / 8 * 8 * a.unit;
    const dim3 chunk_grid((unsigned)items);
    TP_REQUIRE(items < 0x7ffffff0L, "ssm_scan: too many pieces");
#define CHUNK_DISPATCH(OUT_)                                                                                                          \
  do {                                                                                                                                \
    if (n_state == 16) hipLaunchKernelGGL((ssm_chunk_kernel<1, OUT_>), chunk_grid, dim3(256), 0, s, a, n_req);                        \
    else if (n_state == 32) hipLaunchKernelGGL((ssm_chunk_kernel<2, OUT_>), chunk_grid, dim3(256), 0, s, a, n_req);                   \
    else if (n_state == 64) hipLaunchKernelGGL((ssm_chunk_kernel<4, OUT_>), chunk_grid, dim3(256), 0, s, a, n_req);                   \
    else hipLaunchKernelGGL((ssm_chunk_kernel<8, OUT_>), chunk_grid, dim3(256), 0, s, a, n_req);                                      \
  } while (0)
    a.mode = SCAN_LOCAL;
    if (chunked) CHUNK_DISPATCH(false);
    else SCAN_DISPATCH(dim3(n_req, heads, slices * a.max_pieces));
    hipLaunchKernelGGL(ssm_carry_kernel, dim3((unsigned)carry_blocks, heads), dim3(256), 0, s, a);
    a.mode = SCAN_OUTPUT;
    if (chunked) CHUNK_DISPATCH(true);
    else SCAN_DISPATCH(dim3(n_req, heads, slices * a.max_pieces));
#undef CHUNK_DISPATCH
  }
#undef SCAN_DISPATCH
#undef SCAN_LAUNCH
  TP_CHECK_LAUNCH("ssm_scan");
  return 0;
}

// ---- gate, grouped norm, weight ---------------------------------------------------------------
// v = y * silu(z) (z: column z_col0 + j of the projection's rows), normed in `groups` equal parts, each by its own
// root mean square (eps inside the root), times w [inner]; out [n, inner] float32 or bfloat16.
// One block per (token, part).
#define GN_ITEMS 8   // values a thread keeps between the sum and the store (parts up to 8 x the block)
template <typename TO>
__global__ void gated_group_norm_kernel(const float* __restrict__ y, const float* __restrict__ proj, int proj_stride,
                                        int z_col0, const float* __restrict__ w, float eps, TO* __restrict__ out, int inner,
                                        int part) {
  __shared__ float scratch[32];
  const int t = blockIdx.x, q = blockIdx.y;
  const float* yr = y + (size_t)t * inner + (size_t)q * part;
  const float* zr = proj + (size_t)t * proj_stride + z_col0 + (size_t)q * part;
  TO* o = out + (size_t)t * inner + (size_t)q * part;
  const float* wr = w + (size_t)q * part;
  if (part <= GN_ITEMS * (int)blockDim.x) {
    float v[GN_ITEMS];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < GN_ITEMS; ++i) {
      const int j = threadIdx.x + i * blockDim.x;
      v[i] = j < part ? yr[j] * silu_f(zr[j]) : 0.f;
      ss = fmaf(v[i], v[i], ss);
    }
    const float rstd = 1.0f / sqrtf(block_sum(ss, scratch) / (float)part + eps);
#pragma unroll
    for (int i = 0; i < GN_ITEMS; ++i) {
      const int j = threadIdx.x + i * blockDim.x;
      if (j < part) from_float(o + j, v[i] * rstd * wr[j]);
    }
    return;
  }
  float ss = 0.f;
  for (int j = threadIdx.x; j < part; j += blockDim.x) {
    const float v = yr[j] * silu_f(zr[j]);
    ss = fmaf(v, v, ss);
  }
  const float total = block_sum(ss, scratch);
  const float rstd = 1.0f / sqrtf(total / (float)part + eps);
  for (int j = threadIdx.x; j < part; j += blockDim.x) from_float(o + j, yr[j] * silu_f(zr[j]) * rstd * wr[j]);
}

// The same with a part of at most 4,096 in registers, a thread four neighbouring columns, all loads in front of the sum.
// 8,192 columns in eight parts, against loads of four bytes: one row 3.30 -> 2.27 us, 2,048 rows 50.5 -> 30.7 (5.4 TB/s).
template <typename TO, int T>
__global__ __launch_bounds__(T) void gated_group_norm4_kernel(const float* __restrict__ y, const float* __restrict__ proj, int proj_stride,
                                                                 int z_col0, const float* __restrict__ w, float eps, TO* __restrict__ out,
                                                                 int inner, int part) {
  __shared__ __attribute__((aligned(16))) float scratch[T / TP_WAVE];
  const int t = blockIdx.x, c = 4 * threadIdx.x;   // (T >= part / 4; a part of one wave sums without LDS)
  const size_t col = (size_t)blockIdx.y * part + c;
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f), z = v, wv = v;
  if (c < part) {
    v = *(const float4*)(y + (size_t)t * inner + col);
    z = *(const float4*)(proj + (size_t)t * proj_stride + z_col0 + col);
    wv = *(const float4*)(w + col);
  }
  v.x *= silu_f(z.x);
  v.y *= silu_f(z.y);
  v.z *= silu_f(z.z);
  v.w *= silu_f(z.w);
  const float ss = fmaf(v.w, v.w, fmaf(v.z, v.z, fmaf(v.y, v.y, v.x * v.x)));
  const float rstd = 1.0f / sqrtf(block_sum_once<T>(ss, scratch) / (float)part + eps);
  if (c < part) from_float4(out + (size_t)t * inner + col, v.x * rstd * wv.x, v.y * rstd * wv.y, v.z * rstd * wv.z, v.w * rstd * wv.w);
}

extern "C" int tp_gated_group_norm(const float* y, const float* proj, int proj_stride, int z_col0, const float* w, float eps,
                                   void* out, int out_dt, int n, int inner, int groups, hipStream_t s) {
  TP_REQUIRE(n >= 0 && inner > 0 && groups > 0 && inner % groups == 0 && groups <= 65535, "gated_group_norm: bad sizes");
  if (n == 0) return 0;
  const int part = inner / groups;
  const dim3 grid(n, groups);
  TP_REQUIRE(out_dt == TP_F32 || out_dt == TP_BF16, "gated_group_norm: unknown dtype %d", out_dt);
  // (a part of up to 64 columns leaves three quarters of a wave without work, and loads of four bytes are faster: 2,048 rows of 512 columns in
  // eight parts 6.4 us against 7.4, of 768 7.7 against 7.5.  Threads for as many columns as there are: 2,048 rows of 8,224 columns in eight parts
  // with 512 threads 42.7 us, with 1,024 65.5, by loads of four bytes 57.8; of 12,288 48.5, 69.3 and 65.0.)
  if (part % 4 == 0 && part > 64 && part <= 4096 && proj_stride % 4 == 0 && z_col0 % 4 == 0 &&
      (((uintptr_t)y | (uintptr_t)proj | (uintptr_t)w | (uintptr_t)out) & 15) == 0) {
#define GN4(T_)                                                                                                                                    \
  do {                                                                                                                                              \
    if (out_dt == TP_F32)                                                                                                                           \
      hipLaunchKernelGGL((gated_group_norm4_kernel<float, T_>), grid, dim3(T_), 0, s, y, proj, proj_stride, z_col0, w, eps, (float*)out, inner, part); \
    else                                                                                                                                            \
      hipLaunchKernelGGL((gated_group_norm4_kernel<bf16_t, T_>), grid, dim3(T_), 0, s, y, proj, proj_stride, z_col0, w, eps, (bf16_t*)out, inner, part); \
  } while (0)
    if (part <= 256) GN4(64);
    else if (part <= 1024) GN4(256);
    else if (part <= 2048) GN4(512);
    else GN4(1024);
#undef GN4
    TP_CHECK_LAUNCH("gated_group_norm");
    return 0;
  }
  const int threads = part >= 2048 ? 1024 : (part >= 256 ? 256 : 64);
  if (out_dt == TP_F32)
    hipLaunchKernelGGL(gated_group_norm_kernel<float>, grid, dim3(threads), 0, s, y, proj, proj_stride, z_col0, w, eps,
                       (float*)out, inner, part);
  else if (out_dt == TP_BF16)
    hipLaunchKernelGGL(gated_group_norm_kernel<bf16_t>, grid, dim3(threads), 0, s, y, proj, proj_stride, z_col0, w, eps,
                       (bf16_t*)out, inner, part);
  else
    TP_REQUIRE(false, "gated_group_norm: unknown dtype %d", out_dt);
  TP_CHECK_LAUNCH("gated_group_norm");
  return 0;
}
