// The gated delta rule token by token: what the kernels of delta.hip and delta_chunks.hip share.
#pragma once
#include <math.h>

#include "common.h"
#include "column_sum.h"

__device__ inline float d_sigmoid(float v) { return 1.0f / (1.0f + expf(-v)); }

// Per head h (its q and k are those of key head h / (heads / kv_heads)), with q and k made unit vectors
// (x / sqrt(sum x^2 + unit_eps); q also times q_scale), beta = sigmoid(beta_raw) and a decay g per key channel:
//   S <- g * S (rows are key channels);  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q.
// With P = (g * S_old)^T k and R = (g * S_old)^T q the read-out is o = R + u (k . q), so one pass over a thread's
// state entries forms both sums, one reduction over the lanes that share a column adds them, and a second pass
// writes k u^T.
//
// qkv [n, row_stride] float32 holds, per token, q [kv_heads * dim] | k [kv_heads * dim] | v [heads * vdim] (after the
// convolution and its activation); decay [n, heads * dim]; beta_raw is column beta_col0 + h of `proj`.
//
// First, all tokens side by side, a wave per token and key head: q and k become unit vectors in place, and k . q per
// token and key head is left (delta_unit_rows).  Then the chain (delta_chain): a block owns one request, one head and
// CB = 256 / KS value columns; a thread holds PER consecutive key channels of one column in registers, and the KS
// neighbouring lanes that share a column split the key channels among them (their sums meet by row permutes, no
// trip through LDS up to 16 lanes).  A wave has one instruction stream, so the time of a token is the number of
// instructions a wave issues for it: few state entries a lane (8 up to a key size of 128) keep that near 60.
// Tokens are taken TC at a time through LDS (rows padded to KS * PER channels with q = k = 0 and decay 1, so the
// run itself needs no bounds); the next chunk's values travel from memory into registers while this chunk runs.
struct DeltaArgs {
  float* qkv;
  int row_stride;
  const float* decay;
  const float* proj;
  int proj_stride, beta_col0;
  float* state;
  size_t state_stride, state_off;
  const int* cu_seqlens;
  const int* state_slots;
  float* y;
  float* kq;   // [n, kv_heads]
  int heads, kv_heads, dim, vdim;
  float q_scale, unit_eps;
};

// Token t's q and k of key head g become unit vectors in place, k . q goes to kq: a wave's work.
__device__ inline void delta_unit_rows(const DeltaArgs& a, long t, int g, int lane) {
  float* q = a.qkv + (size_t)t * a.row_stride + (size_t)g * a.dim;
  float* k = q + (size_t)a.kv_heads * a.dim;
  float sq = 0.f, sk = 0.f;
  for (int i = lane; i < a.dim; i += TP_WAVE) {
    sq = fmaf(q[i], q[i], sq);
    sk = fmaf(k[i], k[i], sk);
  }
  sq = wave_sum(sq);
  sk = wave_sum(sk);
  const float rq = a.q_scale / sqrtf(sq + a.unit_eps), rk = 1.0f / sqrtf(sk + a.unit_eps);
  float dot = 0.f;
  for (int i = lane; i < a.dim; i += TP_WAVE) {
    const float qv = q[i] * rq, kv = k[i] * rk;
    q[i] = qv;
    k[i] = kv;
    dot = fmaf(qv, kv, dot);
  }
  dot = wave_sum(dot);
  if (lane == 0) a.kq[t * a.kv_heads + g] = dot;
}

// One run of one head, the z-th block of its value columns: a block's work.
template <int PER, int KS>
__device__ inline void delta_chain(const DeltaArgs& a, int r, int h, int z) {
  constexpr int DP = PER * KS, CW = TP_WAVE / KS, CB = 4 * CW;
  constexpr int TC = DP <= 256 ? 16 : 4096 / DP;
  constexpr int NI = (TC * DP + 255) / 256, NV = (TC * CB + 255) / 256;
  __shared__ __attribute__((aligned(16))) float qs[TC * DP];
  __shared__ __attribute__((aligned(16))) float kk[TC * DP];
  __shared__ __attribute__((aligned(16))) float gs[TC * DP];
  __shared__ float vs[TC * CB];
  __shared__ float bs[TC];
  __shared__ float kqs[TC];
  const int start = a.cu_seqlens[r], len = a.cu_seqlens[r + 1] - start;
  if (len <= 0) return;
  const int tid = threadIdx.x, wave = tid / TP_WAVE, lane = tid % TP_WAVE;
  const int ks = lane % KS, jl = wave * CW + lane / KS;
  const int j = z * CB + jl;
  const bool col_ok = j < a.vdim;
  const int kvh = h / (a.heads / a.kv_heads);

  // a head's state lies in memory column by column, [vdim][dim]: the key channels of one value column are
  // neighbours, so a lane's entries are one or two 16-byte pieces and a wave's columns one contiguous run
  float* S_mem = a.state + (size_t)a.state_slots[r] * a.state_stride + a.state_off + ((size_t)h * a.vdim + (col_ok ? j : 0)) * a.dim;
  const bool vec = a.dim % 4 == 0 && ((uintptr_t)S_mem % 16) == 0;
  float S[PER];
#pragma unroll
  for (int e4 = 0; e4 < PER / 4; ++e4) {
    const int i = ks * PER + e4 * 4;
    if (vec && col_ok && i < a.dim) {
      const float4 v = *(const float4*)(S_mem + i);
      S[e4 * 4 + 0] = v.x; S[e4 * 4 + 1] = v.y; S[e4 * 4 + 2] = v.z; S[e4 * 4 + 3] = v.w;
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c) S[e4 * 4 + c] = (col_ok && i + c < a.dim) ? S_mem[i + c] : 0.f;
    }
  }
  const int q_col = kvh * a.dim, k_col = (a.kv_heads + kvh) * a.dim, v_col = 2 * a.kv_heads * a.dim + h * a.vdim;
  const int out_width = a.heads * a.vdim;
  const size_t decay_stride = (size_t)a.heads * a.dim;

  float rq[NI], rk[NI], rg[NI], rv[NV], rb = 0.f, rkq = 0.f;
  auto fetch = [&](int t0) {
#pragma unroll
    for (int it = 0; it < NI; ++it) {
      const int idx = it * 256 + tid;
      const int t = idx / DP, i = idx % DP;
      const bool in = idx < TC * DP && t0 + t < len && i < a.dim;
      const size_t row = (size_t)(start + t0 + t);
      rq[it] = in ? a.qkv[row * a.row_stride + q_col + i] : 0.f;
      rk[it] = in ? a.qkv[row * a.row_stride + k_col + i] : 0.f;
      rg[it] = in ? a.decay[row * decay_stride + (size_t)h * a.dim + i] : 1.f;
    }
#pragma unroll
    for (int it = 0; it < NV; ++it) {
      const int idx = it * 256 + tid;
      const int t = idx / CB, c = idx % CB;
      const int col = z * CB + c;
      rv[it] = (idx < TC * CB && t0 + t < len && col < a.vdim) ? a.qkv[(size_t)(start + t0 + t) * a.row_stride + v_col + col] : 0.f;
    }
    if (tid < TC && t0 + tid < len) {
      const size_t row = (size_t)(start + t0 + tid);
      rb = d_sigmoid(a.proj[row * a.proj_stride + a.beta_col0 + h]);
      rkq = a.kq[row * a.kv_heads + kvh];
    }
  };
  struct Tok {
    float4 q[PER / 4], k[PER / 4], g[PER / 4];
    float b, v, kq;
  };
  auto take = [&](Tok& x, int t) {
    const float4* q4 = (const float4*)(qs + t * DP + ks * PER);
    const float4* k4 = (const float4*)(kk + t * DP + ks * PER);
    const float4* g4 = (const float4*)(gs + t * DP + ks * PER);
#pragma unroll
    for (int e4 = 0; e4 < PER / 4; ++e4) {
      x.q[e4] = q4[e4];
      x.k[e4] = k4[e4];
      x.g[e4] = g4[e4];
    }
    x.b = bs[t];
    x.v = vs[t * CB + jl];
    x.kq = kqs[t];
  };
  auto step = [&](const Tok& x, int t_run) {
    float pred[PER / 4], read[PER / 4];
#pragma unroll
    for (int e4 = 0; e4 < PER / 4; ++e4) {
      const float qa[4] = {x.q[e4].x, x.q[e4].y, x.q[e4].z, x.q[e4].w}, ka[4] = {x.k[e4].x, x.k[e4].y, x.k[e4].z, x.k[e4].w},
                  ga[4] = {x.g[e4].x, x.g[e4].y, x.g[e4].z, x.g[e4].w};
      float p = 0.f, rd = 0.f;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int e = e4 * 4 + c;
        S[e] *= ga[c];
        p = fmaf(S[e], ka[c], p);
        rd = fmaf(S[e], qa[c], rd);
      }
      pred[e4] = p;
      read[e4] = rd;
    }
    float ps = pred[0], rs = read[0];
#pragma unroll
    for (int e4 = 1; e4 < PER / 4; ++e4) {   // (a fixed order: the same sums wherever the token stands)
      ps += pred[e4];
      rs += read[e4];
    }
    ps = column_sum<KS>(ps);
    rs = column_sum<KS>(rs);
    const float u = x.b * (x.v - ps);
#pragma unroll
    for (int e4 = 0; e4 < PER / 4; ++e4) {
      S[e4 * 4 + 0] = fmaf(x.k[e4].x, u, S[e4 * 4 + 0]);
      S[e4 * 4 + 1] = fmaf(x.k[e4].y, u, S[e4 * 4 + 1]);
      S[e4 * 4 + 2] = fmaf(x.k[e4].z, u, S[e4 * 4 + 2]);
      S[e4 * 4 + 3] = fmaf(x.k[e4].w, u, S[e4 * 4 + 3]);
    }
    if (ks == 0 && col_ok) a.y[(size_t)(start + t_run) * out_width + (size_t)h * a.vdim + j] = fmaf(u, x.kq, rs);
  };
  fetch(0);
  for (int t0 = 0; t0 < len; t0 += TC) {
    const int tc = min(TC, len - t0);
    __syncthreads();   // the chunk before has been consumed
#pragma unroll
    for (int it = 0; it < NI; ++it) {
      const int idx = it * 256 + tid;
      if (idx < TC * DP) {
        qs[idx] = rq[it];
        kk[idx] = rk[it];
        gs[idx] = rg[it];
      }
    }
#pragma unroll
    for (int it = 0; it < NV; ++it) {
      const int idx = it * 256 + tid;
      if (idx < TC * CB) vs[idx] = rv[it];
    }
    if (tid < TC) {
      bs[tid] = rb;
      kqs[tid] = rkq;
    }
    __syncthreads();
    if (t0 + TC < len) fetch(t0 + TC);   // on its way while this chunk runs
    // two tokens a turn, each token's LDS reads issued before the token ahead of it is worked on: a wave issues in
    // order, and reads that start only when the chain reaches them would add their whole latency to every token
    Tok A, B;
    take(A, 0);
    for (int t = 0; t < tc; t += 2) {
      if (t + 1 < tc) take(B, t + 1);
      step(A, t0 + t);
      if (t + 1 < tc) {
        if (t + 2 < tc) take(A, t + 2);
        step(B, t0 + t + 1);
      }
    }
  }
#pragma unroll
  for (int e4 = 0; e4 < PER / 4; ++e4) {
    const int i = ks * PER + e4 * 4;
    if (vec && col_ok && i < a.dim) {
      *(float4*)(S_mem + i) = make_float4(S[e4 * 4 + 0], S[e4 * 4 + 1], S[e4 * 4 + 2], S[e4 * 4 + 3]);
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (col_ok && i + c < a.dim) S_mem[i + c] = S[e4 * 4 + c];
    }
  }
}
