// One token of a recurrent mixer: the work of a block of 512 threads on one request's head (see step_mixers.hip).  In a header for the
// launches that run it alone and beside other blocks.
#pragma once
#include <math.h>

#include "column_sum.h"
#include "common.h"

__device__ inline float s_sigmoid(float v) { return 1.0f / (1.0f + expf(-v)); }
__device__ inline float s_softplus(float v) { return fmaxf(v, 0.f) + log1pf(expf(-fabsf(v))); }
__device__ inline float s_silu(float v) { return v / (1.0f + expf(-v)); }

enum { STEP_DELTA = 0, STEP_GENERAL = 1, STEP_LINEAR = 2 };

struct LowRank {          // f(g(x) wt): see lowrank_up_kernel for the modes
  const float* x;         // first column of the inner rows, or nullptr
  const float* wt;        // [rank, columns]
  const float* a_log;
  const float* bias;
  int rank, columns, mode, in_act;
  float rate;
};

struct StepArgs {
  const float *q, *k, *v, *a;          // first columns of the rows (delta: of the convolution's inputs; a: general's raw removal rates)
  const float *beta, *a_bias, *bonus;  // delta's raw beta; general's rate biases; linear's bonus (nullptr: read behind the update)
  const float* conv_w;                 // [taps, channels] over q | k | v of all heads
  LowRank decay, gate_lr;
  const float* gate;                   // raw gate rows (nullptr: gate_lr's)
  const float* norm_w;
  float* state;
  const int *token_req, *state_slots;
  void* out;
  size_t q_stride, k_stride, v_stride, x_stride, gate_stride, state_stride, state_off, conv_off, out_stride;
  int out_col0, heads, dim, vdim, taps, gate_act, norm_stride;
  float q_scale, unit_eps, norm_eps, scale;
};

// a step written down for a launch that runs it beside other blocks
struct PreparedStep {
  StepArgs args;
  int kind, n;
};

// what the low-rank product of one column becomes (the modes of lowrank_up)
__device__ inline float step_lowrank_f(const LowRank& l, float v, float a_log, float b) {
  if (l.mode == 0) return v;
  if (l.mode == 1) return s_sigmoid(v);
  if (l.mode == 2) return expf(-expf(a_log) * s_softplus(v + b));
  if (l.mode == 3) return expf(-l.rate * s_sigmoid(v + b));
  if (l.mode == 4) return expf(-expf(v + b));
  return expf(-l.rate * s_softplus(-(v + b)));
}

// what the waves exchange here lies in LDS: __syncthreads would wait for the state on its way as well
#define STEP_BARRIER()                                  \
  do {                                                  \
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); \
    __builtin_amdgcn_s_barrier();                       \
    asm volatile("" ::: "memory");                      \
  } while (0)

// t: the token's row, h: the head
template <int KIND, int KS, typename TO>
__device__ inline void mixer_step_block(const StepArgs& a, int t, int h) {
  constexpr int PER = 8, C = 512 / KS, NP = 128 / C;   // columns a pass, passes over up to 128 columns
  __shared__ __attribute__((aligned(16))) float qs[128], kk[128], ws[128], us[128], as[128];
  __shared__ __attribute__((aligned(16))) float vs[128], gs[128], ys[128];
  __shared__ __attribute__((aligned(16))) float xa[128], xg[128];
  __shared__ float part[4][256];
  __shared__ float dots[2];
  const int tid = threadIdx.x, lane = tid % TP_WAVE;
  const int ks = tid % KS, jl = tid / KS;
  const int dim = a.dim, vdim = a.vdim;
  constexpr bool LR_GATE = KIND == STEP_DELTA;      // the gate comes from a low-rank product of its own, not as raw columns
  // ---- everything that depends on no other load is requested before anything is waited for: in a decode step nothing of this
  // is in a cache near the CU, and each trip that starts only behind a barrier would add its whole latency.  No load stands behind a condition
  // (places are clamped, values past the end replaced where they are used): at a join behind one, and at a store into the state in front of
  // a load from it, all loads on their way are waited for.
  const int req = a.token_req[t];
  // low-rank products: column tid % 256 (decay, then gate), its sum in eight shares of the rank, half of them a thread
  const int lr = tid % 256, lc = lr % 128;
  const int part_of = __builtin_amdgcn_readfirstlane(tid / 128), half = part_of / 2;
  const bool to_gate = LR_GATE && (part_of & 1);
  const LowRank& l = to_gate ? a.gate_lr : a.decay;
  const int lwidth = to_gate ? vdim : dim, lat = min(lc, lwidth - 1);
  const bool have = (LR_GATE || lr < 128) && lc < lwidth;
  const float* wt = l.wt + (size_t)h * lwidth;      // (one for the wave; the lane's column is an offset)
  // the head's inputs.  Thread c: element c % 128 of q, k, v or (general) the removal rates
  const int i = tid % 128;
  const int width = part_of == 2 || (part_of == 3 && KIND != STEP_GENERAL) ? vdim : dim;
  const size_t col = (size_t)h * width + min(i, width - 1);
  const float* in = part_of == 0 ? a.q + (size_t)t * a.q_stride : part_of == 1 ? a.k + (size_t)t * a.k_stride
                    : part_of == 3 && KIND == STEP_GENERAL ? a.a + (size_t)t * a.q_stride : a.v + (size_t)t * a.v_stride;
  float elem = in[col];
  const float inner = l.x[(size_t)t * a.x_stride + min(lc, l.rank - 1)];
  float cw[4];
  size_t ch = 0;
  const int channels = 2 * a.heads * dim + a.heads * vdim;
  if constexpr (KIND == STEP_DELTA) {
    ch = (size_t)min(part_of, 2) * a.heads * dim + col;
#pragma unroll
    for (int j = 0; j < 4; ++j) cw[j] = a.conv_w[(size_t)min(j, a.taps - 1) * channels + ch];
  }
  const int slot = a.state_slots[req];
  float lw[2][4][4];       // the first 64 of the rank
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int d = 0; d < 4; ++d) lw[b][p][d] = (wt + (size_t)min(b * 32 + (half * 4 + p) * 4 + d, l.rank - 1) * l.columns)[lat];
  const float lb = a.decay.bias[(size_t)h * dim + min(lc, dim - 1)];
  const float la = KIND == STEP_DELTA ? a.decay.a_log[h] : 0.f;
  float* st = a.state + (size_t)slot * a.state_stride;
  float* S_mem = st + a.state_off + (size_t)h * a.vdim * a.dim;
  float* cs = a.taps > 1 ? st + a.conv_off + ch : S_mem;
  float carried[3];
  if constexpr (KIND == STEP_DELTA) {
#pragma unroll
    for (int j = 0; j < 3; ++j) carried[j] = cs[(size_t)max(0, min(j, a.taps - 2)) * channels];
  }
  float S[NP][PER];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int j = p * C + jl;
#pragma unroll
    for (int e4 = 0; e4 < PER / 4; ++e4) {
      const float4 f = *(const float4*)(S_mem + (size_t)min(j, vdim - 1) * dim + min(ks * PER + e4 * 4, dim - 4));
      S[p][e4 * 4] = f.x; S[p][e4 * 4 + 1] = f.y; S[p][e4 * 4 + 2] = f.z; S[p][e4 * 4 + 3] = f.w;
    }
  }
  // what the end of the step needs: the norm's weights and the gate, four elements of the first lanes; the bonus
  int group = 1;
  while (group < 64 && group * 4 < vdim) group *= 2;
  const int d4 = lane % group * 4;
  const float4 wv = *(const float4*)(a.norm_w + (size_t)h * a.norm_stride + min(d4, vdim - 4));
  float4 gv = make_float4(1.f, 1.f, 1.f, 1.f);
  if constexpr (!LR_GATE) gv = *(const float4*)(a.gate + (size_t)t * a.gate_stride + (size_t)h * vdim + min(d4, vdim - 4));
  const float beta_raw = KIND == STEP_DELTA ? a.beta[(size_t)t * a.x_stride + h] : 0.f;
  float rate_bias[2];
  if constexpr (KIND == STEP_GENERAL) {
#pragma unroll
    for (int e = 0; e < 2; ++e) rate_bias[e] = a.a_bias[(size_t)h * dim + min(lane + e * TP_WAVE, dim - 1)];
  }
  float bonus[PER];
  if constexpr (KIND == STEP_LINEAR) {
    const float* from = (a.bonus != nullptr ? a.bonus : a.decay.bias) + (size_t)h * dim;      // (without a bonus: not used)
#pragma unroll
    for (int e = 0; e < PER; ++e) bonus[e] = from[min(ks * PER + e, dim - 1)];
  }
  // ---- the head's inputs, on their way above
  {
    if constexpr (KIND == STEP_DELTA) {
      if (part_of < 3 && i < width) {
        float acc = 0.f;
        if (a.taps <= 4) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            if (j >= a.taps) break;
            const float y = j < 3 && j < a.taps - 1 ? carried[j < 3 ? j : 0] : elem;
            if (j > 0) cs[(size_t)(j - 1) * channels] = y;
            acc = fmaf(cw[j], y, acc);
          }
        } else {
          for (int j = 0; j < a.taps; ++j) {
            const float y = j < a.taps - 1 ? cs[(size_t)j * channels] : elem;
            if (j > 0) cs[(size_t)(j - 1) * channels] = y;
            acc = fmaf(a.conv_w[(size_t)j * channels + ch], y, acc);
          }
        }
        elem = s_silu(acc);
      }
    }
    if (KIND == STEP_LINEAR && part_of == 0) elem *= a.q_scale;
    if (i >= width) elem = 0.f;
    if (part_of == 0) qs[i] = elem;
    else if (part_of == 1) kk[i] = elem;
    else if (part_of == 2) vs[i] = elem;
    else as[i] = elem;
    const float y = lc < l.rank ? inner : 0.f;
    if (tid < 128) xa[lc] = a.decay.in_act ? tanhf(y) : y;
    else if (LR_GATE && tid < 256) xg[lc] = y;
  }
  STEP_BARRIER();
  // ---- low-rank products
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  if (have) {
    const float* xs = lr < 128 ? xa : xg;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const int e = b * 32 + (half * 4 + p) * 4 + d;
          acc[p] = fmaf(xs[e], e < l.rank ? lw[b][p][d] : 0.f, acc[p]);
        }
    for (int i0 = 64; i0 < l.rank; i0 += 32) {
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const int i = i0 + (half * 4 + p) * 4;
#pragma unroll
        for (int d = 0; d < 4; ++d) acc[p] = fmaf(xs[i + d], i + d < l.rank ? wt[(size_t)(i + d) * l.columns + lat] : 0.f, acc[p]);
      }
    }
    if (half == 1)
#pragma unroll
      for (int p = 0; p < 4; ++p) part[p][lr] = acc[p];
  }
  // (the last wave, beside the products above: unit vectors and the dot products that do not need the state)
  if (KIND != STEP_LINEAR && tid >= 448) {
    if (KIND == STEP_DELTA) {
      float sq = 0.f, sk = 0.f;
      for (int i = lane; i < dim; i += TP_WAVE) {
        sq = fmaf(qs[i], qs[i], sq);
        sk = fmaf(kk[i], kk[i], sk);
      }
      sq = wave_sum(sq);
      sk = wave_sum(sk);
      const float rq = a.q_scale / sqrtf(sq + a.unit_eps), rk = 1.0f / sqrtf(sk + a.unit_eps);
      float dot = 0.f;
      for (int i = lane; i < dim; i += TP_WAVE) {
        const float qv = qs[i] * rq, kv = kk[i] * rk;
        qs[i] = qv;
        kk[i] = kv;
        dot = fmaf(qv, kv, dot);
      }
      dot = wave_sum(dot);
      if (lane == 0) dots[0] = dot;
    } else {
      float sk = 0.f;
      for (int i = lane; i < dim; i += TP_WAVE) sk = fmaf(kk[i], kk[i], sk);
      sk = wave_sum(sk);
      const float rk = 1.0f / sqrtf(sk + a.unit_eps);
      float d1 = 0.f, d2 = 0.f;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int i = lane + e * TP_WAVE;
        const float u = i < dim ? kk[i] * rk : 0.f;
        const float au = i < dim ? s_sigmoid(as[i] + rate_bias[e]) * u : 0.f;
        us[i] = u;
        as[i] = au;
        if (i < dim) {
          d1 = fmaf(au, qs[i], d1);
          d2 = fmaf(kk[i], qs[i], d2);
        }
      }
      d1 = wave_sum(d1);
      d2 = wave_sum(d2);
      if (lane == 0) {
        dots[0] = d1;
        dots[1] = d2;
      }
    }
  }
  STEP_BARRIER();
  if (half == 0) {
    float v = 0.f;
#pragma unroll
    for (int p = 0; p < 4; ++p) v += acc[p];
    if (have) {
#pragma unroll
      for (int p = 0; p < 4; ++p) v += part[p][lr];
      v = step_lowrank_f(l, v, la, lb);
    } else {
      v = 1.f;             // (a key channel past the last one decays nothing)
    }
    if (lr < 128) ws[lc] = v;
    else gs[lc] = v;
  }
  STEP_BARRIER();
  // ---- the step
#pragma unroll
  for (int p = 0; p < NP; ++p)
#pragma unroll
    for (int e = 0; e < PER; ++e)
      if (p * C + jl >= vdim || ks * PER + e >= dim) S[p][e] = 0.f;
  const float beta = KIND == STEP_DELTA ? s_sigmoid(beta_raw) : 0.f;
  const int o8 = ks * PER;
  float qa[PER], ka[PER], wa[PER], ua[PER], aa[PER];
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    qa[e] = qs[o8 + e];
    ka[e] = kk[o8 + e];
    wa[e] = ws[o8 + e];
    if (KIND == STEP_GENERAL) {
      ua[e] = us[o8 + e];
      aa[e] = as[o8 + e];
    } else if (KIND == STEP_LINEAR) {
      ua[e] = o8 + e < dim ? bonus[e] : 0.f;
    }
  }
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int j = p * C + jl;
    const float v = vs[j];
    float y;
    if (KIND == STEP_DELTA) {
      float pred[2], read[2];
#pragma unroll
      for (int e4 = 0; e4 < 2; ++e4) {
        float pv = 0.f, rd = 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int e = e4 * 4 + c;
          S[p][e] *= wa[e];
          pv = fmaf(S[p][e], ka[e], pv);
          rd = fmaf(S[p][e], qa[e], rd);
        }
        pred[e4] = pv;
        read[e4] = rd;
      }
      const float ps = column_sum<KS>(pred[0] + pred[1]), rs = column_sum<KS>(read[0] + read[1]);
      const float u = beta * (v - ps);
#pragma unroll
      for (int e = 0; e < PER; ++e) S[p][e] = fmaf(ka[e], u, S[p][e]);
      y = fmaf(u, dots[0], rs);
    } else if (KIND == STEP_GENERAL) {
      float seen = 0.f, read = 0.f;
#pragma unroll
      for (int e = 0; e < PER; ++e) {
        seen = fmaf(S[p][e], ua[e], seen);   // (the old state)
        S[p][e] *= wa[e];
        read = fmaf(S[p][e], qa[e], read);
      }
      seen = column_sum<KS>(seen);
      read = column_sum<KS>(read);
#pragma unroll
      for (int e = 0; e < PER; ++e) S[p][e] = fmaf(ka[e], v, fmaf(-aa[e], seen, S[p][e]));
      y = fmaf(dots[1], v, fmaf(-dots[0], seen, read));
    } else {
      float read = 0.f, own = 0.f;
#pragma unroll
      for (int e = 0; e < PER; ++e) {
        if (a.bonus != nullptr) {
          own = fmaf(ua[e] * ka[e], qa[e], own);
          read = fmaf(S[p][e], qa[e], read);   // (the state as the token before left it)
        }
        S[p][e] = fmaf(wa[e], S[p][e], ka[e] * v);
        if (a.bonus == nullptr) read = fmaf(S[p][e], qa[e], read);
      }
      if (a.bonus != nullptr) read = fmaf(own, v, read);
      y = column_sum<KS>(read);
    }
    if (ks == 0) ys[j] = y;
#pragma unroll
    for (int e4 = 0; e4 < 2; ++e4) {
      const int i = o8 + e4 * 4;
      if (j < vdim && i < dim) *(float4*)(S_mem + (size_t)j * dim + i) = make_float4(S[p][e4 * 4], S[p][e4 * 4 + 1], S[p][e4 * 4 + 2], S[p][e4 * 4 + 3]);
    }
  }
  STEP_BARRIER();
  // ---- norm and gate: four elements a lane, `group` lanes
  if (tid >= TP_WAVE) return;
  const float4 x = d4 < vdim ? *(const float4*)(ys + d4) : make_float4(0.f, 0.f, 0.f, 0.f);
  float ss = 0.f;
  ss = fmaf(x.x, x.x, ss);
  ss = fmaf(x.y, x.y, ss);
  ss = fmaf(x.z, x.z, ss);
  ss = fmaf(x.w, x.w, ss);
  ss = lanes_sum_of(ss, group);
  if (lane >= group || d4 >= vdim) return;
  const float rstd = 1.0f / sqrtf(ss / (float)vdim + a.norm_eps);
  float v[4] = {x.x * rstd * wv.x, x.y * rstd * wv.y, x.z * rstd * wv.z, x.w * rstd * wv.w};
  float4 g = gv;
  if constexpr (!LR_GATE) {
    if (a.gate_act == 2) g = make_float4(g.x * s_sigmoid(g.x), g.y * s_sigmoid(g.y), g.z * s_sigmoid(g.z), g.w * s_sigmoid(g.w));
    else g = make_float4(s_sigmoid(g.x), s_sigmoid(g.y), s_sigmoid(g.z), s_sigmoid(g.w));
  } else {
    g = *(const float4*)(gs + d4);
  }
  from_float4((TO*)a.out + (size_t)t * a.out_stride + a.out_col0 + (size_t)h * vdim + d4, v[0] * g.x * a.scale, v[1] * g.y * a.scale,
              v[2] * g.z * a.scale, v[3] * g.w * a.scale);
}
