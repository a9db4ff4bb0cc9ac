// One decoded token a request through a whole recurrent mixer: everything between the input product and the output product of a
// gated delta rule, a generalized delta rule or a linear recurrence in one launch.
//
// Each of those mixers is, for a prompt, three to six kernels over all tokens (convolution, low-rank decay and gate, unit keys, the
// chain, the norm per head with its gate).  For one token a head each of them is a launch and a dependent trip to memory of 2 to 3 us
// around a few hundred bytes, and only the state (64 KB for a head of 128 x 128) is worth a memory system.  Here a block of 512
// threads owns one request and one head: it requests its state first (32 entries a thread), works out the head's inputs from LDS
// while those loads travel, takes the step, norms its own read-out and writes the output columns.  It needs every head's inputs to be
// its own: as many key heads as heads, keys of 33 to 128 and values of up to 128 elements, ranks of up to 128.
// Sums are formed in the order of the kernels that serve runs of tokens (delta.hip, general_delta.hip, linear_scan.hip): the same bits up
// to 64 requests (of more rows tp_lowrank_up adds its products in ascending order, here as of up to 64 in eight shares).
// Bound by those dependent trips up to a block a CU, by the state's 128 KB a head (read and written) beyond.  Gated delta rule, a
// captured chain, separate kernels / one launch: 16 heads of 128 x 128, one request 17.8 / 8.8 us, four 19.2 / 9.4; 32 heads, eight
// requests 26 / 14 us, 64 requests 85 / 68 us.  (At 128 registers a thread, two blocks a CU: 136 without the bound are 0.3 us less
// for one request and 20 us more for 64.)
#include <math.h>

#include "common.h"
#include "column_sum.h"

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

// what the low-rank product of one column becomes (the modes of lowrank_up)
__device__ inline float step_lowrank_f(const LowRank& l, float v, float a_log, float b) {
  if (l.mode == 0) return v;
  if (l.mode == 1) return s_sigmoid(v);
  if (l.mode == 2) return expf(-expf(a_log) * s_softplus(v + b));
  if (l.mode == 3) return expf(-l.rate * s_sigmoid(v + b));
  if (l.mode == 4) return expf(-expf(v + b));
  return expf(-l.rate * s_softplus(-(v + b)));
}

template <int KIND, int KS, typename TO>
__global__ __launch_bounds__(512, 4) void mixer_step_kernel(StepArgs a) {
  constexpr int PER = 8, C = 512 / KS, NP = 128 / C;   // columns a pass, passes over up to 128 columns
  __shared__ __attribute__((aligned(16))) float qs[128], kk[128], ws[128], us[128], as[128];
  __shared__ __attribute__((aligned(16))) float vs[128], gs[128], ys[128];
  __shared__ __attribute__((aligned(16))) float xa[128], xg[128];
  __shared__ float part[4][256];
  __shared__ float dots[2];
  const int t = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid % TP_WAVE;
  const int ks = tid % KS, jl = tid / KS;
  const int dim = a.dim, vdim = a.vdim;
  // ---- everything that depends on no other load is requested before anything is waited for: in a decode step nothing of this
  // is in a cache near the CU, and each trip that starts only behind a barrier would add its whole latency
  // low-rank products: column tid % 256 (decay, then gate), its sum in eight shares of the rank, half of them a thread
  const int lr = tid % 256, half = tid / 256, lc = lr % 128;
  const LowRank& l = lr < 128 ? a.decay : a.gate_lr;
  const bool have = l.x != nullptr && lc < (lr < 128 ? dim : vdim);
  const int lcol = h * (lr < 128 ? dim : vdim) + lc;
  const float* wt = l.wt + lcol;
  float lw[2][4][4];       // the first 64 of the rank
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const int i = b * 32 + (half * 4 + p) * 4 + d;
        lw[b][p][d] = have && i < l.rank ? wt[(size_t)i * l.columns] : 0.f;
      }
  float lb = 0.f, la = 0.f;
  if (have && half == 0 && l.mode >= 2) {
    lb = l.bias[lcol];
    if (l.mode == 2) la = l.a_log[lcol / dim];
  }
  float* st = a.state + (size_t)a.state_slots[a.token_req[t]] * a.state_stride;
  float* S_mem = st + a.state_off + (size_t)h * a.vdim * a.dim;
  float S[NP][PER];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int j = p * C + jl;
#pragma unroll
    for (int e4 = 0; e4 < PER / 4; ++e4) {
      const int i = ks * PER + e4 * 4;
      const float4 f = j < a.vdim && i < a.dim ? *(const float4*)(S_mem + (size_t)j * a.dim + i) : make_float4(0.f, 0.f, 0.f, 0.f);
      S[p][e4 * 4] = f.x; S[p][e4 * 4 + 1] = f.y; S[p][e4 * 4 + 2] = f.z; S[p][e4 * 4 + 3] = f.w;
    }
  }
  // what the end of the step needs: the norm's weights and the gate, four elements of the first lanes; the bonus
  int group = 1;
  while (group < 64 && group * 4 < vdim) group *= 2;
  const int d4 = lane % group * 4;
  float4 wv = make_float4(0.f, 0.f, 0.f, 0.f), gv = make_float4(1.f, 1.f, 1.f, 1.f);
  if (tid < TP_WAVE && d4 < vdim) {
    wv = *(const float4*)(a.norm_w + (size_t)h * a.norm_stride + d4);
    if (a.gate != nullptr) gv = *(const float4*)(a.gate + (size_t)t * a.gate_stride + (size_t)h * vdim + d4);
  }
  const float beta_raw = KIND == STEP_DELTA ? a.beta[(size_t)t * a.x_stride + h] : 0.f;
  float bonus[PER];
#pragma unroll
  for (int e = 0; e < PER; ++e)
    bonus[e] = KIND == STEP_LINEAR && a.bonus != nullptr && ks * PER + e < dim ? a.bonus[(size_t)h * dim + ks * PER + e] : 0.f;
  // ---- the head's inputs
  {
    // thread c: element c % 128 of q, k, v or (general) the removal rates
    const int i = tid % 128, part_of = tid / 128;
    const int width = part_of == 2 ? vdim : dim;
    const size_t col = (size_t)h * width + i;
    float x = 0.f;
    if (i < width) {
      if (part_of == 0) x = a.q[(size_t)t * a.q_stride + col];
      else if (part_of == 1) x = a.k[(size_t)t * a.k_stride + col];
      else if (part_of == 2) x = a.v[(size_t)t * a.v_stride + col];
      else if (KIND == STEP_GENERAL) x = a.a[(size_t)t * a.q_stride + col];
      if (KIND == STEP_DELTA && part_of < 3) {
        const int channels = 2 * a.heads * dim + a.heads * vdim;
        const size_t ch = (size_t)part_of * a.heads * dim + col;
        float* cs = st + a.conv_off + ch;
        float acc = 0.f;
        for (int j = 0; j < a.taps; ++j) {
          const float y = j < a.taps - 1 ? cs[(size_t)j * channels] : x;
          if (j > 0) cs[(size_t)(j - 1) * channels] = y;
          acc = fmaf(a.conv_w[(size_t)j * channels + ch], y, acc);
        }
        x = s_silu(acc);
      }
      if (KIND == STEP_LINEAR && part_of == 0) x *= a.q_scale;
    }
    if (part_of == 0) qs[i] = x;
    else if (part_of == 1) kk[i] = x;
    else if (part_of == 2) vs[i] = x;
    else as[i] = x;
    if (tid < 128) {
      const float y = tid < a.decay.rank ? a.decay.x[(size_t)t * a.x_stride + tid] : 0.f;
      xa[tid] = a.decay.in_act ? tanhf(y) : y;
    } else if (tid < 256 && a.gate_lr.x != nullptr) {
      xg[i] = i < a.gate_lr.rank ? a.gate_lr.x[(size_t)t * a.x_stride + i] : 0.f;
    }
  }
  __syncthreads();
  // ---- low-rank products
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  if (have) {
    const float* xs = lr < 128 ? xa : xg;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int d = 0; d < 4; ++d) acc[p] = fmaf(xs[b * 32 + (half * 4 + p) * 4 + d], lw[b][p][d], acc[p]);
    for (int i0 = 64; i0 < l.rank; i0 += 32) {
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const int i = i0 + (half * 4 + p) * 4;
#pragma unroll
        for (int d = 0; d < 4; ++d) acc[p] = fmaf(xs[i + d], i + d < l.rank ? wt[(size_t)(i + d) * l.columns] : 0.f, acc[p]);
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
      for (int i = lane; i < 128; i += TP_WAVE) {
        const float u = i < dim ? kk[i] * rk : 0.f;
        const float au = i < dim ? s_sigmoid(as[i] + a.a_bias[(size_t)h * dim + i]) * u : 0.f;
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
  __syncthreads();
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
  __syncthreads();
  // ---- the step
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
      ua[e] = bonus[e];
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
  __syncthreads();
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
  if (a.gate != nullptr) {
    if (a.gate_act == 2) g = make_float4(g.x * s_sigmoid(g.x), g.y * s_sigmoid(g.y), g.z * s_sigmoid(g.z), g.w * s_sigmoid(g.w));
    else g = make_float4(s_sigmoid(g.x), s_sigmoid(g.y), s_sigmoid(g.z), s_sigmoid(g.w));
  } else if (a.gate_lr.x != nullptr) {
    g = *(const float4*)(gs + d4);
  }
  from_float4((TO*)a.out + (size_t)t * a.out_stride + a.out_col0 + (size_t)h * vdim + d4, v[0] * g.x * a.scale, v[1] * g.y * a.scale,
              v[2] * g.z * a.scale, v[3] * g.w * a.scale);
}

// Sizes and places that the kernel takes (a step of n requests with one token each).
static int step_check(const StepArgs& a, int n) {
  const int hv = a.heads * a.vdim;
  TP_REQUIRE(n >= 0 && a.heads > 0 && a.heads <= 65535 && a.dim > 32 && a.dim <= 128 && a.dim % 4 == 0 && a.vdim > 0 && a.vdim <= 128 && a.vdim % 4 == 0,
             "mixer_step: sizes %d / %d are not its own", a.dim, a.vdim);
  TP_REQUIRE(a.decay.rank > 0 && a.decay.rank <= 128 && a.gate_lr.rank <= 128, "mixer_step: ranks of up to 128");
  TP_REQUIRE(((uintptr_t)a.state | (uintptr_t)a.out | (uintptr_t)a.norm_w | (uintptr_t)a.gate) % 16 == 0 && a.state_stride % 4 == 0 && a.state_off % 4 == 0 &&
                 a.out_stride % 4 == 0 && a.out_col0 % 4 == 0 && a.gate_stride % 4 == 0 && a.out_stride >= (size_t)(a.out_col0 + hv),
             "mixer_step: rows must lie on 16-byte places");
  TP_REQUIRE(a.state_stride >= a.state_off + (size_t)hv * a.dim, "mixer_step: state rows too short");
  return 0;
}

template <int KIND>
static void launch_step(const StepArgs& a, int n, int out_dt, hipStream_t s) {
  const dim3 grid(n, a.heads);
#define STEP(KS)                                                                                          \
  do {                                                                                                    \
    if (out_dt == TP_F32)                                                                                 \
      hipLaunchKernelGGL((mixer_step_kernel<KIND, KS, float>), grid, dim3(512), 0, s, a);                 \
    else                                                                                                  \
      hipLaunchKernelGGL((mixer_step_kernel<KIND, KS, bf16_t>), grid, dim3(512), 0, s, a);                \
  } while (0)
  if (a.dim <= 64) STEP(8);
  else STEP(16);
#undef STEP
}

// Gated delta rule: columns of `proj` (rows of proj_stride): q | k | v from col0, beta, the decay's and the gate's inner rows.
// state row: the convolution's carried inputs [taps - 1, channels] from conv_off on, the state [heads, vdim, dim] from state_off on.
extern "C" int tp_delta_step(const float* proj, size_t proj_stride, int col0, int beta_col0, int a_col0, int a_rank, int g_col0, int g_rank,
                             const float* conv_w, int taps, const float* a2_t, const float* g2_t, const float* a_log, const float* dt_bias,
                             const float* norm_w, float* state, size_t state_stride, size_t conv_off, size_t state_off, const int* token_req,
                             const int* state_slots, void* out, int out_dt, size_t out_stride, int out_col0, int n, int heads, int dim, int vdim,
                             float q_scale, float unit_eps, float norm_eps, float scale, hipStream_t s) {
  TP_REQUIRE(out_dt == TP_F32 || out_dt == TP_BF16, "delta_step: unknown dtype %d", out_dt);
  StepArgs a{};
  a.q = proj + col0;
  a.k = a.q + heads * dim;
  a.v = a.k + heads * dim;
  a.beta = proj + beta_col0;
  a.conv_w = conv_w;
  a.decay = LowRank{proj + a_col0, a2_t, a_log, dt_bias, a_rank, heads * dim, 2, 0, 0.f};
  a.gate_lr = LowRank{proj + g_col0, g2_t, nullptr, nullptr, g_rank, heads * vdim, 1, 0, 0.f};
  a.norm_w = norm_w;
  a.state = state;
  a.token_req = token_req;
  a.state_slots = state_slots;
  a.out = out;
  a.q_stride = a.k_stride = a.v_stride = a.x_stride = proj_stride;
  a.state_stride = state_stride;
  a.state_off = state_off;
  a.conv_off = conv_off;
  a.out_stride = out_stride;
  a.out_col0 = out_col0;
  a.heads = heads;
  a.dim = dim;
  a.vdim = vdim;
  a.taps = taps;
  a.q_scale = q_scale;
  a.unit_eps = unit_eps;
  a.norm_eps = norm_eps;
  a.scale = scale;
  TP_REQUIRE(taps >= 1 && g_rank > 0, "delta_step: bad sizes");
  TP_REQUIRE(state_stride >= conv_off + (size_t)(taps - 1) * heads * (2 * dim + vdim), "delta_step: state rows too short");
  if (const int rc = step_check(a, n)) return rc;
  if (n == 0) return 0;
  launch_step<STEP_DELTA>(a, n, out_dt, s);
  TP_CHECK_LAUNCH("delta_step");
  return 0;
}

// Generalized delta rule: columns r | k | v | a from col0, the gate's raw columns, the decay's inner rows (tanh).
extern "C" int tp_general_delta_step(const float* proj, size_t proj_stride, int col0, int gate_col0, int w_col0, int w_rank, const float* w2_t,
                                     const float* w0, float rate, const float* a_bias, const float* norm_w, float* state, size_t state_stride,
                                     size_t state_off, const int* token_req, const int* state_slots, void* out, int out_dt, size_t out_stride,
                                     int out_col0, int n, int heads, int dim, float unit_eps, float norm_eps, float scale, hipStream_t s) {
  TP_REQUIRE(out_dt == TP_F32 || out_dt == TP_BF16, "general_delta_step: unknown dtype %d", out_dt);
  StepArgs a{};
  const int hd = heads * dim;
  a.q = proj + col0;
  a.k = a.q + hd;
  a.v = a.k + hd;
  a.a = a.v + hd;
  a.a_bias = a_bias;
  a.decay = LowRank{proj + w_col0, w2_t, nullptr, w0, w_rank, hd, 3, 1, rate};
  a.gate = proj + gate_col0;
  a.gate_stride = proj_stride;
  a.gate_act = 1;
  a.norm_w = norm_w;
  a.norm_stride = heads > 1 ? dim : 0;
  a.state = state;
  a.token_req = token_req;
  a.state_slots = state_slots;
  a.out = out;
  a.q_stride = a.k_stride = a.v_stride = a.x_stride = proj_stride;
  a.state_stride = state_stride;
  a.state_off = state_off;
  a.out_stride = out_stride;
  a.out_col0 = out_col0;
  a.heads = heads;
  a.dim = a.vdim = dim;
  a.q_scale = 1.f;
  a.unit_eps = unit_eps;
  a.norm_eps = norm_eps;
  a.scale = scale;
  if (const int rc = step_check(a, n)) return rc;
  if (n == 0) return 0;
  launch_step<STEP_GENERAL>(a, n, out_dt, s);
  TP_CHECK_LAUNCH("general_delta_step");
  return 0;
}

// Linear recurrence: q, k, v rows of their own strides; x: the decay's inner rows (rank columns, rows of x_stride), mode and rate as
// in tp_lowrank_up; bonus [heads, dim] or nullptr; gate: raw rows of gate_stride (gate_act 1 sigmoid, 2 SiLU).
extern "C" int tp_linear_step(const float* q, size_t q_stride, const float* k, size_t k_stride, const float* v, size_t v_stride, const float* x,
                              size_t x_stride, int rank, const float* w2_t, const float* bias, int mode, int in_act, float rate,
                              const float* bonus, float q_scale, const float* gate, size_t gate_stride, int gate_act, const float* norm_w,
                              int norm_per_head, float* state, size_t state_stride, size_t state_off, const int* token_req,
                              const int* state_slots, void* out, int out_dt, size_t out_stride, int out_col0, int n, int heads, int dim,
                              int vdim, float norm_eps, float scale, hipStream_t s) {
  TP_REQUIRE(out_dt == TP_F32 || out_dt == TP_BF16, "linear_step: unknown dtype %d", out_dt);
  TP_REQUIRE(mode >= 3 && mode <= 5 && bias != nullptr && gate != nullptr && (gate_act == 1 || gate_act == 2), "linear_step: bad decay or gate");
  StepArgs a{};
  a.q = q;
  a.k = k;
  a.v = v;
  a.bonus = bonus;
  a.decay = LowRank{x, w2_t, nullptr, bias, rank, heads * dim, mode, in_act, rate};
  a.gate = gate;
  a.gate_stride = gate_stride;
  a.gate_act = gate_act;
  a.norm_w = norm_w;
  a.norm_stride = norm_per_head ? vdim : 0;
  a.state = state;
  a.token_req = token_req;
  a.state_slots = state_slots;
  a.out = out;
  a.q_stride = q_stride;
  a.k_stride = k_stride;
  a.v_stride = v_stride;
  a.x_stride = x_stride;
  a.state_stride = state_stride;
  a.state_off = state_off;
  a.out_stride = out_stride;
  a.out_col0 = out_col0;
  a.heads = heads;
  a.dim = dim;
  a.vdim = vdim;
  a.q_scale = q_scale;
  a.norm_eps = norm_eps;
  a.scale = scale;
  if (const int rc = step_check(a, n)) return rc;
  if (n == 0) return 0;
  launch_step<STEP_LINEAR>(a, n, out_dt, s);
  TP_CHECK_LAUNCH("linear_step");
  return 0;
}
