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
#include "step_mixer.h"

template <int KIND, int KS, typename TO>
__global__ __launch_bounds__(512, 4) void mixer_step_kernel(StepArgs a) {
  mixer_step_block<KIND, KS, TO>(a, blockIdx.x, blockIdx.y);
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

// `prepared` (host memory of tp_step_prepared_size bytes): the step is checked and written down there, for a launch that runs it beside
// other blocks (tp_attention_rows), instead of launched.
extern "C" size_t tp_step_prepared_size() { return sizeof(PreparedStep); }
static int step_prepare(const StepArgs& a, int kind, int n, int out_dt, void* prepared) {
  TP_REQUIRE(out_dt == TP_BF16, "mixer_step: a step beside others writes bfloat16");
  *(PreparedStep*)prepared = PreparedStep{a, kind, n};
  return 0;
}

// Gated delta rule: columns of `proj` (rows of proj_stride): q | k | v from col0, beta, the decay's and the gate's inner rows.
// state row: the convolution's carried inputs [taps - 1, channels] from conv_off on, the state [heads, vdim, dim] from state_off on.
extern "C" int tp_delta_step(const float* proj, size_t proj_stride, int col0, int beta_col0, int a_col0, int a_rank, int g_col0, int g_rank,
                             const float* conv_w, int taps, const float* a2_t, const float* g2_t, const float* a_log, const float* dt_bias,
                             const float* norm_w, float* state, size_t state_stride, size_t conv_off, size_t state_off, const int* token_req,
                             const int* state_slots, void* out, int out_dt, size_t out_stride, int out_col0, int n, int heads, int dim, int vdim,
                             float q_scale, float unit_eps, float norm_eps, float scale, void* prepared, hipStream_t s) {
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
  if (prepared != nullptr) return step_prepare(a, STEP_DELTA, n, out_dt, prepared);
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
                              int vdim, float norm_eps, float scale, void* prepared, hipStream_t s) {
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
  if (prepared != nullptr) return step_prepare(a, STEP_LINEAR, n, out_dt, prepared);
  launch_step<STEP_LINEAR>(a, n, out_dt, s);
  TP_CHECK_LAUNCH("linear_step");
  return 0;
}
