// Small kernels around the products of a layer: an embedding with a hashed bigram table, the gate on an attention's
// output, the norm behind a sublayer added into the residual stream, a plain activation, and the router of a
// mixture of experts and what moves rows into the order of the experts and back.  Float32 arithmetic throughout; a row's result
// never depends on other rows.
#include <math.h>

#include "common.h"
#include "moe_route.h"
#include "activations.h"

__device__ inline float l_sigmoid(float v) { return 1.0f / (1.0f + expf(-v)); }

// ---- embedding plus a row of a hashed bigram table --------------------------------------------
// out[t] = table[token] * scale + bigram[row] (+ pos_table[position], a learned row per position), row = (previous * mul_prev + token * mul_cur) mod buckets, and row `buckets`
// (the table's last) for the token at position 0.  The previous token is the one before it in the step's run, or,
// for a run's first token, what the request's state row holds: that token's block alone reads it, and then leaves the run's last token there.
template <typename T>
__global__ void embed_bigram_kernel(const int* __restrict__ tokens, const int* __restrict__ positions,
                                    const int* __restrict__ token_req, const int* __restrict__ cu_seqlens,
                                    const int* __restrict__ state_slots, int* __restrict__ prev_state,
                                    const T* __restrict__ table, const T* __restrict__ bigram, float* __restrict__ out,
                                    int hidden, long long mul_prev, long long mul_cur, long long buckets, float scale,
                                    const T* __restrict__ pos_table, int four) {
  const int t = blockIdx.x;
  const int tok = tokens[t], pos = positions[t];
  long long row = buckets;
  if (bigram != nullptr) {
    const int r = token_req[t], start = cu_seqlens[r];
    const int prev = t > start ? tokens[t - 1] : prev_state[state_slots[r]];
    if (pos != 0) row = ((long long)prev * mul_prev + (long long)tok * mul_cur) % buckets;
    if (t == start) {
      __syncthreads();   // (every thread has read the carried token)
      if (threadIdx.x == 0) prev_state[state_slots[r]] = tokens[cu_seqlens[r + 1] - 1];
    }
  }
  const T* a = table + (size_t)tok * hidden;
  const T* b = bigram != nullptr ? bigram + (size_t)row * hidden : nullptr;
  // (scale 1 and no position table: the sum of the two rows as it always was)
  const T* p = pos_table != nullptr ? pos_table + (size_t)pos * hidden : nullptr;
  if (four) {            // four neighbouring elements a thread, the rows' pieces in flight together
    for (int c = threadIdx.x * 4; c < hidden; c += blockDim.x * 4) {
      const float4 x = load_float4(a + c);
      const float4 y = b != nullptr ? load_float4(b + c) : make_float4(0.f, 0.f, 0.f, 0.f);
      const float4 z = p != nullptr ? load_float4(p + c) : make_float4(0.f, 0.f, 0.f, 0.f);
      float4 v = make_float4(x.x * scale, x.y * scale, x.z * scale, x.w * scale);
      if (b != nullptr) v = make_float4(v.x + y.x, v.y + y.y, v.z + y.z, v.w + y.w);
      if (p != nullptr) v = make_float4(v.x + z.x, v.y + z.y, v.z + z.z, v.w + z.w);
      *(float4*)(out + (size_t)t * hidden + c) = v;
    }
    return;
  }
  for (int c = threadIdx.x; c < hidden; c += blockDim.x) {
    float v = to_float(a[c]) * scale;
    if (b != nullptr) v += to_float(b[c]);
    if (p != nullptr) v += to_float(p[c]);
    out[(size_t)t * hidden + c] = v;
  }
}

extern "C" int tp_embed_bigram(const int* tokens, const int* positions, const int* token_req, const int* cu_seqlens,
                               const int* state_slots, int* prev_state, const void* table, const void* bigram, int dt,
                               float* out, int n, int n_req, int hidden, long long mul_prev, long long mul_cur,
                               long long buckets, float scale, const void* pos_table, hipStream_t s) {
  // (bigram may be missing: the token's row times scale, plus the position's row)
  TP_REQUIRE(n >= 0 && n_req >= 0 && hidden > 0 && (bigram == nullptr || buckets > 0) && mul_prev >= 0 && mul_cur >= 0, "embed_bigram: bad sizes");
  if (n == 0) return 0;
  // (a row of 4,096 as one piece of four a thread: one token 22 -> 5 us, with the launch that left the last tokens)
  const int four = hidden % 4 == 0 && (((uintptr_t)table | (uintptr_t)bigram | (uintptr_t)pos_table | (uintptr_t)out) & 15) == 0;
  const int threads = four ? min(1024, max(64, (hidden / 4 + 63) / 64 * 64)) : hidden >= 256 ? 256 : 64;
  if (dt == TP_F32)
    hipLaunchKernelGGL(embed_bigram_kernel<float>, dim3(n), dim3(threads), 0, s, tokens, positions, token_req, cu_seqlens,
                       state_slots, prev_state, (const float*)table, (const float*)bigram, out, hidden, mul_prev, mul_cur, buckets, scale,
                       (const float*)pos_table, four);
  else if (dt == TP_BF16)
    hipLaunchKernelGGL(embed_bigram_kernel<bf16_t>, dim3(n), dim3(threads), 0, s, tokens, positions, token_req, cu_seqlens,
                       state_slots, prev_state, (const bf16_t*)table, (const bf16_t*)bigram, out, hidden, mul_prev, mul_cur, buckets, scale,
                       (const bf16_t*)pos_table, four);
  else
    TP_REQUIRE(false, "embed_bigram: unknown dtype %d", dt);
  TP_CHECK_LAUNCH("embed_bigram");
  return 0;
}

// ---- gate on a mixer's output -----------------------------------------------------------------
// out[t, out_col0 + c] = a[t, c] * sigmoid(proj[t, gate_col0 + c / per]) * scale (no gate: a * scale; per 1: a gate per
// column, per = head size: one per head); the product is formed in float32 and rounded once.
template <typename T>
__global__ void sigmoid_gate_kernel(const T* __restrict__ a, const float* __restrict__ proj, int proj_stride, int gate_col0,
                                    float scale, T* __restrict__ out, int out_stride, int out_col0, int width, size_t total, int per) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const size_t t = i / width;
  const int c = (int)(i % width);
  float v = to_float(a[i]);
  if (proj != nullptr) v *= l_sigmoid(proj[t * proj_stride + gate_col0 + c / per]);
  from_float(out + t * out_stride + out_col0 + c, v * scale);
}

// the same, four neighbouring columns a thread (every width, stride and first column a multiple of four; per 1 or a
// multiple of four)
template <typename T>
__global__ void sigmoid_gate4_kernel(const T* __restrict__ a, const float* __restrict__ proj, int proj_stride, int gate_col0,
                                     float scale, T* __restrict__ out, int out_stride, int out_col0, int width, size_t total4, int per) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total4) return;
  const int w4 = width / 4;
  const size_t t = i / w4;
  const int c = (int)(i % w4) * 4;
  float v[4];
  if constexpr (sizeof(T) == 2) {
    const uint2 raw = *(const uint2*)(a + t * width + c);
    bf16_t h0{(uint16_t)(raw.x & 0xffff)}, h1{(uint16_t)(raw.x >> 16)}, h2{(uint16_t)(raw.y & 0xffff)}, h3{(uint16_t)(raw.y >> 16)};
    v[0] = bf16_to_float(h0); v[1] = bf16_to_float(h1); v[2] = bf16_to_float(h2); v[3] = bf16_to_float(h3);
  } else {
    const float4 raw = *(const float4*)(a + t * width + c);
    v[0] = raw.x; v[1] = raw.y; v[2] = raw.z; v[3] = raw.w;
  }
  if (proj != nullptr && per != 1) {
    const float g = l_sigmoid(proj[t * proj_stride + gate_col0 + c / per]);
    v[0] *= g; v[1] *= g; v[2] *= g; v[3] *= g;
  } else if (proj != nullptr) {
    const float4 g = *(const float4*)(proj + t * proj_stride + gate_col0 + c);
    v[0] *= l_sigmoid(g.x); v[1] *= l_sigmoid(g.y); v[2] *= l_sigmoid(g.z); v[3] *= l_sigmoid(g.w);
  }
  from_float4(out + t * out_stride + out_col0 + c, v[0] * scale, v[1] * scale, v[2] * scale, v[3] * scale);
}

extern "C" int tp_sigmoid_gate(const void* a, int dt, const float* proj, int proj_stride, int gate_col0, float scale, void* out,
                               int out_stride, int out_col0, int n, int width, int per, hipStream_t s) {
  TP_REQUIRE(n >= 0 && width > 0 && out_col0 >= 0 && out_stride >= out_col0 + width, "sigmoid_gate: bad sizes");
  TP_REQUIRE(per >= 1 && width % per == 0, "sigmoid_gate: %d columns are not runs of %d", width, per);
  TP_REQUIRE(proj == nullptr || (gate_col0 >= 0 && proj_stride >= gate_col0 + width / per), "sigmoid_gate: gate rows too short");
  TP_REQUIRE(dt == TP_F32 || dt == TP_BF16, "sigmoid_gate: unknown dtype %d", dt);
  if (n == 0) return 0;
  const size_t esz = dt == TP_F32 ? 4 : 2;
  const bool four = width % 4 == 0 && out_stride % 4 == 0 && out_col0 % 4 == 0 &&
                    (proj == nullptr || (per == 1 ? proj_stride % 4 == 0 && gate_col0 % 4 == 0 && (uintptr_t)proj % 16 == 0 : per % 4 == 0)) &&
                    (uintptr_t)a % 16 == 0 && (uintptr_t)out % 16 == 0 && esz * 4 <= 16;
  if (four) {
    const size_t total4 = (size_t)n * (width / 4);
    const dim3 grid((unsigned)((total4 + 255) / 256));
    if (dt == TP_F32)
      hipLaunchKernelGGL(sigmoid_gate4_kernel<float>, grid, dim3(256), 0, s, (const float*)a, proj, proj_stride, gate_col0, scale,
                         (float*)out, out_stride, out_col0, width, total4, per);
    else
      hipLaunchKernelGGL(sigmoid_gate4_kernel<bf16_t>, grid, dim3(256), 0, s, (const bf16_t*)a, proj, proj_stride, gate_col0, scale,
                         (bf16_t*)out, out_stride, out_col0, width, total4, per);
  } else {
    const size_t total = (size_t)n * width;
    const dim3 grid((unsigned)((total + 255) / 256));
    if (dt == TP_F32)
      hipLaunchKernelGGL(sigmoid_gate_kernel<float>, grid, dim3(256), 0, s, (const float*)a, proj, proj_stride, gate_col0, scale,
                         (float*)out, out_stride, out_col0, width, total, per);
    else
      hipLaunchKernelGGL(sigmoid_gate_kernel<bf16_t>, grid, dim3(256), 0, s, (const bf16_t*)a, proj, proj_stride, gate_col0, scale,
                         (bf16_t*)out, out_stride, out_col0, width, total, per);
  }
  TP_CHECK_LAUNCH("sigmoid_gate");
  return 0;
}

// ---- a sublayer's output, normed, into the residual stream ------------------------------------
// h[t] += y[t] / sqrt(mean(y[t]^2) + eps) * w; then, with w_next, the next sublayer's input
// x[t] = h[t] / sqrt(mean(h[t]^2) + eps_next) * w_next as TO.  One block per row.
// With gate rows, y stands for y[t, c] * sigmoid(gate.rows[t, gate.col0 + c] + gate.bias[c]).  Not normed: h[t] += y[t] * w.
// blocked: the rows x leave as [width / 8, n, 8], what products of a few rows read best.
struct InputGate {
  const float* rows;   // float32 [n, stride], or nullptr: no gate
  const float* bias;   // [width], or nullptr
  size_t stride;
  int col0;
};

template <typename TO>
__global__ __launch_bounds__(256) void norm_add_kernel(float* __restrict__ h, const float* __restrict__ y,
                                                       const float* __restrict__ w, float eps,
                                                       const float* __restrict__ w_next, float eps_next,
                                                       TO* __restrict__ x, int width, InputGate gate, int normed, int blocked, int parts) {
  __shared__ float scratch[32];
  const size_t base = (size_t)blockIdx.x * width;
  const float* gr = gate.rows != nullptr ? gate.rows + (size_t)blockIdx.x * gate.stride + gate.col0 : nullptr;
  auto value = [&](int c) {
    float v = y[base + c];
    for (int p = 1; p < parts; ++p) v += y[(size_t)p * gridDim.x * width + base + c];
    return gr != nullptr ? v * l_sigmoid(gr[c] + (gate.bias != nullptr ? gate.bias[c] : 0.f)) : v;
  };
  float rstd = 1.0f;
  if (normed) {   // (uniform)
    float ss = 0.f;
    for (int c = threadIdx.x; c < width; c += blockDim.x) {
      const float v = value(c);
      ss = fmaf(v, v, ss);
    }
    ss = block_sum(ss, scratch);
    rstd = 1.0f / sqrtf(ss / (float)width + eps);
  }
  float ss2 = 0.f;
  for (int c = threadIdx.x; c < width; c += blockDim.x) {
    const float v = h[base + c] + value(c) * rstd * w[c];
    h[base + c] = v;
    ss2 = fmaf(v, v, ss2);
  }
  if (w_next == nullptr) return;
  ss2 = block_sum(ss2, scratch);
  const float rstd2 = 1.0f / sqrtf(ss2 / (float)width + eps_next);
  // (each thread reads back what it wrote itself)
  for (int c = threadIdx.x; c < width; c += blockDim.x)
    from_float(x + (blocked ? ((size_t)(c >> 3) * gridDim.x + blockIdx.x) * 8 + (c & 7) : base + c), h[base + c] * rstd2 * w_next[c]);
}

// The same with the row in registers: every value is read once, sixteen bytes a load, all loads of a pass in flight
// together (width a multiple of four, at most 4 * T * NV).  S: the values a thread brings to a sum, whose order is that of a block of S * T threads
// whatever T is, so a row's bits do not depend on how many rows there are.
// Few rows wait for one request of all their operands and for the sums, so a thread has as little of a row as can be (one row of 4,096 in two
// parts 4.14 -> 3.20 us against 256 threads that load in turn, with a gate 5.49 -> 3.73); many rows wait for memory.
// LATE (y in one part): the gate and the next norm's weight are requested where they are used, so that fewer registers leave room for more rows.
template <typename TO, int T, int NV, bool GATE, int S, bool LATE>
__global__ __launch_bounds__(T) void norm_add_reg_kernel(float* __restrict__ h, const float* __restrict__ y,
                                                           const float* __restrict__ w, float eps,
                                                           const float* __restrict__ w_next, float eps_next,
                                                           TO* __restrict__ x, int width, InputGate gate, int normed, int blocked, int parts) {
  __shared__ __attribute__((aligned(16))) float scratch[2][S * T / TP_WAVE];
  const size_t base = (size_t)blockIdx.x * width;
  const int w4 = width / 4;
  const size_t part = (size_t)gridDim.x * width;
  const float* gr = GATE ? gate.rows + (size_t)blockIdx.x * gate.stride + gate.col0 : nullptr;
  float4 yv[NV], y1[NV], y2[NV], y3[NV], hv[NV], wv[NV], gv[GATE ? NV : 1], bv[GATE ? NV : 1], nv[NV];
  auto fetch_gate = [&](int k) {
    const int c = k * T + threadIdx.x;
    if (c < w4) {
      gv[k] = *(const float4*)(gr + 4 * c);
      bv[k] = gate.bias != nullptr ? *(const float4*)(gate.bias + 4 * c) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  auto fetch_next = [&](int k) {
    const int c = k * T + threadIdx.x;
    if (c < w4) nv[k] = *(const float4*)(w_next + 4 * c);
  };
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int c = k * T + threadIdx.x;
    if (c < w4) {
      const float* yp = y + base + 4 * c;
      yv[k] = *(const float4*)yp;
      if (!LATE && parts > 1) y1[k] = *(const float4*)(yp + part);
      if (!LATE && parts > 2) y2[k] = *(const float4*)(yp + 2 * part);
      if (!LATE && parts > 3) y3[k] = *(const float4*)(yp + 3 * part);
      if constexpr (GATE && !LATE) fetch_gate(k);
      hv[k] = *(const float4*)(h + base + 4 * c);
      wv[k] = *(const float4*)(w + 4 * c);
      if (!LATE && w_next != nullptr) fetch_next(k);
    }
  }
  // (parts > 1: y is that many partial sums of a product, added in ascending order)
  auto add = [](float4& a, const float4& b) {
    a.x += b.x;
    a.y += b.y;
    a.z += b.z;
    a.w += b.w;
  };
  if constexpr (GATE && LATE) {
#pragma unroll
    for (int k = 0; k < NV; ++k) fetch_gate(k);
  }
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int c = k * T + threadIdx.x;
    if (c < w4) {
      if (!LATE && parts > 1) add(yv[k], y1[k]);
      if (!LATE && parts > 2) add(yv[k], y2[k]);
      if (!LATE && parts > 3) add(yv[k], y3[k]);
      for (int p = 4; !LATE && p < parts; ++p) add(yv[k], *(const float4*)(y + p * part + base + 4 * c));
      if constexpr (GATE) {
        yv[k].x *= l_sigmoid(gv[k].x + bv[k].x);
        yv[k].y *= l_sigmoid(gv[k].y + bv[k].y);
        yv[k].z *= l_sigmoid(gv[k].z + bv[k].z);
        yv[k].w *= l_sigmoid(gv[k].w + bv[k].w);
      }
    }
  }
  float rstd = 1.0f;
  if (normed) {
    float ss[S] = {};
#pragma unroll
    for (int k = 0; k < NV; ++k)
      if (k * T + threadIdx.x < w4) {
        ss[k % S] = fmaf(yv[k].x, yv[k].x, ss[k % S]);
        ss[k % S] = fmaf(yv[k].y, yv[k].y, ss[k % S]);
        ss[k % S] = fmaf(yv[k].z, yv[k].z, ss[k % S]);
        ss[k % S] = fmaf(yv[k].w, yv[k].w, ss[k % S]);
      }
    rstd = 1.0f / sqrtf(block_sum_once<T>(ss, scratch[0]) / (float)width + eps);
  }
  float ss2[S] = {};
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int c = k * T + threadIdx.x;
    if (c < w4) {
      hv[k].x += yv[k].x * rstd * wv[k].x;
      hv[k].y += yv[k].y * rstd * wv[k].y;
      hv[k].z += yv[k].z * rstd * wv[k].z;
      hv[k].w += yv[k].w * rstd * wv[k].w;
      *(float4*)(h + base + 4 * c) = hv[k];
      ss2[k % S] = fmaf(hv[k].x, hv[k].x, ss2[k % S]);
      ss2[k % S] = fmaf(hv[k].y, hv[k].y, ss2[k % S]);
      ss2[k % S] = fmaf(hv[k].z, hv[k].z, ss2[k % S]);
      ss2[k % S] = fmaf(hv[k].w, hv[k].w, ss2[k % S]);
    }
  }
  if (w_next == nullptr) return;
  if constexpr (LATE) {
#pragma unroll
    for (int k = 0; k < NV; ++k) fetch_next(k);
  }
  const float rstd2 = 1.0f / sqrtf(block_sum_once<T>(ss2, scratch[1]) / (float)width + eps_next);
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int c = k * T + threadIdx.x;
    if (c < w4) from_float4(x + (blocked ? ((size_t)(c >> 1) * gridDim.x + blockIdx.x) * 8 + (c & 1) * 4 : base + 4 * c), hv[k].x * rstd2 * nv[k].x, hv[k].y * rstd2 * nv[k].y, hv[k].z * rstd2 * nv[k].z, hv[k].w * rstd2 * nv[k].w);
  }
}

extern "C" int tp_norm_add(float* h, const float* y, const float* w, float eps, const float* w_next, float eps_next, void* x,
                           int x_dt, int n, int width, const float* gate_rows, size_t gate_stride, int gate_col0,
                           const float* gate_bias, int normed, int blocked, int parts, hipStream_t s) {
  TP_REQUIRE(parts >= 1, "norm_add: bad parts");
  TP_REQUIRE(n >= 0 && width > 0, "norm_add: bad sizes");
  TP_REQUIRE(gate_rows == nullptr || (gate_col0 >= 0 && gate_stride >= (size_t)gate_col0 + width), "norm_add: gate rows too short");
  const InputGate gate{gate_rows, gate_bias, gate_stride, gate_col0};
  TP_REQUIRE(w_next == nullptr || x != nullptr, "norm_add: no place for the next rows");
  if (n == 0) return 0;
  TP_REQUIRE(w_next == nullptr || x_dt == TP_F32 || x_dt == TP_BF16, "norm_add: unknown dtype %d", x_dt);
  TP_REQUIRE(!blocked || width % 8 == 0, "norm_add: k-blocked rows need a width that is a multiple of eight");
  const bool aligned = ((uintptr_t)h % 16) == 0 && ((uintptr_t)y % 16) == 0 && ((uintptr_t)w % 16) == 0 && ((uintptr_t)w_next % 16) == 0 &&
                       ((uintptr_t)x % 16) == 0 &&
                       (gate_rows == nullptr || (((uintptr_t)gate_rows | (uintptr_t)gate_bias) % 16 == 0 && gate_stride % 4 == 0 && gate_col0 % 4 == 0));
  if (width % 4 == 0 && width >= 1024 && width <= 256 * 4 * 8 && aligned) {
    const bool bf = w_next != nullptr && x_dt == TP_BF16;
#define NA1(TO, T, NV, G, S, L) \
  hipLaunchKernelGGL((norm_add_reg_kernel<TO, T, NV, G, S, L>), dim3(n), dim3(T), 0, s, h, y, w, eps, w_next, eps_next, (TO*)x, width, gate, normed, blocked, parts)
#define NAP(T, NV, S, L)                     \
  do {                                       \
    if (bf) NA1(bf16_t, T, NV, false, S, L);  \
    else NA1(float, T, NV, false, S, L);      \
  } while (0)
#define NA(T, NV, S, L)                      \
  do {                                       \
    if (gate_rows == nullptr) NAP(T, NV, S, L);  \
    else if (bf) NA1(bf16_t, T, NV, true, S, L); \
    else NA1(float, T, NV, true, S, L);       \
  } while (0)
    // A thread for every 16 bytes, and fewer from two rows a CU on: more blocks then share a CU and hide one another's barriers.  Rows of many
    // parts need their registers and keep more threads for longer (2,048 rows of 2,048 in three parts 15.9 us, with 256 threads 16.3).
    // From there on rows of one part request their gate and the next norm's weight late (LATE), which leaves room for more of them.  Without a gate still fewer threads
    // take a row where there are many, whose sums cost fewer instructions.  us, threads x pieces (l: late), without a gate:
    //   1,408 columns   512x1 / 256x2 / 256x2l / 128x4l   200 rows 3.2 / 3.5 / 3.6 / 3.9, 560 4.5 / 4.3 / 4.3 / 4.7, 1,100 6.2 / 6.0 / 5.5 / 5.6, 3,033 11.8 / 10.8 / 10.9 / 9.3
    //   3,072           1,024x1 / 512x2 / 512x2l / 256x4l  256 rows 4.2 / 4.2 / 4.3 / 4.7, 400 5.4 / 5.0 / 5.0 / 5.4, 640 7.3 / 6.4 / 6.3 / 6.3, 1,500 13.0 / 11.5 / 11.9 / 10.5
    //   5,120           1,024x2 / 1,024x2l / 512x3 / 512x3l  200 rows 4.8 / 4.8 / 4.9 / 4.9, 400 6.9 / 6.7 / 6.5 / 6.4, 640 9.2 / 9.1 / 9.4 / 8.1, 2,337 28.0 / 28.8 / 29.8 / 26.4
    // and with one, 2,048: 1,500 rows 10.5 / 10.4 / 10.1 / 12.4; 3,072: 256 rows 4.8 / 4.9 / 5.0 / 5.5, 640 8.7 / 8.3 / 8.4 / 8.6, 1,024 11.8 / 11.2 / 10.4 / 10.9; 5,120: 400 rows
    // 9.4 / 8.6 / 8.6 / 8.7, 2,337 41.6 / 34.9 / 37.1 / 34.3; 8,192 (1,024x2 / 512x4l): 1,100 rows 35.3 / 28.8.
    if (width <= 1024) NA(256, 1, 1, false);
    else if (width < 2048 && n > 2048 && parts == 1 && gate_rows == nullptr) NAP(128, 4, 4, true);
    else if (width <= 2048 && n > 512 && parts == 1) NA(256, 2, 2, true);
    else if (width <= 2048) NA(512, 1, 1, false);
    else if (width <= 4096 && n > 768 && parts == 1 && gate_rows == nullptr) NAP(256, 4, 4, true);
    else if (width <= 4096 && n > (gate_rows != nullptr ? 768 : 256) && parts == 1) NA(512, 2, 2, true);
    else if (width <= 4096 && n > 256 && parts == 1) NA(512, 2, 2, false);
    else if (width <= 4096 && n > 512) NA(512, 2, 2, false);
    else if (width <= 4096) NA(1024, 1, 1, false);
    else if (width <= 6144 && n > 512 && parts == 1) NA(512, 3, 2, true);
    else if (n > 512 && parts == 1) NA(512, 4, 2, true);
    else if (n > 256 && parts == 1) NA(1024, 2, 1, true);
    else NA(1024, 2, 1, false);
#undef NA
#undef NAP
#undef NA1
    TP_CHECK_LAUNCH("norm_add");
    return 0;
  }
  const int threads = width >= 1024 ? 256 : (width >= 256 ? 128 : 64);
  if (w_next == nullptr || x_dt == TP_F32)
    hipLaunchKernelGGL(norm_add_kernel<float>, dim3(n), dim3(threads), 0, s, h, y, w, eps, w_next, eps_next, (float*)x, width, gate, normed, blocked, parts);
  else if (x_dt == TP_BF16)
    hipLaunchKernelGGL(norm_add_kernel<bf16_t>, dim3(n), dim3(threads), 0, s, h, y, w, eps, w_next, eps_next, (bf16_t*)x, width, gate, normed, blocked, parts);
  else
    TP_REQUIRE(false, "norm_add: unknown dtype %d", x_dt);
  TP_CHECK_LAUNCH("norm_add");
  return 0;
}

// ---- a plain activation -----------------------------------------------------------------------
// (the kinds: activations.h)
// Rows of a wider float32 tensor: out[t, c] = act(in[t, col0 + c]) for c < width, times sigmoid(in[t, gate_col]) when
// gate_col >= 0 (one gate a row: what a product behind it would be multiplied by, folded into its input).
template <typename TO>
__global__ void activation_rows_kernel(const float* __restrict__ in, size_t in_stride, int col0, int width, int gate_col,
                                       TO* __restrict__ out, size_t total, int kind) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const size_t t = i / width;
  const int c = (int)(i % width);
  const float* row = in + t * in_stride;
  float v = act_f(row[col0 + c], kind);
  if (gate_col >= 0) v *= l_sigmoid(row[gate_col]);
  from_float(out + i, v);
}

// the same without a gate, four neighbouring columns a thread (every width, stride and first column a multiple of four)
template <typename TO>
__global__ void activation_rows4_kernel(const float* __restrict__ in, size_t in_stride, int col0, int width, TO* __restrict__ out,
                                        size_t total4, int kind) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total4) return;
  const int w4 = width / 4;
  const size_t t = i / w4;
  const float4 z = *(const float4*)(in + t * in_stride + col0 + 4 * (int)(i % w4));
  from_float4(out + 4 * i, act_f(z.x, kind), act_f(z.y, kind), act_f(z.z, kind), act_f(z.w, kind));
}

extern "C" int tp_activation_rows(const float* in, size_t in_stride, int col0, int width, int gate_col, void* out, int out_dt, int n,
                                  int kind, hipStream_t s) {
  TP_REQUIRE(kind >= 0 && kind <= 3, "activation: unknown kind %d", kind);
  TP_REQUIRE(n >= 0 && width > 0 && col0 >= 0 && (size_t)(col0 + width) <= in_stride && gate_col < (long)in_stride, "activation: bad rows");
  const size_t total = (size_t)n * width;
  if (total == 0) return 0;
  if (gate_col < 0 && width % 4 == 0 && in_stride % 4 == 0 && col0 % 4 == 0 && (uintptr_t)in % 16 == 0 && (uintptr_t)out % 16 == 0 &&
      (out_dt == TP_F32 || out_dt == TP_BF16)) {
    const size_t total4 = total / 4;
    const dim3 grid4((unsigned)((total4 + 255) / 256));
    if (out_dt == TP_F32)
      hipLaunchKernelGGL(activation_rows4_kernel<float>, grid4, dim3(256), 0, s, in, in_stride, col0, width, (float*)out, total4, kind);
    else
      hipLaunchKernelGGL(activation_rows4_kernel<bf16_t>, grid4, dim3(256), 0, s, in, in_stride, col0, width, (bf16_t*)out, total4, kind);
    TP_CHECK_LAUNCH("activation_rows");
    return 0;
  }
  const dim3 grid((unsigned)((total + 255) / 256));
  if (out_dt == TP_F32)
    hipLaunchKernelGGL(activation_rows_kernel<float>, grid, dim3(256), 0, s, in, in_stride, col0, width, gate_col, (float*)out, total, kind);
  else if (out_dt == TP_BF16)
    hipLaunchKernelGGL(activation_rows_kernel<bf16_t>, grid, dim3(256), 0, s, in, in_stride, col0, width, gate_col, (bf16_t*)out, total, kind);
  else
    TP_REQUIRE(false, "activation: unknown dtype %d", out_dt);
  TP_CHECK_LAUNCH("activation_rows");
  return 0;
}

template <typename TI, typename TO>
__global__ void activation_kernel(const TI* __restrict__ in, TO* __restrict__ out, size_t total, int kind) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  from_float(out + i, act_f(to_float(in[i]), kind));
}

// float32 in, four neighbouring elements a thread
template <typename TO>
__global__ void activation4_kernel(const float* __restrict__ in, TO* __restrict__ out, size_t total4, int kind) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total4) return;
  const float4 z = *(const float4*)(in + 4 * i);
  from_float4(out + 4 * i, act_f(z.x, kind), act_f(z.y, kind), act_f(z.z, kind), act_f(z.w, kind));
}

// float32 rows [m, width] -> [width / 8, m, 8]
template <typename TO>
__global__ void activation_blocked_kernel(const float* __restrict__ in, TO* __restrict__ out, int m, int width, int kind) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, quads = width / 4;
  if (i >= m * quads) return;
  const int t = i / quads, c = i % quads * 4;
  const float4 z = *(const float4*)(in + (size_t)t * width + c);
  from_float4(out + ((size_t)(c >> 3) * m + t) * 8 + (c & 7), act_f(z.x, kind), act_f(z.y, kind), act_f(z.z, kind), act_f(z.w, kind));
}

extern "C" int tp_activation_blocked(const float* in, void* out, int out_dt, int m, int width, int kind, hipStream_t s) {
  TP_REQUIRE(kind >= 0 && kind <= 3, "activation: unknown kind %d", kind);
  TP_REQUIRE(m > 0 && width > 0 && width % 8 == 0 && (long)m * width < 0x7fffffffL && (((uintptr_t)in | (uintptr_t)out) & 15) == 0, "activation: bad rows");
  TP_REQUIRE(out_dt == TP_F32 || out_dt == TP_BF16, "activation: unknown dtype %d", out_dt);
  const dim3 grid((m * (width / 4) + 255) / 256);
  if (out_dt == TP_F32)
    hipLaunchKernelGGL(activation_blocked_kernel<float>, grid, dim3(256), 0, s, in, (float*)out, m, width, kind);
  else
    hipLaunchKernelGGL(activation_blocked_kernel<bf16_t>, grid, dim3(256), 0, s, in, (bf16_t*)out, m, width, kind);
  TP_CHECK_LAUNCH("activation_blocked");
  return 0;
}

extern "C" int tp_activation(const void* in, int in_dt, void* out, int out_dt, size_t total, int kind, hipStream_t s) {
  TP_REQUIRE(kind >= 0 && kind <= 3, "activation: unknown kind %d", kind);
  if (total == 0) return 0;
  if (in_dt == TP_F32 && total % 4 == 0 && (uintptr_t)in % 16 == 0 && (uintptr_t)out % 16 == 0 && (out_dt == TP_F32 || out_dt == TP_BF16)) {
    const size_t total4 = total / 4;
    const dim3 grid4((unsigned)((total4 + 255) / 256));
    if (out_dt == TP_F32)
      hipLaunchKernelGGL(activation4_kernel<float>, grid4, dim3(256), 0, s, (const float*)in, (float*)out, total4, kind);
    else
      hipLaunchKernelGGL(activation4_kernel<bf16_t>, grid4, dim3(256), 0, s, (const float*)in, (bf16_t*)out, total4, kind);
    TP_CHECK_LAUNCH("activation");
    return 0;
  }
  const dim3 grid((unsigned)((total + 255) / 256));
#define ACT(TI, TO) hipLaunchKernelGGL((activation_kernel<TI, TO>), grid, dim3(256), 0, s, (const TI*)in, (TO*)out, total, kind)
  if (in_dt == TP_F32 && out_dt == TP_F32)
    ACT(float, float);
  else if (in_dt == TP_F32 && out_dt == TP_BF16)
    ACT(float, bf16_t);
  else if (in_dt == TP_BF16 && out_dt == TP_BF16)
    ACT(bf16_t, bf16_t);
  else
    TP_REQUIRE(false, "activation: unsupported dtypes %d -> %d", in_dt, out_dt);
#undef ACT
  TP_CHECK_LAUNCH("activation");
  return 0;
}

// ---- router of a mixture of experts (see moe_route.h) ------------------------------------------
template <int ROUTE_LANE>
__global__ __launch_bounds__(256) void moe_route_kernel(Route r, const float* __restrict__ logits, int logit_stride, int n) {
  extern __shared__ float lds[];   // per wave: choice scores [experts], then group scores [groups]
  const int wave = threadIdx.x / TP_WAVE;
  // (a wave past the last token works on the last token again and stores nothing: every wave reaches every barrier)
  const bool live = blockIdx.x * 4 + wave < n;
  const int t = live ? blockIdx.x * 4 + wave : n - 1;
  float* choice_l = lds + (size_t)wave * (r.experts + max(r.groups, 1));
  route_token<ROUTE_LANE>(r, logits + (size_t)t * logit_stride, t, live, choice_l, choice_l + r.experts);
}

__global__ __launch_bounds__(256) void moe_route_few_kernel(Route r, const float* __restrict__ logits, int logit_stride, int n) {
  const int t = blockIdx.x * (256 / ROUTE_FEW) + threadIdx.x / ROUTE_FEW;
  route_few(r, logits + (size_t)min(t, n - 1) * logit_stride, t, t < n);
}

extern "C" int tp_moe_route(const float* logits, int logit_stride, const float* correction, int experts, int top, int groups,
                            int keep, float* dense, int* ids, float* weights, int n, int score_kind, int group_best,
                            int normalize, float sum_eps, float scale, const float* logit_bias, hipStream_t s) {
  TP_REQUIRE(n >= 0 && experts > 0 && top > 0 && top <= experts && logit_stride >= experts, "moe_route: bad sizes");
  TP_REQUIRE(experts <= TP_WAVE * ROUTE_PER_LANE, "moe_route: %d experts exceed %d", experts, TP_WAVE * ROUTE_PER_LANE);
  TP_REQUIRE(groups <= 1 || (experts % groups == 0 && keep >= 1 && keep <= groups), "moe_route: bad groups");
  TP_REQUIRE((score_kind == 0 || score_kind == 1) && group_best >= 1, "moe_route: bad score kind or group_best");
  if (n == 0) return 0;
  const size_t shmem = sizeof(float) * 4 * (size_t)(experts + (groups > 1 ? groups : 1));
  // (as many experts a lane as there are: eight experts in four groups, eight tokens, 7.9 -> 7.5 us with one instead of eight)
  const Route r = {correction, logit_bias, experts, top, groups, keep, score_kind, group_best, normalize, sum_eps, scale, dense, ids, weights};
#define ROUTE(L) hipLaunchKernelGGL(moe_route_kernel<L>, dim3((n + 3) / 4), dim3(256), shmem, s, r, logits, logit_stride, n)
  if (experts <= ROUTE_FEW)
    hipLaunchKernelGGL(moe_route_few_kernel, dim3((n + 256 / ROUTE_FEW - 1) / (256 / ROUTE_FEW)), dim3(256), 0, s, r, logits, logit_stride, n);
  else if (experts <= TP_WAVE) ROUTE(1);
  else if (experts <= 2 * TP_WAVE) ROUTE(2);
  else ROUTE(ROUTE_PER_LANE);
#undef ROUTE
  TP_CHECK_LAUNCH("moe_route");
  return 0;
}

// ---- rows sorted by expert --------------------------------------------------------------------
// For steps of many rows the chosen (token, expert) pairs are brought into the order of the experts, so that
// every expert is one product over its own rows.  ids [n, top] lists each token's experts; pair p = t * top + k.
// moe_plan: counts[e] = pairs of expert e, rank[p] = how many pairs of the same expert come before p (in the order
// of p), so the order inside an expert's rows is the order of the tokens whatever else the batch holds; then
// offsets[e] = pairs of the experts before e.  One block per expert walks all pairs; a one-block kernel adds up.
__global__ __launch_bounds__(256) void moe_rank_kernel(const int* __restrict__ ids, int pairs, int* __restrict__ counts,
                                                       int* __restrict__ rank) {
  __shared__ int wave_total[4];
  const int e = blockIdx.x, lane = threadIdx.x % TP_WAVE, wave = threadIdx.x / TP_WAVE;
  int base = 0;
  for (int p0 = 0; p0 < pairs; p0 += 256) {
    const int p = p0 + threadIdx.x;
    const bool mine = p < pairs && ids[p] == e;
    const unsigned long long mask = __ballot(mine);
    const int before = __popcll(mask & ((1ull << lane) - 1ull));
    __syncthreads();   // (the totals of the chunk before have been read)
    if (lane == 0) wave_total[wave] = __popcll(mask);
    __syncthreads();
    int prior = 0, total = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      if (w < wave) prior += wave_total[w];
      total += wave_total[w];
    }
    if (mine) rank[p] = base + prior + before;
    base += total;
  }
  if (threadIdx.x == 0) counts[e] = base;
}

__global__ void moe_offsets_kernel(const int* __restrict__ counts, int* __restrict__ offsets, int experts) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  int acc = 0;
  for (int e = 0; e < experts; ++e) {
    offsets[e] = acc;
    acc += counts[e];
  }
  offsets[experts] = acc;
}

extern "C" int tp_moe_plan(const int* ids, int n, int top, int experts, int* counts, int* offsets, int* rank, hipStream_t s) {
  TP_REQUIRE(n >= 0 && top > 0 && experts > 0 && (long)n * top < 0x7fffffffL, "moe_plan: bad sizes");
  hipLaunchKernelGGL(moe_rank_kernel, dim3(experts), dim3(256), 0, s, ids, n * top, counts, rank);
  hipLaunchKernelGGL(moe_offsets_kernel, dim3(1), dim3(64), 0, s, counts, offsets, experts);
  TP_CHECK_LAUNCH("moe_plan");
  return 0;
}

// xg[offsets[ids[p]] + rank[p]] = x[p / top] (rows of 4-byte words); row_of[p] remembers the place.
__global__ void moe_gather_kernel(const uint32_t* __restrict__ x, const int* __restrict__ ids, const int* __restrict__ rank,
                                  const int* __restrict__ offsets, uint32_t* __restrict__ xg, int* __restrict__ row_of, int top,
                                  int words) {
  const int p = blockIdx.x;
  const int row = offsets[ids[p]] + rank[p];
  if (threadIdx.x == 0) row_of[p] = row;
  const uint32_t* src = x + (size_t)(p / top) * words;
  uint32_t* dst = xg + (size_t)row * words;
  for (int c = threadIdx.x; c < words; c += blockDim.x) dst[c] = src[c];
}

// the same in 16-byte pieces
__global__ void moe_gather16_kernel(const uint4* __restrict__ x, const int* __restrict__ ids, const int* __restrict__ rank,
                                    const int* __restrict__ offsets, uint4* __restrict__ xg, int* __restrict__ row_of, int top,
                                    int pieces) {
  const int p = blockIdx.x;
  const int row = offsets[ids[p]] + rank[p];
  if (threadIdx.x == 0) row_of[p] = row;
  for (int c = threadIdx.x; c < pieces; c += blockDim.x) xg[(size_t)row * pieces + c] = x[(size_t)(p / top) * pieces + c];
}

extern "C" int tp_moe_gather(const void* x, const int* ids, const int* rank, const int* offsets, void* xg, int* row_of, int n, int top,
                             int row_bytes, hipStream_t s) {
  TP_REQUIRE(n >= 0 && top > 0 && row_bytes > 0 && row_bytes % 4 == 0, "moe_gather: rows must be a multiple of four bytes");
  if (n == 0) return 0;
  if (row_bytes % 16 == 0 && (((uintptr_t)x | (uintptr_t)xg) & 15) == 0) {
    hipLaunchKernelGGL(moe_gather16_kernel, dim3(n * top), dim3(row_bytes / 16 >= 256 ? 256 : 64), 0, s, (const uint4*)x, ids, rank, offsets,
                       (uint4*)xg, row_of, top, row_bytes / 16);
    TP_CHECK_LAUNCH("moe_gather");
    return 0;
  }
  hipLaunchKernelGGL(moe_gather_kernel, dim3(n * top), dim3(row_bytes / 4 >= 256 ? 256 : 64), 0, s, (const uint32_t*)x, ids, rank, offsets,
                     (uint32_t*)xg, row_of, top, row_bytes / 4);
  TP_CHECK_LAUNCH("moe_gather");
  return 0;
}

// y[t] (+)= sum_k weights[t, k] * yg[row_of[t, k]], k ascending.
__global__ void moe_scatter_kernel(const float* __restrict__ yg, const int* __restrict__ row_of, const float* __restrict__ weights,
                                   float* __restrict__ y, int top, int width, int accumulate) {
  const int t = blockIdx.x;
  for (int c = threadIdx.x; c < width; c += blockDim.x) {
    float acc = accumulate ? y[(size_t)t * width + c] : 0.f;
    for (int k = 0; k < top; ++k) acc = fmaf(weights[(size_t)t * top + k], yg[(size_t)row_of[(size_t)t * top + k] * width + c], acc);
    y[(size_t)t * width + c] = acc;
  }
}

// the same, four neighbouring columns a thread (the same sums in the same order): 2,048 tokens of two experts, 4,096 columns, 30 -> 23 us
__global__ __launch_bounds__(256) void moe_scatter4_kernel(const float* __restrict__ yg, const int* __restrict__ row_of,
                                                           const float* __restrict__ weights, float* __restrict__ y, int top, int width,
                                                           int accumulate) {
  const int t = blockIdx.x, c = (blockIdx.y * 256 + threadIdx.x) * 4;
  if (c >= width) return;
  float4* out = (float4*)(y + (size_t)t * width + c);
  float4 acc = accumulate ? *out : make_float4(0.f, 0.f, 0.f, 0.f);
  for (int k = 0; k < top; ++k) {
    const float w = weights[(size_t)t * top + k];
    const float4 v = *(const float4*)(yg + (size_t)row_of[(size_t)t * top + k] * width + c);
    acc = make_float4(fmaf(w, v.x, acc.x), fmaf(w, v.y, acc.y), fmaf(w, v.z, acc.z), fmaf(w, v.w, acc.w));
  }
  *out = acc;
}

extern "C" int tp_moe_scatter(const float* yg, const int* row_of, const float* weights, float* y, int n, int top, int width,
                              int accumulate, hipStream_t s) {
  TP_REQUIRE(n >= 0 && top > 0 && width > 0, "moe_scatter: bad sizes");
  if (n == 0) return 0;
  if (width % 4 == 0 && width <= 65535 * 1024 && (((uintptr_t)yg | (uintptr_t)y) & 15) == 0) {
    hipLaunchKernelGGL(moe_scatter4_kernel, dim3(n, (width + 1023) / 1024), dim3(256), 0, s, yg, row_of, weights, y, top, width, accumulate);
    TP_CHECK_LAUNCH("moe_scatter");
    return 0;
  }
  hipLaunchKernelGGL(moe_scatter_kernel, dim3(n), dim3(width >= 256 ? 256 : 64), 0, s, yg, row_of, weights, y, top, width, accumulate);
  TP_CHECK_LAUNCH("moe_scatter");
  return 0;
}

// out[e][t][c] = a[t][e * ff + c] * dense[t][e]: the activations of all experts of a few rows, each expert's as rows
// of its own, times the token's weight for the expert (zero where it was not chosen); formed in float32, rounded once.
template <typename T>
__global__ void moe_spread_kernel(const T* __restrict__ a, const float* __restrict__ dense, T* __restrict__ out, int n, int experts,
                                  int ff, size_t total) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const int c = (int)(i % ff);
  const size_t te = i / ff;
  const int e = (int)(te % experts);
  const size_t t = te / experts;
  from_float(out + ((size_t)e * n + t) * ff + c, to_float(a[i]) * dense[t * experts + e]);
}

extern "C" int tp_moe_spread(const void* a, int dt, const float* dense, void* out, int n, int experts, int ff, hipStream_t s) {
  TP_REQUIRE(n >= 0 && experts > 0 && ff > 0, "moe_spread: bad sizes");
  if (n == 0) return 0;
  const size_t total = (size_t)n * experts * ff;
  const dim3 grid((unsigned)((total + 255) / 256));
  if (dt == TP_F32)
    hipLaunchKernelGGL(moe_spread_kernel<float>, grid, dim3(256), 0, s, (const float*)a, dense, (float*)out, n, experts, ff, total);
  else if (dt == TP_BF16)
    hipLaunchKernelGGL(moe_spread_kernel<bf16_t>, grid, dim3(256), 0, s, (const bf16_t*)a, dense, (bf16_t*)out, n, experts, ff, total);
  else
    TP_REQUIRE(false, "moe_spread: unknown dtype %d", dt);
  TP_CHECK_LAUNCH("moe_spread");
  return 0;
}

// ---- RMS norm in equal parts of a run of columns ----------------------------------------------
// The `width` columns from col0 on of float32 rows [*, x_stride] are split into `groups` equal consecutive parts;
// each part is divided by its own sqrt(mean(part^2) + eps) and the whole multiplied by w [width].  `rows` (optional)
// picks the input row of each output row; out [n_out, width].  One block per output row, a wave per part in turn.
template <typename TO>
__global__ __launch_bounds__(256) void group_rmsnorm_kernel(const float* __restrict__ x, size_t x_stride, int col0,
                                                            const float* __restrict__ w, const int* __restrict__ rows,
                                                            TO* __restrict__ out, int width, int groups, float eps) {
  const int r = blockIdx.x;
  const float* xr = x + (size_t)(rows ? rows[r] : r) * x_stride + col0;
  TO* o = out + (size_t)r * width;
  const int wave = threadIdx.x / TP_WAVE, lane = threadIdx.x % TP_WAVE, waves = blockDim.x / TP_WAVE;
  const int per = width / groups;
  for (int g = wave; g < groups; g += waves) {
    const float* p = xr + (size_t)g * per;
    float ss = 0.f;
    for (int i = lane; i < per; i += TP_WAVE) ss = fmaf(p[i], p[i], ss);
    ss = wave_sum(ss);
    const float scale = 1.0f / sqrtf(ss / (float)per + eps);
    for (int i = lane; i < per; i += TP_WAVE) from_float(o + (size_t)g * per + i, p[i] * scale * w[(size_t)g * per + i]);
  }
}

// The same, a part in the registers of one wave (WAVES 1: four parts a block) or of a block of four (parts of a whole row), read
// once in pieces of four elements (parts a multiple of four, at most WAVES * 256 * NV).  Only the order of the sum of squares
// differs from the kernel above.
template <typename TO, int NV, int WAVES>
__global__ __launch_bounds__(256) void group_rmsnorm_reg_kernel(const float* __restrict__ x, size_t x_stride, int col0,
                                                                const float* __restrict__ w, const int* __restrict__ rows,
                                                                TO* __restrict__ out, int width, int groups, float eps) {
  __shared__ float scratch[32];
  constexpr int T = WAVES * TP_WAVE;
  const int r = blockIdx.x, g = WAVES == 1 ? blockIdx.y * 4 + threadIdx.x / TP_WAVE : blockIdx.y;
  if (g >= groups) return;       // (a wave of its own: no barrier follows)
  const int tid = threadIdx.x % T, per = width / groups, p4 = per / 4;
  const float* p = x + (size_t)(rows ? rows[r] : r) * x_stride + col0 + (size_t)g * per;
  float4 v[NV], wv[NV];
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int c = k * T + tid;
    if (c < p4) {
      v[k] = *(const float4*)(p + 4 * c);
      wv[k] = *(const float4*)(w + (size_t)g * per + 4 * c);
    }
  }
#pragma unroll
  for (int k = 0; k < NV; ++k)
    if (k * T + tid < p4) {
      ss = fmaf(v[k].x, v[k].x, ss);
      ss = fmaf(v[k].y, v[k].y, ss);
      ss = fmaf(v[k].z, v[k].z, ss);
      ss = fmaf(v[k].w, v[k].w, ss);
    }
  if constexpr (WAVES == 1)
    ss = wave_sum(ss);
  else
    ss = block_sum(ss, scratch);
  const float scale = 1.0f / sqrtf(ss / (float)per + eps);
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int c = k * T + tid;
    if (c < p4)
      from_float4(out + (size_t)r * width + (size_t)g * per + 4 * c, v[k].x * scale * wv[k].x, v[k].y * scale * wv[k].y,
                  v[k].z * scale * wv[k].z, v[k].w * scale * wv[k].w);
  }
}

template <typename TO>
static bool launch_group_rmsnorm_reg(const float* x, size_t x_stride, int col0, const float* w, const int* rows, void* out, int n_out,
                                     int width, int groups, float eps, hipStream_t s) {
  const int per = width / groups;
  if (per % 4 != 0 || x_stride % 4 != 0 || col0 % 4 != 0 || (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15) != 0 || groups > 65535 * 4)
    return false;
#define GN(NV, WAVES, GY)                                                                                                         do {                                                                                                                              hipLaunchKernelGGL((group_rmsnorm_reg_kernel<TO, NV, WAVES>), dim3(n_out, GY), dim3(256), 0, s, x, x_stride, col0, w, rows,                        (TO*)out, width, groups, eps);                                                                               return true;                                                                                                                  } while (0)
  // (a part of up to 512 by one wave: 4,096 in eight parts, eight rows, 11 -> 4.5 us; larger ones by a block: 1,024 in one part, four
  // rows, 9.7 -> 4.5 us)
  if (per <= 256) GN(1, 1, (groups + 3) / 4);
  if (per <= 512) GN(2, 1, (groups + 3) / 4);
  if (groups > 65535) return false;
  if (per <= 1024) GN(1, 4, groups);
  if (per <= 2048) GN(2, 4, groups);
  if (per <= 4096) GN(4, 4, groups);
  if (per <= 8192) GN(8, 4, groups);
#undef GN
  return false;
}

extern "C" int tp_group_rmsnorm(const float* x, size_t x_stride, int col0, const float* w, const int* rows, void* out, int out_dt,
                                int n_out, int width, int groups, float eps, hipStream_t s) {
  TP_REQUIRE(n_out >= 0 && width > 0 && groups > 0 && width % groups == 0 && col0 >= 0 && x_stride >= (size_t)col0 + width,
             "group_rmsnorm: bad sizes");
  if (n_out == 0) return 0;
  TP_REQUIRE(out_dt == TP_F32 || out_dt == TP_BF16, "group_rmsnorm: unknown dtype %d", out_dt);
  if (out_dt == TP_F32 ? launch_group_rmsnorm_reg<float>(x, x_stride, col0, w, rows, out, n_out, width, groups, eps, s)
                       : launch_group_rmsnorm_reg<bf16_t>(x, x_stride, col0, w, rows, out, n_out, width, groups, eps, s)) {
    TP_CHECK_LAUNCH("group_rmsnorm");
    return 0;
  }
  const int threads = groups >= 4 ? 256 : (groups * TP_WAVE);
  if (out_dt == TP_F32)
    hipLaunchKernelGGL(group_rmsnorm_kernel<float>, dim3(n_out), dim3(threads), 0, s, x, x_stride, col0, w, rows, (float*)out, width, groups, eps);
  else
    hipLaunchKernelGGL(group_rmsnorm_kernel<bf16_t>, dim3(n_out), dim3(threads), 0, s, x, x_stride, col0, w, rows, (bf16_t*)out, width, groups, eps);
  TP_CHECK_LAUNCH("group_rmsnorm");
  return 0;
}

// ---- what sublayers read of normed rows: the rows plus a short convolution of them over time ---
// x float32 [n, width]; w [subs, taps, width] (tap-major; the last tap is the current token's).  For sublayer s:
// out_s[t, c] = x[t, c] + sum_k w[s, k, c] * x[t - (taps - 1 - k), c], the rows before a run's first token coming from
// the request's state row (from element state_off on: [taps - 1, width], oldest first; zeros for a fresh request).
// The sublayers read the same rows, so one state serves them all; a second kernel leaves the run's last rows there.
template <typename TO>
__global__ void residual_conv_kernel(const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ state,
                                     size_t state_stride, size_t state_off, const int* __restrict__ cu_seqlens,
                                     const int* __restrict__ token_req, const int* __restrict__ state_slots, TO* __restrict__ out,
                                     size_t out_stride_sub, int width, int taps, int subs, int channel_blocks) {
  const int t = blockIdx.x / channel_blocks;
  const int c = (blockIdx.x % channel_blocks) * blockDim.x + threadIdx.x;
  if (c >= width) return;
  const int r = token_req[t];
  const int start = cu_seqlens[r];
  const int i = t - start;
  const float* st = state + (size_t)state_slots[r] * state_stride + state_off;
  const float cur = x[(size_t)t * width + c];
  for (int sub = 0; sub < subs; ++sub) {
    float acc = 0.f;
    for (int k = 0; k < taps; ++k) {
      const int src = i - (taps - 1 - k);
      const float v = src >= 0 ? x[(size_t)(start + src) * width + c] : st[(size_t)(taps - 1 + src) * width + c];
      acc = fmaf(w[((size_t)sub * taps + k) * width + c], v, acc);
    }
    from_float(out + (size_t)sub * out_stride_sub + (size_t)t * width + c, cur + acc);
  }
}

// the same, four neighbouring channels a thread (width a multiple of four, at most four sublayers): 16-byte loads of
// the rows and the weights; the request's carried rows are read element by element (their place in the state row
// need not be aligned).  Every channel's sum is formed in the order of the kernel above: the same bits.
// SINGLE: every request brings one token; a thread is then the only reader of its channels' carried rows and moves them on
// itself, so that no second kernel follows.
#define RCONV_MAX_SUBS 4
#define RCONV_MAX_TAPS 4   // (of norm_residual_conv_kernel)
template <typename TO, bool SINGLE>
__global__ void residual_conv4_kernel(const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ state,
                                      size_t state_stride, size_t state_off, const int* __restrict__ cu_seqlens,
                                      const int* __restrict__ token_req, const int* __restrict__ state_slots, TO* __restrict__ out,
                                      size_t out_stride_sub, int width, int taps, int subs, int channel_blocks, int blocked) {
  const int t = blockIdx.x / channel_blocks;
  const int c = ((blockIdx.x % channel_blocks) * blockDim.x + threadIdx.x) * 4;
  if (c >= width) return;
  const int r = token_req[t];
  const int start = SINGLE ? t : cu_seqlens[r];
  const int i = t - start;
  float* st = state + (size_t)state_slots[r] * state_stride + state_off;
  const float4 cur = *(const float4*)(x + (size_t)t * width + c);
  float4 acc[RCONV_MAX_SUBS];
#pragma unroll
  for (int sub = 0; sub < RCONV_MAX_SUBS; ++sub) acc[sub] = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int k = 0; k < taps; ++k) {
    const int src = i - (taps - 1 - k);
    float4 v;
    if (src >= 0) {
      v = *(const float4*)(x + (size_t)(start + src) * width + c);
    } else {
      const float* p = st + (size_t)(taps - 1 + src) * width + c;
      v = make_float4(p[0], p[1], p[2], p[3]);
    }
    if (SINGLE && k > 0) {   // (place k - 1 has been read)
      float* p = st + (size_t)(k - 1) * width + c;
      p[0] = v.x;
      p[1] = v.y;
      p[2] = v.z;
      p[3] = v.w;
    }
#pragma unroll
    for (int sub = 0; sub < RCONV_MAX_SUBS; ++sub)
      if (sub < subs) {
        const float4 wv = *(const float4*)(w + ((size_t)sub * taps + k) * width + c);
        acc[sub].x = fmaf(wv.x, v.x, acc[sub].x);
        acc[sub].y = fmaf(wv.y, v.y, acc[sub].y);
        acc[sub].z = fmaf(wv.z, v.z, acc[sub].z);
        acc[sub].w = fmaf(wv.w, v.w, acc[sub].w);
      }
  }
#pragma unroll
  for (int sub = 0; sub < RCONV_MAX_SUBS; ++sub)
    if (sub < subs) {
      const size_t place = (SINGLE && (blocked >> sub & 1)) ? ((size_t)(c >> 3) * (gridDim.x / channel_blocks) + t) * 8 + (c & 7) : (size_t)t * width + c;
      from_float4(out + (size_t)sub * out_stride_sub + place, cur.x + acc[sub].x, cur.y + acc[sub].y, cur.z + acc[sub].z, cur.w + acc[sub].w);
    }
}

// The norm of a row's parts and what the sublayers read of it, single tokens: the sums of group_rmsnorm_reg_kernel and, of the same elements
// in the same thread, those of residual_conv4_kernel (the same bits; the normed rows go nowhere else), the carried rows and the
// taps requested with the row in front of the sum.  Two trips to memory and a launch instead of two of each; a captured chain, two kernels / one: 4,096 in
// eight parts, 1 / 8 / 64 rows 6.1 / 4.1, 6.3 / 4.3 and 7.1 / 4.6 us, 2,048 in eight 6.1 / 3.2 of eight rows, 1,024 5.8 / 3.2.  (With the
// taps loaded behind the sum, sublayer by sublayer, 5.9 of eight rows of 4,096.)
template <typename TO, int NV, int WAVES, int SUBS>
__global__ __launch_bounds__(256) void norm_residual_conv_kernel(const float* __restrict__ x, const float* __restrict__ nw, int groups, float eps,
                                                                 const float* __restrict__ w, float* __restrict__ state, size_t state_stride,
                                                                 size_t state_off, const int* __restrict__ token_req,
                                                                 const int* __restrict__ state_slots, TO* __restrict__ out, size_t out_stride_sub,
                                                                 int width, int taps, int blocked) {
  __shared__ float scratch[32];
  constexpr int T = WAVES * TP_WAVE;
  const int t = blockIdx.x, g = WAVES == 1 ? blockIdx.y * 4 + threadIdx.x / TP_WAVE : blockIdx.y;
  if (g >= groups) return;       // (a wave of its own: no barrier follows)
  const int tid = threadIdx.x % T, per = width / groups, p4 = per / 4;
  const float* p = x + (size_t)t * width + (size_t)g * per;
  float4 v[NV], wv[NV], old[NV][RCONV_MAX_TAPS], f[NV][SUBS][RCONV_MAX_TAPS];   // (old: the last place is the token's own row)
  float* st = state + (size_t)state_slots[token_req[t]] * state_stride + state_off + (size_t)g * per;
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int c = k * T + tid;
    if (c < p4) {
      v[k] = *(const float4*)(p + 4 * c);
      wv[k] = *(const float4*)(nw + (size_t)g * per + 4 * c);
#pragma unroll
      for (int j = 0; j < RCONV_MAX_TAPS; ++j) {
        // (places and taps beyond the last repeat one that is there and are dropped below: every load is requested before the sum)
        const float* q = st + (size_t)min(j, taps - 2) * width + 4 * c;
        old[k][j] = make_float4(q[0], q[1], q[2], q[3]);
#pragma unroll
        for (int sub = 0; sub < SUBS; ++sub)
          f[k][sub][j] = *(const float4*)(w + ((size_t)sub * taps + min(j, taps - 1)) * width + (size_t)g * per + 4 * c);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < NV; ++k)
    if (k * T + tid < p4) {
      ss = fmaf(v[k].x, v[k].x, ss);
      ss = fmaf(v[k].y, v[k].y, ss);
      ss = fmaf(v[k].z, v[k].z, ss);
      ss = fmaf(v[k].w, v[k].w, ss);
    }
  if constexpr (WAVES == 1)
    ss = wave_sum(ss);
  else
    ss = block_sum(ss, scratch);
  const float scale = 1.0f / sqrtf(ss / (float)per + eps);
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int c = k * T + tid;
    if (c >= p4) continue;
    const float4 cur = make_float4(v[k].x * scale * wv[k].x, v[k].y * scale * wv[k].y, v[k].z * scale * wv[k].z, v[k].w * scale * wv[k].w);
    const int col = g * per + 4 * c;
#pragma unroll
    for (int j = 1; j < RCONV_MAX_TAPS; ++j) {
      if (j == taps - 1) old[k][j] = cur;
      if (j < taps) {
        float* q = st + (size_t)(j - 1) * width + 4 * c;
        q[0] = old[k][j].x;
        q[1] = old[k][j].y;
        q[2] = old[k][j].z;
        q[3] = old[k][j].w;
      }
    }
#pragma unroll
    for (int sub = 0; sub < SUBS; ++sub) {
      float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int j = 0; j < RCONV_MAX_TAPS; ++j)
        if (j < taps) {
          acc.x = fmaf(f[k][sub][j].x, old[k][j].x, acc.x);
          acc.y = fmaf(f[k][sub][j].y, old[k][j].y, acc.y);
          acc.z = fmaf(f[k][sub][j].z, old[k][j].z, acc.z);
          acc.w = fmaf(f[k][sub][j].w, old[k][j].w, acc.w);
        }
      const size_t place = (blocked >> sub & 1) ? ((size_t)(col >> 3) * gridDim.x + t) * 8 + (col & 7) : (size_t)t * width + col;
      from_float4(out + (size_t)sub * out_stride_sub + place, cur.x + acc.x, cur.y + acc.y, cur.z + acc.z, cur.w + acc.w);
    }
  }
}

// x [n, width]: the norm in `groups` parts (nw, eps), then residual_conv over runs of one token (see tp_residual_conv); width / groups at most
// 4,096 and a multiple of four, 2 to RCONV_MAX_TAPS taps
extern "C" int tp_norm_residual_conv(const float* x, const float* nw, int groups, float eps, const float* w, float* state, size_t state_stride,
                                     size_t state_off, const int* token_req, const int* state_slots, void* out, int out_dt, int n, int width,
                                     int taps, int subs, int blocked, hipStream_t s) {
  TP_REQUIRE(n >= 0 && width > 0 && groups > 0 && groups <= 65535 && width % groups == 0 && width / groups % 4 == 0 && width / groups <= 4096 &&
             taps >= 2 && taps <= RCONV_MAX_TAPS && subs >= 1 && subs <= 2, "norm_residual_conv: bad sizes");
  TP_REQUIRE((((uintptr_t)x | (uintptr_t)nw | (uintptr_t)w | (uintptr_t)out) & 15) == 0, "norm_residual_conv: operands must be aligned to 16 bytes");
  TP_REQUIRE(state != nullptr && state_stride >= state_off + (size_t)(taps - 1) * width, "norm_residual_conv: state rows too short");
  TP_REQUIRE((blocked == 0 || width % 8 == 0) && (out_dt == TP_F32 || out_dt == TP_BF16), "norm_residual_conv: bad output");
  if (n == 0) return 0;
  const int per = width / groups;
  const size_t sub_stride = (size_t)n * width;
#define NRC(TO, NV, WAVES, GY)                                                                                                      \
  do {                                                                                                                              \
    if (subs == 1)                                                                                                                  \
      hipLaunchKernelGGL((norm_residual_conv_kernel<TO, NV, WAVES, 1>), dim3(n, GY), dim3(256), 0, s, x, nw, groups, eps, w, state, \
                         state_stride, state_off, token_req, state_slots, (TO*)out, sub_stride, width, taps, blocked);              \
    else                                                                                                                            \
      hipLaunchKernelGGL((norm_residual_conv_kernel<TO, NV, WAVES, 2>), dim3(n, GY), dim3(256), 0, s, x, nw, groups, eps, w, state, \
                         state_stride, state_off, token_req, state_slots, (TO*)out, sub_stride, width, taps, blocked);              \
  } while (0)
#define NRC_SIZES(TO)                                            \
  do {                                                           \
    if (per <= 256) NRC(TO, 1, 1, (groups + 3) / 4);             \
    else if (per <= 512) NRC(TO, 2, 1, (groups + 3) / 4);        \
    else if (per <= 1024) NRC(TO, 1, 4, groups);                 \
    else if (per <= 2048) NRC(TO, 2, 4, groups);                 \
    else NRC(TO, 4, 4, groups);                                  \
  } while (0)
  if (out_dt == TP_F32) NRC_SIZES(float);
  else NRC_SIZES(bf16_t);
#undef NRC_SIZES
#undef NRC
  TP_CHECK_LAUNCH("norm_residual_conv");
  return 0;
}

__global__ void residual_conv_state_kernel(const float* __restrict__ x, float* __restrict__ state, size_t state_stride,
                                           size_t state_off, const int* __restrict__ cu_seqlens,
                                           const int* __restrict__ state_slots, int width, int taps) {
  const int r = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= width) return;
  const int start = cu_seqlens[r], len = cu_seqlens[r + 1] - start;
  if (len <= 0) return;
  float* st = state + (size_t)state_slots[r] * state_stride + state_off;
  // in place, ascending: entry j takes entry j + len of the old state or a row of the run; entries below j are never read again
  for (int j = 0; j < taps - 1; ++j) {
    const int src = len - (taps - 1) + j;
    st[(size_t)j * width + c] = src >= 0 ? x[(size_t)(start + src) * width + c] : st[(size_t)(j + len) * width + c];
  }
}

extern "C" int tp_residual_conv(const float* x, const float* w, float* state, size_t state_stride, size_t state_off,
                                const int* cu_seqlens, const int* token_req, const int* state_slots, void* out, int out_dt, int n,
                                int n_req, int width, int taps, int subs, int max_run, int blocked, hipStream_t s) {
  // max_run: the longest run of the step, 0: not known.  blocked (runs of one token): bit i, sublayer i's rows leave k-blocked,
  // [width / 8, n, 8]
  TP_REQUIRE(n >= 0 && n_req >= 0 && width > 0 && taps >= 1 && subs >= 1, "residual_conv: bad sizes");
  TP_REQUIRE(state_stride >= state_off + (size_t)(taps - 1) * width, "residual_conv: state rows too short");
  if (n == 0) return 0;
  const int threads = width >= 256 ? 256 : 64;
  const int cb = (width + threads - 1) / threads;
  TP_REQUIRE(cb <= 65535 && (long)n * cb < 0x7fffffffL, "residual_conv: too many channels or tokens");
  const size_t sub_stride = (size_t)n * width;
  TP_REQUIRE(out_dt == TP_F32 || out_dt == TP_BF16, "residual_conv: unknown dtype %d", out_dt);
  if (width % 4 == 0 && subs <= RCONV_MAX_SUBS && (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15) == 0) {
    const int quads = width / 4;
    const int qthreads = quads >= 256 ? 256 : 64;
    const int qb = (quads + qthreads - 1) / qthreads;
    const dim3 grid((unsigned)((long)n * qb));
#define RCONV(TO, SINGLE)                                                                                                           \
  hipLaunchKernelGGL((residual_conv4_kernel<TO, SINGLE>), grid, dim3(qthreads), 0, s, x, w, state, state_stride, state_off, cu_seqlens, \
                     token_req, state_slots, (TO*)out, sub_stride, width, taps, subs, qb, blocked)
    if (max_run == 1) {
      if (out_dt == TP_F32) RCONV(float, true);
      else RCONV(bf16_t, true);
      TP_CHECK_LAUNCH("residual_conv");
      return 0;
    }
    TP_REQUIRE(blocked == 0, "residual_conv: only runs of one token leave k-blocked");
    if (out_dt == TP_F32) RCONV(float, false);
    else RCONV(bf16_t, false);
#undef RCONV
  } else if (blocked != 0)
    TP_REQUIRE(false, "residual_conv: rows of these sizes do not leave k-blocked");
  else if (out_dt == TP_F32)
    hipLaunchKernelGGL(residual_conv_kernel<float>, dim3((unsigned)((long)n * cb)), dim3(threads), 0, s, x, w, state, state_stride,
                       state_off, cu_seqlens, token_req, state_slots, (float*)out, sub_stride, width, taps, subs, cb);
  else if (out_dt == TP_BF16)
    hipLaunchKernelGGL(residual_conv_kernel<bf16_t>, dim3((unsigned)((long)n * cb)), dim3(threads), 0, s, x, w, state, state_stride,
                       state_off, cu_seqlens, token_req, state_slots, (bf16_t*)out, sub_stride, width, taps, subs, cb);
  else
    TP_REQUIRE(false, "residual_conv: unknown dtype %d", out_dt);
  if (taps > 1 && n_req > 0)
    hipLaunchKernelGGL(residual_conv_state_kernel, dim3(n_req, cb), dim3(threads), 0, s, x, state, state_stride, state_off, cu_seqlens,
                       state_slots, width, taps);
  TP_CHECK_LAUNCH("residual_conv");
  return 0;
}

// ---- one row of a table added to every row of the stream --------------------------------------
__global__ void add_row_kernel(float* __restrict__ h, const float* __restrict__ row, size_t total, int width) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < total) h[i] += row[i % width];
}

extern "C" int tp_add_row(float* h, const float* row, int n, int width, hipStream_t s) {
  TP_REQUIRE(n >= 0 && width > 0, "add_row: bad sizes");
  if (n == 0) return 0;
  const size_t total = (size_t)n * width;
  TP_REQUIRE((total + 255) / 256 < 0x7fffffffUL, "add_row: too many elements");
  hipLaunchKernelGGL(add_row_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, h, row, total, width);
  TP_CHECK_LAUNCH("add_row");
  return 0;
}

// ---- rows of q | k | v for an attention whose keys and values are expanded from a latent --------
// Per token: q [heads, key] comes from the projection's rows as it stands (key = rot + dim elements a head, the
// rotated ones first); head h's key is the ONE shared rotated part (rot elements of the projection's rows, not yet
// rotated) followed by its own dim unrotated elements of the expansion `up` ([heads * dim | heads * vdim] a row);
// its value the head's vdim elements of `up`.  out [n, 2 * heads * key + heads * vdim] float32, the layout the
// rotation-and-store kernel takes.
__global__ void latent_rows_kernel(const float* __restrict__ proj, size_t proj_stride, int q_col0, int rot_col0,
                                   const float* __restrict__ up, size_t up_stride, float* __restrict__ out, int heads, int dim,
                                   int rot, int vdim) {
  const int t = blockIdx.x;
  const int key = rot + dim, qk = heads * key, width = 2 * qk + heads * vdim;
  const float* pr = proj + (size_t)t * proj_stride;
  const float* ur = up + (size_t)t * up_stride;
  float* o = out + (size_t)t * width;
  for (int i = threadIdx.x; i < width; i += blockDim.x) {
    float v;
    if (i < qk) {
      v = pr[q_col0 + i];
    } else if (i < 2 * qk) {
      const int h = (i - qk) / key, d = (i - qk) % key;
      v = d < rot ? pr[rot_col0 + d] : ur[h * dim + d - rot];
    } else {
      v = ur[heads * dim + i - 2 * qk];
    }
    o[i] = v;
  }
}

// The same, four neighbouring elements a thread (sizes, strides and first columns multiples of four): a grid over the columns too, so
// that a few rows are not a loop of one block each (eight rows of 12,288: 17 -> 5 us).
__global__ __launch_bounds__(256) void latent_rows4_kernel(const float* __restrict__ proj, size_t proj_stride, int q_col0, int rot_col0,
                                                           const float* __restrict__ up, size_t up_stride, float* __restrict__ out,
                                                           int heads, int dim, int rot, int vdim) {
  const int t = blockIdx.x;
  const int key = rot + dim, qk = heads * key, width = 2 * qk + heads * vdim;
  const int i = (blockIdx.y * 256 + threadIdx.x) * 4;
  if (i >= width) return;
  const float* pr = proj + (size_t)t * proj_stride;
  const float* ur = up + (size_t)t * up_stride;
  const float* src;
  if (i < qk) {
    src = pr + q_col0 + i;
  } else if (i < 2 * qk) {
    const int h = (i - qk) / key, d = (i - qk) % key;
    src = d < rot ? pr + rot_col0 + d : ur + h * dim + d - rot;
  } else {
    src = ur + heads * dim + i - 2 * qk;
  }
  *(float4*)(out + (size_t)t * width + i) = *(const float4*)src;
}

extern "C" int tp_latent_rows(const float* proj, size_t proj_stride, int q_col0, int rot_col0, const float* up, size_t up_stride,
                              float* out, int n, int heads, int dim, int rot, int vdim, hipStream_t s) {
  TP_REQUIRE(n >= 0 && heads > 0 && dim > 0 && rot >= 0 && vdim > 0 && q_col0 >= 0 && rot_col0 >= 0, "latent_rows: bad sizes");
  TP_REQUIRE(proj_stride >= (size_t)q_col0 + (size_t)heads * (rot + dim) && proj_stride >= (size_t)rot_col0 + rot &&
                 up_stride >= (size_t)heads * (dim + vdim), "latent_rows: rows too short");
  if (n == 0) return 0;
  if (dim % 4 == 0 && rot % 4 == 0 && vdim % 4 == 0 && q_col0 % 4 == 0 && rot_col0 % 4 == 0 && proj_stride % 4 == 0 && up_stride % 4 == 0 &&
      (((uintptr_t)proj | (uintptr_t)up | (uintptr_t)out) & 15) == 0 && (2 * (long)heads * (rot + dim) + (long)heads * vdim + 1023) / 1024 <= 65535) {
    const int width = 2 * heads * (rot + dim) + heads * vdim;
    hipLaunchKernelGGL(latent_rows4_kernel, dim3(n, (width + 1023) / 1024), dim3(256), 0, s, proj, proj_stride, q_col0, rot_col0, up, up_stride,
                       out, heads, dim, rot, vdim);
    TP_CHECK_LAUNCH("latent_rows");
    return 0;
  }
  hipLaunchKernelGGL(latent_rows_kernel, dim3(n), dim3(256), 0, s, proj, proj_stride, q_col0, rot_col0, up, up_stride, out, heads, dim,
                     rot, vdim);
  TP_CHECK_LAUNCH("latent_rows");
  return 0;
}

// ---- norm per head on projected rows, in place --------------------------------------------------
// rows float32 [n, stride]: the `heads` heads of `dim` columns from col0 on become x / sqrt(mean(x^2) + eps) * w[d]
// (one weight [dim] for all of them).  Queries and keys of an attention are two calls' worth of columns, so the entry
// point takes two runs of heads, each with its weight.  One wave per (token, head).
__global__ __launch_bounds__(256) void head_rmsnorm_kernel(float* __restrict__ rows, size_t stride, int col_a, int heads_a,
                                                           const float* __restrict__ w_a, int col_b, int heads_b,
                                                           const float* __restrict__ w_b, int dim, float eps, long pairs) {
  const long p = (long)blockIdx.x * 4 + threadIdx.x / TP_WAVE;
  const int lane = threadIdx.x % TP_WAVE;
  if (p >= pairs) return;
  const int per = heads_a + heads_b;
  const long t = p / per;
  const int hh = (int)(p % per);
  float* x = rows + (size_t)t * stride + (hh < heads_a ? col_a + (size_t)hh * dim : col_b + (size_t)(hh - heads_a) * dim);
  const float* w = hh < heads_a ? w_a : w_b;
  float ss = 0.f;
  for (int d = lane; d < dim; d += TP_WAVE) ss = fmaf(x[d], x[d], ss);
  ss = wave_sum(ss);
  const float rstd = 1.0f / sqrtf(ss / (float)dim + eps);
  for (int d = lane; d < dim; d += TP_WAVE) x[d] = x[d] * rstd * w[d];
}

extern "C" int tp_head_rmsnorm(float* rows, size_t stride, int col_a, int heads_a, const float* w_a, int col_b, int heads_b,
                               const float* w_b, int dim, float eps, int n, hipStream_t s) {
  TP_REQUIRE(n >= 0 && dim > 0 && heads_a >= 0 && heads_b >= 0 && col_a >= 0 && col_b >= 0, "head_rmsnorm: bad sizes");
  TP_REQUIRE((size_t)col_a + (size_t)heads_a * dim <= stride && (size_t)col_b + (size_t)heads_b * dim <= stride, "head_rmsnorm: rows too short");
  TP_REQUIRE((heads_a == 0 || w_a) && (heads_b == 0 || w_b), "head_rmsnorm: a run of heads needs its weight");
  const long pairs = (long)n * (heads_a + heads_b);
  if (pairs == 0) return 0;
  TP_REQUIRE((pairs + 3) / 4 < 0x7fffffffL, "head_rmsnorm: too many rows");
  hipLaunchKernelGGL(head_rmsnorm_kernel, dim3((unsigned)((pairs + 3) / 4)), dim3(256), 0, s, rows, stride, col_a, heads_a, w_a, col_b,
                     heads_b, w_b, dim, eps, pairs);
  TP_CHECK_LAUNCH("head_rmsnorm");
  return 0;
}

// ---- one vector a token into the cache, as key and as value ------------------------------------------
// c [n, dim] goes to cache place slots[t] of keys [page, 1, page_size, dim] and of transposed values
// [page, 1, dim, page_size]: an attention whose keys are its values reads both with the ordinary kernels.
template <typename T>
__global__ void vector_store_kernel(const T* __restrict__ c, const int* __restrict__ slots, T* __restrict__ k_cache,
                                    T* __restrict__ v_cache, size_t total, int dim, int page_size) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const size_t t = i / dim;
  const int d = (int)(i % dim);
  const int slot = slots[t];
  const size_t page = slot / page_size;
  const int off = slot % page_size;
  const T v = c[i];
  k_cache[(page * page_size + off) * dim + d] = v;
  v_cache[(page * dim + d) * page_size + off] = v;
}

extern "C" int tp_vector_store(const void* c, int dt, const int* slots, void* k_cache, void* v_cache, int n, int dim, int page_size,
                               hipStream_t s) {
  TP_REQUIRE(n >= 0 && dim > 0 && page_size > 0, "vector_store: bad sizes");
  const size_t total = (size_t)n * dim;
  if (total == 0) return 0;
  const dim3 grid((unsigned)((total + 255) / 256));
  if (dt == TP_F32)
    hipLaunchKernelGGL(vector_store_kernel<float>, grid, dim3(256), 0, s, (const float*)c, slots, (float*)k_cache, (float*)v_cache, total, dim, page_size);
  else if (dt == TP_BF16)
    hipLaunchKernelGGL(vector_store_kernel<bf16_t>, grid, dim3(256), 0, s, (const bf16_t*)c, slots, (bf16_t*)k_cache, (bf16_t*)v_cache, total, dim, page_size);
  else
    TP_REQUIRE(false, "vector_store: unknown dtype %d", dt);
  TP_CHECK_LAUNCH("vector_store");
  return 0;
}

// Of few rows the two norms in front of an attention over latents in one launch: block (t, 0) norms the query's latent into cq, block (t, 1)
// the key's and puts it into the cache.  The parts, their lanes and the order of their sums are group_rmsnorm_reg_kernel's (up to 512 columns
// a wave, else the block), so the bits are those of the three launches, each a few trips to memory around
// some kilobytes.  Latents of 1,024 and 128, a captured chain, three kernels / one: 1 / 4 / 64 rows 5.0 / 2.2, 5.7 / 2.3 and 6.0 / 2.7 us.
template <typename TO>
__global__ __launch_bounds__(256) void latent_norms_kernel(const float* __restrict__ rows, size_t stride, int q_col0, int q_dim,
                                                           const float* __restrict__ q_w, int c_col0, int c_dim, const float* __restrict__ c_w,
                                                           float eps, TO* __restrict__ cq, const int* __restrict__ slots,
                                                           TO* __restrict__ k_cache, TO* __restrict__ v_cache, int page_size) {
  __shared__ float scratch[32];
  const int t = blockIdx.x, per = blockIdx.y == 0 ? q_dim : c_dim, p4 = per / 4, lanes = per <= 512 ? TP_WAVE : 256, tid = threadIdx.x;
  if (tid >= lanes) return;      // (a wave by itself: no barrier follows)
  const float* p = rows + (size_t)t * stride + (blockIdx.y == 0 ? q_col0 : c_col0);
  const float* w = blockIdx.y == 0 ? q_w : c_w;
  const int slot = blockIdx.y == 0 ? 0 : slots[t];
  float4 v[4], wv[4];
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int c = k * lanes + tid;
    if (c < p4) {
      v[k] = *(const float4*)(p + 4 * c);
      wv[k] = *(const float4*)(w + 4 * c);
    }
  }
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (k * lanes + tid < p4) {
      ss = fmaf(v[k].x, v[k].x, ss);
      ss = fmaf(v[k].y, v[k].y, ss);
      ss = fmaf(v[k].z, v[k].z, ss);
      ss = fmaf(v[k].w, v[k].w, ss);
    }
  ss = lanes == TP_WAVE ? wave_sum(ss) : block_sum(ss, scratch);
  const float scale = 1.0f / sqrtf(ss / (float)per + eps);
  const size_t page = slot / page_size;
  const int off = slot % page_size;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int c = k * lanes + tid;
    if (c >= p4) continue;
    const float4 o = make_float4(v[k].x * scale * wv[k].x, v[k].y * scale * wv[k].y, v[k].z * scale * wv[k].z, v[k].w * scale * wv[k].w);
    if (blockIdx.y == 0) {
      from_float4(cq + (size_t)t * per + 4 * c, o.x, o.y, o.z, o.w);
    } else {
      from_float4(k_cache + (page * page_size + off) * per + 4 * c, o.x, o.y, o.z, o.w);
      TO* vp = v_cache + (page * per + 4 * c) * page_size + off;
      from_float(vp, o.x);
      from_float(vp + page_size, o.y);
      from_float(vp + 2 * (size_t)page_size, o.z);
      from_float(vp + 3 * (size_t)page_size, o.w);
    }
  }
}

// rows float32 [n, stride]: columns q_col0 .. + q_dim normed (q_w, eps) -> cq [n, q_dim]; c_col0 .. + c_dim normed (c_w) -> cache places (see
// tp_vector_store).  All of type dt; dimensions, columns and stride multiples of four, at most 4,096 columns each.
extern "C" int tp_latent_norms(const float* rows, size_t stride, int q_col0, int q_dim, const float* q_w, int c_col0, int c_dim, const float* c_w,
                               float eps, void* cq, const int* slots, void* k_cache, void* v_cache, int dt, int n, int page_size, hipStream_t s) {
  TP_REQUIRE(n >= 0 && n <= 65535 && q_dim > 0 && c_dim > 0 && q_dim <= 4096 && c_dim <= 4096 && page_size > 0 && q_col0 >= 0 && c_col0 >= 0 &&
             (q_dim | c_dim | q_col0 | c_col0) % 4 == 0 && stride % 4 == 0 && stride >= (size_t)q_col0 + q_dim && stride >= (size_t)c_col0 + c_dim,
             "latent_norms: bad sizes");
  TP_REQUIRE((((uintptr_t)rows | (uintptr_t)q_w | (uintptr_t)c_w | (uintptr_t)cq | (uintptr_t)k_cache) & 15) == 0,
             "latent_norms: operands must be aligned to 16 bytes");
  if (n == 0) return 0;
  const dim3 grid(n, 2);
  if (dt == TP_F32)
    hipLaunchKernelGGL(latent_norms_kernel<float>, grid, dim3(256), 0, s, rows, stride, q_col0, q_dim, q_w, c_col0, c_dim, c_w, eps, (float*)cq, slots,
                       (float*)k_cache, (float*)v_cache, page_size);
  else if (dt == TP_BF16)
    hipLaunchKernelGGL(latent_norms_kernel<bf16_t>, grid, dim3(256), 0, s, rows, stride, q_col0, q_dim, q_w, c_col0, c_dim, c_w, eps, (bf16_t*)cq,
                       slots, (bf16_t*)k_cache, (bf16_t*)v_cache, page_size);
  else
    TP_REQUIRE(false, "latent_norms: unknown dtype %d", dt);
  TP_CHECK_LAUNCH("latent_norms");
  return 0;
}
