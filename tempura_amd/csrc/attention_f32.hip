// Float32 attention over the paged cache on the matrix cores (v_mfma_f32_16x16x4_f32), for heads of 32, 64, 96 or 128 with values of
// the same size and pages of a multiple of 16 keys; other shapes run the general kernel (attention.hip).
//
// A block takes one kv head of one request and 16 query rows, a row being a (token, head of the group) pair, tokens first; its four
// waves share the keys: a wave takes the 16-key tiles whose number is its own modulo four, keeps a running softmax for the 16 rows,
// and the block adds the four at the end.  Scores are formed transposed (keys as the instruction's rows), so that a lane's four
// results are the probabilities of the four keys that it multiplies with the values next: nothing passes between lanes but the
// maximum.  Keys and values go from memory into operand registers as they lie: 16 rows of 64 bytes a load for keys, a contiguous
// KB for values (pages hold them transposed).
// Single tokens under a long context also cut the keys over blocks (splits), which leave unnormalised sums for a second kernel.
// Tiles, waves and splits go by a key's absolute place, so a row's sum does not depend on where a portion begins; a step of single tokens
// alone cuts its keys by its longest context and the number of requests, which changes rounding only.
//
// Measured with 24 heads of 128 in 8 groups: two single tokens behind 310 keys 318 -> 11 us (the general kernel is one wave a token
// and head whose lanes walk whole keys), a prompt step of 611 tokens 2,366 -> 59 us.
#include <math.h>

#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define AF_WAVES 4
#define AF_ROWS 16
#define AF_KEYS 16

struct AttnF32Args {
  const float* q;
  const float* k_cache;
  const float* v_cache;
  const int* block_tables;
  const int* cu_seqlens;
  const int* context_lens;
  float* out;
  float* scratch;
  const float* dist_bias;
  const float* sink;
  int table_width, n_heads, n_kv, page_size, window, bias_len, keep_first, chunk, splits;
  float scale, softcap;
};

template <int D>
__global__ __launch_bounds__(256) void attn_f32_kernel(AttnF32Args a) {
  constexpr int NT = D / 16;
  __shared__ float so[AF_WAVES][AF_ROWS][D + 4];   // (rows four banks apart)
  __shared__ float sm[AF_WAVES][AF_ROWS], sl[AF_WAVES][AF_ROWS];
  const int lane = threadIdx.x % TP_WAVE, wave = threadIdx.x / TP_WAVE;
  const int col = lane % 16, quad = lane / 16;
  const int kvh = blockIdx.x % a.n_kv, r = blockIdx.y, split = blockIdx.z;
  const int group = a.n_heads / a.n_kv;
  const int q_start = a.cu_seqlens[r], q_len = a.cu_seqlens[r + 1] - q_start;
  const int tiles = (int)(gridDim.x / a.n_kv);
  // (the last query rows see the most keys: their blocks go first)
  const int row0 = (tiles - 1 - (int)(blockIdx.x / a.n_kv)) * AF_ROWS, rows = q_len * group;
  if (row0 >= rows) return;
  const int first_pos = a.context_lens[r] - q_len;
  auto low_of = [&](int pos) { return a.chunk > 0 ? pos / a.chunk * a.chunk : (a.window > 0 && pos - a.window + 1 > 0) ? pos - a.window + 1 : 0; };
  // this lane's query row (rows past the request's last repeat it and are not stored)
  const int row = min(row0 + col, rows - 1);
  const int tok = row / group, head = kvh * group + row % group;
  const int pos = first_pos + tok, lo = low_of(pos);
  const int kept = (a.keep_first > 0 && lo > 0) ? min(a.keep_first, lo) : 0;    // keys 0..kept-1 that the window has left behind
  // the tile's keys: what its first row sees from, what its last row sees to
  const int tok_a = row0 / group, tok_b = min(row0 + AF_ROWS, rows) - 1;
  const int pos_b = first_pos + tok_b / group, lo_a = low_of(first_pos + tok_a), lo_b = low_of(pos_b);
  const int kept_b = (a.keep_first > 0 && lo_b > 0) ? min(a.keep_first, lo_b) : 0;
  const int* table = a.block_tables + (size_t)r * a.table_width;

  f32x4 qr[NT];
  {
    const float* p = a.q + ((size_t)(q_start + tok) * a.n_heads + head) * D + quad * 4;
#pragma unroll
    for (int t = 0; t < NT; ++t) qr[t] = *(const f32x4*)(p + 16 * t);
  }
  f32x4 o[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) o[t] = (f32x4)(0.f);
  float m = -INFINITY, l = 0.f;

  // two runs of tiles: the kept first keys, then the window (or everything); a tile that both touch belongs to the second
  const int main_t0 = lo_a / AF_KEYS, main_t1 = pos_b / AF_KEYS;
  const int kept_t1 = min((kept_b + AF_KEYS - 1) / AF_KEYS, main_t0);
  const int step = AF_WAVES * a.splits, mine = split * AF_WAVES + wave;
  for (int seg = 0; seg < 2; ++seg) {
    const int t0 = seg == 0 ? 0 : main_t0, t1 = seg == 0 ? kept_t1 - 1 : main_t1;
    for (int tile = t0 + ((mine - t0) % step + step) % step; tile <= t1; tile += step) {
      const int key0 = tile * AF_KEYS;
      const int page = table[key0 / a.page_size], off = key0 % a.page_size;
      const size_t base = (size_t)page * a.n_kv + kvh;
      const float* kp = a.k_cache + (base * a.page_size + off + col) * D + quad * 4;
      const float* vp = a.v_cache + (base * D + col) * a.page_size + off + quad * 4;
      f32x4 kr[NT], vr[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) kr[t] = *(const f32x4*)(kp + 16 * t);
#pragma unroll
      for (int t = 0; t < NT; ++t) vr[t] = *(const f32x4*)(vp + (size_t)16 * t * a.page_size);
      f32x4 s0 = (f32x4)(0.f), s1 = (f32x4)(0.f);
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (t % 2 == 0)
            s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[t][j], qr[t][j], s0, 0, 0, 0);
          else
            s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[t][j], qr[t][j], s1, 0, 0, 0);
        }
      float s[4], mt = -INFINITY;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = key0 + quad * 4 + i;
        float v = (s0[i] + s1[i]) * a.scale;
        if (a.softcap > 0.f) v = a.softcap * tanhf(v / a.softcap);
        const bool sees = key <= pos && (key >= lo || key < kept);
        if (a.dist_bias != nullptr && sees) v += a.dist_bias[(size_t)head * a.bias_len + min(pos - key, a.bias_len - 1)];
        s[i] = sees ? v : -INFINITY;
        mt = fmaxf(mt, s[i]);
      }
      mt = fmaxf(mt, __shfl_xor(mt, 16, TP_WAVE));
      mt = fmaxf(mt, __shfl_xor(mt, 32, TP_WAVE));
      const float m_new = fmaxf(m, mt);
      const float alpha = m_new == -INFINITY ? 1.f : expf(m - m_new);
      float p[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        p[i] = s[i] == -INFINITY ? 0.f : expf(s[i] - m_new);
        l = i == 0 ? fmaf(l, alpha, p[i]) : l + p[i];
      }
      m = m_new;
      // A place of the tile that no row of the block sees holds anything (the rest of a page, a page given back): no
      // product may touch it.  A key that some row sees and another does not is multiplied with a zero there, which is only
      // right while its values are finite; a tile with others is added row by row below.
      float odd = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int key = key0 + quad * 4 + j;
        const bool any = key <= pos_b && (key >= lo_a || key < kept_b);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          if (!any) vr[t][j] = 0.f;
          odd = fmaf(vr[t][j], 0.f, odd);
        }
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) o[t] *= alpha;
      if (!__any(odd != 0.f)) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int j = 0; j < 4; ++j) o[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[t][j], p[j], o[t], 0, 0, 0);
      } else {
        f32x4 keep[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) keep[t] = o[t];
        for (int c = 0; c < 16; ++c) {
          const int cpos = __shfl(pos, c, TP_WAVE), clo = __shfl(lo, c, TP_WAVE), ckept = __shfl(kept, c, TP_WAVE);
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            f32x4 sum = keep[t];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const int key = key0 + quad * 4 + j;
              const bool sees = key <= cpos && (key >= clo || key < ckept);
              sum = __builtin_amdgcn_mfma_f32_16x16x4f32(sees ? vr[t][j] : 0.f, p[j], sum, 0, 0, 0);
            }
            if (col == c) o[t] = sum;
          }
        }
      }
    }
  }
  // one row's sums lie in the four lanes of its column
  l += __shfl_xor(l, 16, TP_WAVE);
  l += __shfl_xor(l, 32, TP_WAVE);
  if (quad == 0) {
    sm[wave][col] = m;
    sl[wave][col] = l;
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) *(f32x4*)&so[wave][col][16 * t + quad * 4] = o[t];
  __syncthreads();
  for (int i = threadIdx.x; i < AF_ROWS * D; i += 256) {
    const int c = i / D, d = i % D;
    if (row0 + c >= rows) continue;
    const int ct = (row0 + c) / group, ch = kvh * group + (row0 + c) % group;
    float mg = sm[0][c];
#pragma unroll
    for (int w = 1; w < AF_WAVES; ++w) mg = fmaxf(mg, sm[w][c]);
    if (a.splits == 1 && a.sink != nullptr) mg = fmaxf(mg, a.sink[ch]);
    float lg = 0.f, og = 0.f;
#pragma unroll
    for (int w = 0; w < AF_WAVES; ++w) {
      const float f = sm[w][c] == -INFINITY ? 0.f : expf(sm[w][c] - mg);
      lg = fmaf(f, sl[w][c], lg);
      og = fmaf(f, so[w][c][d], og);
    }
    if (a.splits == 1) {
      if (a.sink != nullptr) lg += expf(a.sink[ch] - mg);
      a.out[((size_t)(q_start + ct) * a.n_heads + ch) * D + d] = og * (1.0f / lg);
    } else {      // (single tokens only: one row a head)
      float* b = a.scratch + (((size_t)r * a.n_heads + ch) * a.splits + split) * (D + 2);
      b[d] = og;
      if (d == 0) {
        b[D] = mg;
        b[D + 1] = lg;
      }
    }
  }
}

// Adds the splits of a single token's head in ascending order.  grid: (requests, heads), a thread for every element in whole waves, each
// of which works out the splits' factors for itself.  The first splits' values are requested with their maxima and sums, so a head of up to eight splits is
// one trip to memory: with the attention in front, captured, 24 heads of 128, two requests of 300 / 700 keys 14.2 / 17.1 -> 12.0 / 13.4 us, one of
// 2,000 22.0 -> 15.6 (a wave a head and the values behind the factors before).
template <int D>
__global__ __launch_bounds__((D + 63) / 64 * 64) void attn_f32_combine_kernel(const float* __restrict__ scratch, const int* __restrict__ cu_seqlens,
                                                                           float* __restrict__ out, int n_heads, int splits,
                                                                           const float* __restrict__ sink) {
  constexpr int EARLY = 8;
  const int r = blockIdx.x, h = blockIdx.y, lane = threadIdx.x % TP_WAVE, d = min((int)threadIdx.x, D - 1);
  const float* base = scratch + ((size_t)r * n_heads + h) * splits * (D + 2);
  float v[EARLY];
#pragma unroll
  for (int s = 0; s < EARLY; ++s) v[s] = base[(size_t)min(s, splits - 1) * (D + 2) + d];
  // (at most 64 splits: a lane holds one's maximum and sum)
  const float ms = lane < splits ? base[(size_t)lane * (D + 2) + D] : -INFINITY;
  const float ls = lane < splits ? base[(size_t)lane * (D + 2) + D + 1] : 0.f;
  const float sk = sink != nullptr ? sink[h] : -INFINITY;
  const int t = cu_seqlens[r];
  const float mg = fmaxf(wave_max(ms), sk);
  const float f = ms == -INFINITY ? 0.f : expf(ms - mg);
  const float inv = 1.0f / (wave_sum(f * ls) + (sink != nullptr ? expf(sk - mg) : 0.f));
  float og = 0.f;
#pragma unroll
  for (int s = 0; s < EARLY; ++s)
    if (s < splits) og = fmaf(lane_value(f, s), v[s], og);
  for (int s = EARLY; s < splits; ++s) og = fmaf(lane_value(f, s), base[(size_t)s * (D + 2) + d], og);
  if ((int)threadIdx.x < D) out[((size_t)t * n_heads + h) * D + d] = og * inv;
}

template <int D>
static void launch_f32(const AttnF32Args& a, int n_req, int max_q_len, hipStream_t s) {
  const int tiles = (max_q_len * (a.n_heads / a.n_kv) + AF_ROWS - 1) / AF_ROWS;
  hipLaunchKernelGGL((attn_f32_kernel<D>), dim3((unsigned)tiles * a.n_kv, n_req, a.splits), dim3(256), 0, s, a);
  if (a.splits > 1)
    hipLaunchKernelGGL((attn_f32_combine_kernel<D>), dim3(n_req, a.n_heads), dim3((D + 63) / 64 * 64), 0, s, a.scratch, a.cu_seqlens, a.out, a.n_heads,
                       a.splits, a.sink);
}

// Returns -1 for shapes that the general kernel runs.  num_splits > 1 (every request brings one token): scratch of
// n_req * n_heads * num_splits * (head_dim + 2) floats.
int tp_paged_attention_f32(const float* q, const float* k_cache, const float* v_cache, const int* block_tables, int table_width,
                           const int* cu_seqlens, const int* context_lens, float* out, int n_tokens, int n_req, int n_heads, int n_kv,
                           int head_dim, int value_dim, int page_size, float scale, int window, int max_q_len, int num_splits,
                           float* scratch, const float* dist_bias, int bias_len, int keep_first, const float* sink, int chunk,
                           float softcap, hipStream_t s) {
  if (head_dim != value_dim || page_size % AF_KEYS != 0 || n_req > 65535 || max_q_len <= 0 || n_tokens < n_req ||
      ((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache) % 16 != 0)
    return -1;
  const bool split = num_splits > 1 && scratch != nullptr && max_q_len == 1 && n_tokens == n_req;
  const AttnF32Args a = {q,    k_cache,    v_cache,     block_tables, cu_seqlens, context_lens, out,        scratch, dist_bias,
                         sink, table_width, n_heads,    n_kv,         page_size,  window,       bias_len,   keep_first, chunk,
                         split ? num_splits : 1, scale, softcap};
  switch (head_dim) {
    case 32: launch_f32<32>(a, n_req, max_q_len, s); break;
    case 64: launch_f32<64>(a, n_req, max_q_len, s); break;
    case 96: launch_f32<96>(a, n_req, max_q_len, s); break;
    case 128: launch_f32<128>(a, n_req, max_q_len, s); break;
    default: return -1;
  }
  TP_CHECK_LAUNCH("paged_attention (float32)");
  return 0;
}
