// bfloat16 products on the gfx950 matrix cores: out[M, N] (+)= x[M, K] * w[N, K]^T,
// float32 accumulation (v_mfma_f32_16x16x32_bf16).
//
// Three kernels:
//  * few (M <= 16, a decode step): bound by the weights' stream from memory.  A block owns 16 output columns (16 weight rows); its eight
//    waves split K in runs of 128 and each lane pulls its 16 bytes of a weight row straight from global memory into the MFMA operand
//    registers (no LDS: a weight is used by exactly one wave).  Partial tiles are summed through LDS in the order of the waves, so results
//    are deterministic and a row's value does not depend on the other rows of the batch.
//  * skinny (17 to 64 rows without scratch): the same with two to four tiles of rows.
//  * tiled (M > 64, prefill): 128x128 block tile, 64x64 per wave, K in steps of 64 (or
//    32), operands staged through padded LDS tiles; the next tile is fetched into
//    registers while the current one is multiplied.
// Fragment layout of the 16x16x32 instruction: lane l holds row (l % 16) of its operand
// and 8 consecutive k at (l / 16) * 8; the result lane l holds rows (l / 16) * 4 + r,
// r = 0..3, of column l % 16.
#include "activations.h"
#include <cstddef>
#include <tuple>
#include <type_traits>

#include "common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

// OUT_SWIGLU: the weight rows alternate eight gate rows and eight up rows; output column
// 8*b + i is silu(row 16*b + i) * (row 16*b + 8 + i), stored as bfloat16 [M, N / 2].
enum { OUT_F32 = 0, OUT_BF16 = 1, OUT_ACC_F32 = 2, OUT_SWIGLU = 3 };


__device__ inline bf16x8_t as_frag(u32x4_t v) { return __builtin_bit_cast(bf16x8_t, v); }

// the gated SiLU without constants: the products of a few rows have only this gate in their common kernels (their time is the weights'
// stream, and the general gate's constants in the epilogue cost every one of them half a microsecond, measured); with constants they take
// the kernels of the split epilogue
__device__ inline float silu_mul(float g, float u) {
  return g * u * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g * -1.4426950408889634f));
}

// the same with constants, as the activation's own kernel has it: the same bits as the product and that kernel
__device__ inline float gated_few(float g, float u, const GateAct& a) { return gated_value(g, u, a.slope, a.limit, a.offset); }

// A decode product reads every weight once per step and never again before the whole model has streamed through
// the caches: the loads say so (nontemporal), which leaves the cache lines to the activations and measures faster
// on a chain of streaming kernels (5.7 -> 6.4 TB/s on products of these sizes).
#ifndef TP_WEIGHTS_TEMPORAL
#define TP_WLOAD(p) __builtin_nontemporal_load(p)
#else
#define TP_WLOAD(p) (*(p))
#endif

// Layouts of bfloat16 activations of at most 16 rows.  Row-major [M, K], or k-blocked [K / 8, M, 8]:
// eight consecutive k of all rows side by side, so that the operand fragments that the lanes of a
// wave fetch straight from global memory (16 bytes per row and k group) lie next to each other.
// Layout of a weight.  Row-major [N, K], or tiled (N % 16 == 0, K % 64 == 0): [N / 16][K / 32][64][8], the operand
// fragment of the MFMA for 16 weight rows and 32 of k as one run of 1,024 bytes, lane l's eight elements (row l % 16,
// k group l / 16) at l * 16.  A wave's load of a fragment then covers eight whole cache lines instead of 64-byte
// pieces of sixteen rows, which is what the address path of a CU can keep up with when the weights stream from HBM
// (the down projection of 8 rows: 26.0 -> 23.4 us), and a stage of the pipelined kernels is a plain copy.
enum { X_KBLOCKED = 1, OUT_KBLOCKED = 2, W_TILED = 4, XG_KBLOCKED = 8 };

__device__ inline void store_gated(void* out, int layout, int M, int width, int m, int col, float v) {
  const size_t idx = (layout & OUT_KBLOCKED) ? ((size_t)(col >> 3) * M + m) * 8 + (col & 7) : (size_t)m * width + col;
  ((bf16_t*)out)[idx] = float_to_bf16(v);
}

__device__ inline void store_out(void* out, int mode, size_t idx, float v) {
  if (mode == OUT_F32)
    ((float*)out)[idx] = v;
  else if (mode == OUT_BF16)
    ((bf16_t*)out)[idx] = float_to_bf16(v);
  else
    ((float*)out)[idx] += v;
}

// mode OUT_SPLIT (see GateAct); layout OUT_KBLOCKED: the activated columns k-blocked
__device__ inline void store_split(void* out, int layout, const GateAct& ga, int M, int m, int n, float v) {
  if (n < ga.act_cols)
    store_gated(out, layout, M, ga.act_ld, m, n, ga.act_kind1 == 0 ? relu_squared(v) : act_f(v, ga.act_kind1 - 1));
  else
    ga.side[(size_t)m * ga.side_ld + n - ga.act_cols] = v;
}

// What the rotation of one column of one row reads besides its sums, requested before the weights.
struct RopeIn {
  float2 cs;
  int slot;
};
__device__ inline RopeIn rope_request(const RopeOut& rp, int m, int n) {
  RopeIn in = {make_float2(1.f, 0.f), rp.slots[m]};
  const int d = n % rp.head_dim;
  if (rp.cos_sin != nullptr) in.cs = rp.cos_sin[(size_t)m * (rp.rotary_dim >> 1) + min(d, max(rp.rotary_dim - 1, 0)) / 2];
  return in;
}

// v: this lane's sum of column n of row m; other: the sum of column n ^ 1 (the partner of a rotary pair)
__device__ inline void rope_store(const RopeOut& rp, const RopeIn& in, int m, int n, float v, float other) {
  const int h = n / rp.head_dim, d = n % rp.head_dim;
  float y = v;
  if (h < rp.n_heads + rp.n_kv && d < rp.rotary_dim) {
    float c = in.cs.x, sn = in.cs.y;
    if (rp.cos_sin == nullptr) rope_cos_sin(rp.positions[m], rp.inv_freq[d >> 1], rp.factor, c, sn);
    // the pair is (x0, x1) = (even column, odd column): x0 c - x1 s and x0 s + x1 c
    y = (d & 1) ? other * sn + v * c : v * c - other * sn;
  }
  if (h < rp.n_heads) {
    rp.q_out[((size_t)m * rp.n_heads + h) * rp.head_dim + d] = float_to_bf16(y);
    return;
  }
  const size_t page = (size_t)(in.slot / rp.page_size), off = (size_t)(in.slot % rp.page_size);
  if (h < rp.n_heads + rp.n_kv)
    rp.k_cache[((page * rp.n_kv + (h - rp.n_heads)) * rp.page_size + off) * rp.head_dim + d] = float_to_bf16(y);
  else
    rp.v_cache[((page * rp.n_kv + (h - rp.n_heads - rp.n_kv)) * rp.head_dim + d) * rp.page_size + off] = float_to_bf16(y);
}

// A root-mean-square norm split over two products (rows of at most 16 tokens).  The product that
// adds into the residual stream h also writes xg = bfloat16(h * norm weight) and, per block and row,
// the sum of squares of the columns it owns (NormPrep).  The product that consumes xg adds those
// partial sums in a fixed order and multiplies its float32 result rows by rsqrt(mean square + eps)
// (RowScale): the norm kernel between the two products is gone, and the scale is applied in float32
// after the sum instead of before the rounding to bfloat16.
struct NormPrep {
  const float* w;    // norm weight [N]; nullptr: no preparation
  bf16_t* xg;        // [M, N]
  float* ss;         // [M, blocks]
};
struct RowScale {
  const float* ss;   // [M, count] partial sums of squares; nullptr: no scaling
  int count;
  float inv_k, eps;
};

// v of another lane of the same four, by the order of a DPP quad_perm (0xB1: neighbours swapped, 0x4E: pairs swapped)
template <int ORDER>
__device__ inline float quad_swapped(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ORDER, 0xf, 0xf, false));
}

// ---- few rows ---------------------------------------------------------------------------
// What happens to the sums: stored (float32, bfloat16, added into float32), the gated SiLU, added into the stream with the next norm prepared,
// rotation and cache, the split epilogue (mode OUT_SPLIT, or a gate with constants).  Each is a kernel of its own: what one of them
// needs of constants and branches costs every other half a microsecond.  (The split epilogue: an activation's own launch and trip through memory, 4.9 us behind
// a product of one row, is gone.)
enum { FEW_STORE, FEW_SWIGLU, FEW_POST, FEW_ROPE, FEW_SPLIT };
#define FEW_WAVES 8
#define FEW_RED 80      // floats between the four column groups of a wave's tile: a thread a (row, column) then reads without more conflicts than 64 lanes have anyway

// The wave's share of K: runs of four steps of 32 (256 contiguous bytes of each weight row), run r to wave r % 8, one run on its way at a
// time, and nothing between the loads but their addresses: a loop whose loads stand behind conditions (a second run only where there is one, a chunk of rows
// only for the threads that copy it) waits for every load on its way at each join, and what the epilogue reads of the kernel's arguments must not
// stand in front of the first load either.  From memory, a captured chain, float32 results, against two runs at a time with such conditions
// (plain reads of the same bytes: 4.5, 6.1, 16.7, 6.5, 9.2, 19.5 us): one row of K x N 3,072 x 3,072 6.6 -> 5.0 us, 3,072 x 5,120 10.2 -> 7.4, 3,072 x 16,384 20.0 -> 16.4,
// 4,096 x 4,096 7.9 -> 6.9, 8,192 x 3,072 11.5 -> 9.7, 14,336 x 4,096 21.1 -> 18.9; eight rows 6.2 -> 5.2, 9.4 -> 8.3, 18.6 -> 16.8, 8.8 -> 6.9,
// 13.5 -> 10.4, 21.8 -> 18.9.  Sixteen waves with a run each: the same within 3 %.
// P > 0: row-major rows through LDS, P pieces of 16 bytes a thread (padded rows: 16-byte reads of 16 rows then hit different banks); 0: straight from memory.
// PRE: the norm of the rows is finished here (RowScale).
// What the end reads of the arguments stands in one structure behind those that arrive in registers.  It is read through few_end(), behind the first
// requests: the compiler asks for a structure's members at the start of a kernel and waits for them at its first branch.
struct FewEnd {
  RowScale pre;
  NormPrep post;
  RopeOut rp;
};
// (the kernel's arguments as they lie in memory: each on its own alignment, in their order.  A parameter of another type or order, here or there,
// does not compile: see the types that gemm_few_kernel is compared with)
struct FewArgs {
  const bf16_t *x, *w;
  void* out;
  int M, N, K, mode, layout;
  FewEnd end;
};
#define FEW_END_AT offsetof(FewArgs, end)
template <typename T>
using constant_ptr = const __attribute__((address_space(4))) T*;
__device__ inline constant_ptr<FewEnd> few_end() {
  constant_ptr<char> args = (constant_ptr<char>)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(args)::"memory");
  return (constant_ptr<FewEnd>)(args + FEW_END_AT);
}

// P < 0: row-major rows through LDS in chunks of 1,024 of K, two of them in LDS, the weights of four and the rows of two on their way.  DEEP: two runs on
// their way (K of at least 16 runs).
#define FEW_CHUNK 1024
#define FEW_CHUNK_LD (FEW_CHUNK * 2 + 16)
template <int P, int KIND, bool PRE, bool WT, bool DEEP>
__global__ __launch_bounds__(FEW_WAVES * 64) void gemm_few_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, void* __restrict__ out, int M,
                                                                  int N, int K, int mode, int layout, FewEnd) {
  constexpr int T = FEW_WAVES * 64;
  extern __shared__ __attribute__((aligned(16))) unsigned char rows_lds[];
  __shared__ __attribute__((aligned(16))) float red[FEW_WAVES][4 * FEW_RED];
  __shared__ float rstd[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, row = min(lane & 15, M - 1), n0 = blockIdx.x * 16;
  const int steps = K / 32, ld = K * 2 + 16;
  u32x4_t xv[P > 0 ? P : 1];
  if constexpr (P > 0) {
    const int total = M * (K / 8);
#pragma unroll
    for (int i = 0; i < P; ++i) xv[i] = ((const u32x4_t*)x)[min(i * T + tid, total - 1)];
  }
  const u32x4_t* wp = WT ? (const u32x4_t*)(w + (size_t)n0 * K) + lane : (const u32x4_t*)(w + (size_t)min(n0 + (lane & 15), N - 1) * K) + g;
  constexpr int wstep = WT ? 64 : 4;   // u32x4 units per 32 of k
  const bool blocked = (layout & X_KBLOCKED) != 0;
  const u32x4_t* xp = (const u32x4_t*)x + (blocked ? g * M + row : row * (K / 8) + g);
  const int xstep = blocked ? 4 * M : 4;
  u32x4_t a[P < 0 ? 4 : DEEP ? 2 : 1][4], b[P < 0 || DEEP ? 2 : 1][4];
  auto request = [&](int d, int run) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; ++u) a[d][u] = TP_WLOAD(wp + (size_t)(run * 4 + u) * wstep);
    if constexpr (P == 0) {
#pragma unroll
      for (int u = 0; u < 4; ++u) b[d][u] = xp[(size_t)(run * 4 + u) * xstep];
    }
  };
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](int d, int run) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const u32x4_t bv = P == 0 ? b[d][u] : *(const u32x4_t*)(rows_lds + (size_t)row * ld + (run * 4 + u) * 64 + g * 16);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(a[d][u]), as_frag(bv), acc, 0, 0, 0);
    }
  };
  // (P < 0) run `wave` of a chunk, and the chunk's rows: 32 threads a row, four pieces of 16 bytes each.  What lies behind the end of K repeats its last
  // pieces and is not multiplied.
  const int chunks = (K + FEW_CHUNK - 1) / FEW_CHUNK, copy_row = tid / 32, copy_at = tid % 32;
  auto request_weights = [&](int d, int chunk) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; ++u) a[d][u] = TP_WLOAD(wp + (size_t)min(chunk * (FEW_CHUNK / 32) + wave * 4 + u, steps - 1) * wstep);
  };
  auto request_rows = [&](int d, int chunk) __attribute__((always_inline)) {
    if (copy_row >= M) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) b[d][i] = ((const u32x4_t*)x)[copy_row * (K / 8) + min(chunk * (FEW_CHUNK / 8) + i * 32 + copy_at, K / 8 - 1)];
  };
  const int runs = steps / 4;      // (whole ones)
  if constexpr (P < 0) {
    request_rows(0, 0);
    request_weights(0, 0);
    if (chunks > 1) {
      request_rows(1, 1);
      request_weights(1, 1);
    }
    if (chunks > 2) request_weights(2, 2);
    if (chunks > 3) request_weights(3, 3);
  } else if constexpr (DEEP) {
    request(0, wave);
    request(1, wave + FEW_WAVES);
  } else {
    if (wave < runs) request(0, wave);
  }
  const constant_ptr<FewEnd> end = few_end();
  const RowScale pre = {end->pre.ss, end->pre.count, end->pre.inv_k, end->pre.eps};
  const NormPrep post = {end->post.w, end->post.xg, end->post.ss};
  RopeOut rp;
  if constexpr (KIND == FEW_ROPE || KIND == FEW_SPLIT) __builtin_memcpy(&rp, (const void*)(uintptr_t)&end->rp, sizeof(rp));
  // what the end needs besides the sums.  A thread of the first four waves has row m, column n; the others repeat them.
  const int m = (tid >> 4) & 15, n = n0 + (tid & 15), mc = min(m, M - 1), nc = min(n, N - 1);
  float held = 0.f, wn = 0.f;
  if constexpr (KIND == FEW_POST) {
    held = ((const float*)out)[(size_t)mc * N + nc];
    wn = post.w[nc];
  }
  RopeIn turn;
  if constexpr (KIND == FEW_ROPE) turn = rope_request(rp, mc, nc);
  float parts[2][4] = {};      // wave v adds up rows v and v + 8: a lane has every 64th partial sum
  if constexpr (PRE) {
    const int last = pre.count - 1;
#pragma unroll
    for (int j = 0; j < 4; ++j) parts[0][j] = pre.ss[min(wave, M - 1) * pre.count + min(lane + 64 * j, last)];
    if (M > 8) {
#pragma unroll
      for (int j = 0; j < 4; ++j) parts[1][j] = pre.ss[min(wave + 8, M - 1) * pre.count + min(lane + 64 * j, last)];
    }
  }
  if constexpr (P > 0) {
    const int kc = K / 8, total = M * kc;
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const int e = min(i * T + tid, total - 1), r = M == 1 ? 0 : e / kc;
      *(u32x4_t*)(rows_lds + (size_t)r * ld + (e - r * kc) * 16) = xv[i];
    }
    // (not __syncthreads: it would wait for the weights as well)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }
  if constexpr (P < 0) {
    for (int chunk0 = 0; chunk0 < chunks; chunk0 += 4) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int chunk = chunk0 + c;
        if (chunk < chunks) {
          unsigned char* rows = rows_lds + (c & 1) * 16 * FEW_CHUNK_LD;
          if (copy_row < M) {
#pragma unroll
            for (int i = 0; i < 4; ++i) *(u32x4_t*)(rows + copy_row * FEW_CHUNK_LD + (i * 32 + copy_at) * 16) = b[c & 1][i];
          }
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
          if (chunk + 2 < chunks) request_rows(c & 1, chunk + 2);
          const int s0 = chunk * (FEW_CHUNK / 32) + wave * 4;
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (s0 + u < steps)
              acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(a[c][u]), as_frag(*(const u32x4_t*)(rows + row * FEW_CHUNK_LD + (wave * 4 + u) * 64 + g * 16)),
                                                            acc, 0, 0, 0);
          if (chunk + 4 < chunks) request_weights(c, chunk + 4);
        }
      }
    }
  } else if constexpr (DEEP) {
    multiply(0, wave);
    multiply(1, wave + FEW_WAVES);
  } else {
    if (wave < runs) multiply(0, wave);
  }
  int run = wave + (DEEP ? 2 : 1) * FEW_WAVES;
  if constexpr (PRE) {
    // The order is part of the result: 32 sums of every 32nd partial sum, then these in ascending order.  (The same time as a sum in pairs: one row of the
    // 3B shape 1,462.1 and 1,461.5 us, eight of the 8B shape 3,262 and 3,269.  What costs is asking for the partial sums in front of the weights, 1,476,
    // and this work in waves that have no row, 1,489.)  Those behind the first 256, of a K of more than 4,096, are asked for with a run of weights each 256, which
    // every wave has (asked for one after the other / so: K x N 8,192 x 3,072 one row 14.2 / 11.1 us, nine 16.1 / 12.8, 14,336 x 4,096 26.9 / 20.8 and 29.5 / 22.1,
    // 8,192 x 28,672 76.6 / 70.7 and 74.8 / 70.7, 28,672 x 8,192 76.7 / 72.1 and 85.2 / 73.3; 6,144 x 6,144 16.1 / 14.9, but three rows 16.2 / 16.8).
    float sums[2] = {0.f, 0.f};
    auto add_parts = [&](int c0) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if (wave + 8 * i >= M) break;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const LanePair both = lanes_32(c0 + lane + 64 * j < pre.count ? parts[i][j] : 0.f);
          sums[i] += both.a;
          sums[i] += both.b;
        }
      }
    };
    auto request_parts = [&](int c0) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) parts[i][j] = pre.ss[min(wave + 8 * i, M - 1) * pre.count + min(c0 + lane + 64 * j, pre.count - 1)];
    };
    add_parts(0);
    if (wave < M) {
      int c0 = 256;
      for (; P >= 0 && c0 < pre.count && run < runs; c0 += 256, run += FEW_WAVES) {
        request(0, run);
        request_parts(c0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(0, run);
        add_parts(c0);
      }
      for (; c0 < pre.count; c0 += 256) {
        request_parts(c0);
        add_parts(c0);
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (wave + 8 * i >= M) break;
      float total = 0.f;
#pragma unroll
      for (int c = 0; c < 32; ++c) total += lane_value(sums[i], c);
      if (lane == 0) rstd[wave + 8 * i] = rsqrtf(total * pre.inv_k + pre.eps);
    }
  }
  if constexpr (DEEP) {
    for (; run + FEW_WAVES < runs; run += 2 * FEW_WAVES) {
      request(0, run);
      request(1, run + FEW_WAVES);
      __builtin_amdgcn_sched_barrier(0);
      multiply(0, run);
      multiply(1, run + FEW_WAVES);
    }
  }
  for (; P >= 0 && run < runs; run += FEW_WAVES) {
    request(0, run);
    __builtin_amdgcn_sched_barrier(0);      // (all of a run's loads in front of its first product)
    multiply(0, run);
  }
  if (P >= 0 && wave == runs % FEW_WAVES) {      // what is left of K, fewer than four steps
    for (int st = runs * 4; st < steps; ++st) {
      const u32x4_t av = TP_WLOAD(wp + (size_t)st * wstep);
      const u32x4_t bv = P == 0 ? xp[(size_t)st * xstep] : *(const u32x4_t*)(rows_lds + (size_t)row * ld + st * 64 + g * 16);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(av), as_frag(bv), acc, 0, 0, 0);
    }
  }
  *(f32x4_t*)(&red[wave][g * FEW_RED + (lane & 15) * 4]) = acc;
  __syncthreads();
  if (wave >= 4 || wave * 4 >= M) return;
  // the waves' partial tiles in wave order
  const int at = ((tid & 15) >> 2) * FEW_RED + m * 4 + (tid & 3);
  float v = 0.f;
#pragma unroll
  for (int i = 0; i < FEW_WAVES; ++i) v += red[i][at];
  if constexpr (PRE) v *= rstd[mc];
  const bool mine = n < N && m < M;
  const bool gated = KIND == FEW_SWIGLU || (KIND == FEW_SPLIT && mode == OUT_SWIGLU);
  if (gated) {
    const float up = row_rotated<8>(v);      // a gate row's up row is eight further on
    if ((tid & 15) < 8 && n + 8 < N && m < M)
      store_gated(out, layout, M, N / 2, m, n0 / 2 + (tid & 15), KIND == FEW_SPLIT ? gated_few(v, up, rp.gate) : silu_mul(v, up));
  } else if constexpr (KIND == FEW_SPLIT) {
    if (mine) store_split(out, layout, rp.gate, M, m, n, v);
  } else if constexpr (KIND == FEW_POST) {
    // residual add, and the next norm's preparation
    const float h = held + v;
    if (mine) {
      ((float*)out)[(size_t)m * N + n] = h;
      // (k-blocked on request: the product that consumes these rows then reads them straight from memory as operands)
      post.xg[(layout & XG_KBLOCKED) ? ((size_t)(n >> 3) * M + m) * 8 + (n & 7) : (size_t)m * N + n] = float_to_bf16(h * wn);
    }
    // (in this order: pairs, fours, then the fours in ascending order)
    float sq = mine ? h * h : 0.f;
    sq += quad_swapped<0xB1>(sq);
    sq += quad_swapped<0x4E>(sq);
    sq = ((sq + row_rotated<12>(sq)) + row_rotated<8>(sq)) + row_rotated<4>(sq);
    if ((tid & 15) == 0 && m < M) post.ss[m * gridDim.x + blockIdx.x] = sq;
  } else if constexpr (KIND == FEW_ROPE) {
    const float other = quad_swapped<0xB1>(v);   // column n ^ 1
    if (mine) rope_store(rp, turn, m, n, v, other);
  } else if (mine) {
    store_out(out, mode, (size_t)m * N + n, v);
  }
}

// ---- 17 to 64 rows ------------------------------------------------------------------------
// The same without scratch for the pipelined kernels: MT 16-row tiles of activations; WAVES waves split K, DEPTH runs on their way.
// SPLIT: mode OUT_SPLIT, or OUT_SWIGLU with a gate that has constants.
template <int MT, int WAVES, int DEPTH, bool WT, bool SPLIT>
__global__ __launch_bounds__(WAVES * 64) void gemm_skinny_mfma_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                                      void* __restrict__ out, int mode, int M, int N, int K, GateAct gate) {
  __shared__ float red[WAVES][MT][256];
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int n0 = blockIdx.x * 16;
  const int kofs = (lane >> 4) * 8;
  const int wrow = min(n0 + (lane & 15), N - 1);
  const u32x4_t* wp = WT ? (const u32x4_t*)(w + (size_t)min(n0, N - 16) * K) + lane : (const u32x4_t*)(w + (size_t)wrow * K + kofs);
  constexpr int wstep = WT ? 64 : 4;   // u32x4 units per 32 of k (a compile-time stride: the four loads of a run share one address)
  const u32x4_t* xp[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) xp[t] = (const u32x4_t*)(x + (size_t)min(t * 16 + (lane & 15), M - 1) * K + kofs);
  f32x4_t acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  const int steps = K / 32;  // a step is 32 k = 4 u32x4 per row
  for (int s0 = wave * 4; s0 < steps; s0 += WAVES * 4 * DEPTH) {
    u32x4_t a[DEPTH][4];
    u32x4_t b[DEPTH][MT][4];
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        // steps past the end repeat the last one; their products are dropped below
        const int sidx = min(s0 + d * WAVES * 4 + u, steps - 1);
        a[d][u] = TP_WLOAD(wp + (size_t)sidx * wstep);
#pragma unroll
        for (int t = 0; t < MT; ++t) b[d][t][u] = xp[t][(size_t)sidx * 4];
      }
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (s0 + d * WAVES * 4 + u < steps) {
#pragma unroll
          for (int t = 0; t < MT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(a[d][u]), as_frag(b[d][t][u]), acc[t], 0, 0, 0);
        }
      }
  }
  // sum the waves' partial tiles in wave order
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wave][t][lane * 4 + r] = acc[t][r];
  __syncthreads();
  for (int e = threadIdx.x; e < MT * 256; e += WAVES * 64) {
    const int t = e / 256, q = e % 256;
    float v = 0.f;
#pragma unroll
    for (int i = 0; i < WAVES; ++i) v += red[i][t][q];
    const int l = q / 4, r = q % 4;
    const int n = n0 + (l >> 4) * 4 + r;   // weight row = output column
    const int m = t * 16 + (l & 15);
    if (SPLIT && mode == OUT_SPLIT) {
      if (n < N && m < M) store_split(out, 0, gate, M, m, n, v);
    } else if (SPLIT || mode == OUT_SWIGLU) {
      if ((l >> 4) < 2 && n + 8 < N && m < M) {       // a gate row: its up row is eight further on
        float u = 0.f;
#pragma unroll
        for (int i = 0; i < WAVES; ++i) u += red[i][t][q + 128];
        store_gated(out, 0, M, N / 2, m, n0 / 2 + (l >> 4) * 4 + r, SPLIT ? gated_few(v, u, gate) : silu_mul(v, u));
      }
    } else if (n < N && m < M) {
      store_out(out, mode, (size_t)m * N + n, v);
    }
  }
}

// ---- tiled ----------------------------------------------------------------------------
// Block of four waves (2 x 2); a wave owns WMT x WNT result tiles of 16 x 16, so the block
// tile is (32 WMT) x (32 WNT).  blockIdx.z splits K: with more than one split every block
// writes its float32 partial tile to `partial` [split, M, N] and a second kernel adds the
// splits in ascending order and applies the epilogue (so the result does not depend on timing).
// Measured on MI355X: two blocks per CU matter more than a larger tile (a 256 x 128 tile or
// a second set of prefetch registers drops occupancy to one wave per SIMD and loses a third).
template <int BK, int WMT, int WNT>
__global__ __launch_bounds__(256) void gemm_tiled_mfma_kernel(const bf16_t* __restrict__ x,
                                                              const bf16_t* __restrict__ w, void* __restrict__ out,
                                                              float* __restrict__ partial, int mode, int M, int N,
                                                              int K, int xcd_order, GateAct ga) {
  constexpr int BM = 32 * WMT, BN = 32 * WNT;
  constexpr int LD = BK + 8;            // padded row, in bf16 elements (conflict-free 16-byte reads)
  constexpr int CPR = BK / 8;           // 16-byte chunks per tile row
  constexpr int XCPT = BM * CPR / 256;  // chunks per thread, x tile
  constexpr int WCPT = BN * CPR / 256;  // chunks per thread, w tile
  __shared__ __attribute__((aligned(16))) uint16_t xs[BM * LD];
  __shared__ __attribute__((aligned(16))) uint16_t ws[BN * LD];
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int wm = wave / 2, wn = wave % 2;
  int bm = blockIdx.y, bn = blockIdx.x;
  if (xcd_order) {
    // Blocks go to the eight XCDs round robin by launch order, and each XCD has an L2 of its own.
    // XCD c takes the column blocks c, c + 8, ...; the blocks it runs at the same time form an
    // 8 x 8 patch of (row block, column block), so that every weight tile and every activation
    // tile it fetches is used by eight blocks while it is still in that L2.
    const int MB = (M + BM - 1) / BM, NB = (N + BN - 1) / BN;
    const int Q = (NB + 7) / 8, MS = (MB + 7) / 8;
    const int c = blockIdx.x % 8, j = blockIdx.x / 8;
    const int t = j / 64, r = j % 64;
    bm = (t % MS) * 8 + r % 8;
    bn = c + 8 * ((t / MS) * 8 + r / 8);
    if (bm >= MB || bn >= NB || (t / MS) * 8 + r / 8 >= Q) return;
  }
  const int m0 = bm * BM, n0 = bn * BN;
  // this block's share of K, in tiles
  const int KT_all = K / BK;
  const int per = (KT_all + gridDim.z - 1) / gridDim.z;
  const int kt_begin = blockIdx.z * per, kt_end = min(KT_all, kt_begin + per);

  f32x4_t acc[WMT][WNT];
#pragma unroll
  for (int i = 0; i < WMT; ++i)
#pragma unroll
    for (int j = 0; j < WNT; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};

  u32x4_t xr[XCPT], wr[WCPT];
  auto load_global = [&](int k0) {
#pragma unroll
    for (int i = 0; i < XCPT; ++i) {
      const int c = tid + 256 * i;
      const int gm = min(m0 + c / CPR, M - 1);
      xr[i] = *(const u32x4_t*)(x + (size_t)gm * K + k0 + (c % CPR) * 8);
    }
#pragma unroll
    for (int i = 0; i < WCPT; ++i) {
      const int c = tid + 256 * i;
      const int gn = min(n0 + c / CPR, N - 1);
      wr[i] = *(const u32x4_t*)(w + (size_t)gn * K + k0 + (c % CPR) * 8);
    }
  };
  auto store_lds = [&]() {
#pragma unroll
    for (int i = 0; i < XCPT; ++i) {
      const int c = tid + 256 * i;
      *(u32x4_t*)(&xs[(c / CPR) * LD + (c % CPR) * 8]) = xr[i];
    }
#pragma unroll
    for (int i = 0; i < WCPT; ++i) {
      const int c = tid + 256 * i;
      *(u32x4_t*)(&ws[(c / CPR) * LD + (c % CPR) * 8]) = wr[i];
    }
  };

  // The next tile travels from global memory into registers while this one is multiplied.
  if (kt_begin < kt_end) load_global(kt_begin * BK);
  for (int kt = kt_begin; kt < kt_end; ++kt) {
    store_lds();
    __syncthreads();
    if (kt + 1 < kt_end) load_global((kt + 1) * BK);
#pragma unroll
    for (int kk = 0; kk < BK / 32; ++kk) {
      bf16x8_t b[WNT];
#pragma unroll
      for (int j = 0; j < WNT; ++j)
        b[j] = as_frag(*(const u32x4_t*)(&ws[(wn * 16 * WNT + j * 16 + (lane & 15)) * LD + kk * 32 + (lane >> 4) * 8]));
#pragma unroll
      for (int i = 0; i < WMT; ++i) {
        const bf16x8_t a =
            as_frag(*(const u32x4_t*)(&xs[(wm * 16 * WMT + i * 16 + (lane & 15)) * LD + kk * 32 + (lane >> 4) * 8]));
#pragma unroll
        for (int j = 0; j < WNT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[j], acc[i][j], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  // result lane l: rows (l / 16) * 4 + r of the x tile (m), column l % 16 of the w tile (n)
#pragma unroll
  for (int i = 0; i < WMT; ++i) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = m0 + wm * 16 * WMT + i * 16 + (lane >> 4) * 4 + r;
      if (m >= M) continue;
#pragma unroll
      for (int j = 0; j < WNT; ++j) {
        const int nt = n0 + wn * 16 * WNT + j * 16;   // first column of this 16-wide tile
        const int n = nt + (lane & 15);
        if (gridDim.z > 1) {
          if (n < N) partial[((size_t)blockIdx.z * M + m) * N + n] = acc[i][j][r];
        } else if (mode == OUT_SWIGLU) {
          const float u = __shfl_xor(acc[i][j][r], 8, 64);   // the up row sits eight columns to the right
          if ((lane & 8) == 0 && n + 8 < N)
            ((bf16_t*)out)[(size_t)m * (N / 2) + nt / 2 + (lane & 7)] = float_to_bf16(gate_mul(acc[i][j][r], u, ga));
        } else if (n < N) {
          store_out(out, mode, (size_t)m * N + n, acc[i][j][r]);
        }
      }
    }
  }
}

// Adds the K splits of `partial` [splits, M, N] in ascending order and applies the epilogue.
__global__ void gemm_splitk_reduce_kernel(const float* __restrict__ partial, void* __restrict__ out, int mode,
                                          int splits, int M, int N, GateAct ga) {
  const size_t total = (size_t)M * N;
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (mode == OUT_SWIGLU) {
    // one thread per output element: column 8 b + i pairs rows 16 b + i and 16 b + 8 + i
    const int half = N / 2;
    if (idx >= (size_t)M * half) return;
    const int m = (int)(idx / half), c = (int)(idx % half);
    const int ng = (c / 8) * 16 + (c % 8);
    float g = 0.f, u = 0.f;
    for (int s = 0; s < splits; ++s) {
      g += partial[(size_t)s * total + (size_t)m * N + ng];
      u += partial[(size_t)s * total + (size_t)m * N + ng + 8];
    }
    ((bf16_t*)out)[idx] = float_to_bf16(gate_mul(g, u, ga));
    return;
  }
  if (idx >= total) return;
  float v = 0.f;
  for (int s = 0; s < splits; ++s) v += partial[(size_t)s * total + idx];
  if (mode == OUT_SPLIT) {
    store_split(out, 0, ga, M, (int)(idx / N), (int)(idx % N), v);
    return;
  }
  store_out(out, mode, idx, v);
}

// Adds the K splits of `partial` [splits, M, N] (ascending) into the float32 residual rows h [M, N] and
// writes the root-mean-square norm of the updated rows: out = h / sqrt(mean(h^2) + eps) * w.  One block
// per row; takes the place of the reduction kernel and the norm kernel that would follow it.
// Each thread owns four neighbouring columns (N % 4 == 0); all its loads are issued before the first sum.
// SP: the most splits (2, 4 or 16); T: threads; NV: groups of four columns a thread (N <= 4 T NV).
template <typename TO, int SP, int T, int NV>
__global__ __launch_bounds__(T) void splitk_add_rmsnorm_kernel(const float* __restrict__ partial, int splits,
                                                                   float* __restrict__ h, const float* __restrict__ w,
                                                                   float eps, TO* __restrict__ out, int M, int N) {
  __shared__ __attribute__((aligned(16))) float red[T / TP_WAVE];
  const int m = blockIdx.x;
  const size_t total = (size_t)M * N;
  float* hr = h + (size_t)m * N;
  f32x4_t acc[NV], wv[NV];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int n = (threadIdx.x + i * T) * 4;
    if (n < N) {
      const float* pr = partial + (size_t)m * N + n;
      f32x4_t p[SP];
      p[0] = *(const f32x4_t*)pr;
#pragma unroll
      for (int s = 1; s < SP; ++s)
        if (s < splits) p[s] = *(const f32x4_t*)(pr + (size_t)s * total);
      const f32x4_t base = *(const f32x4_t*)(hr + n);
      wv[i] = *(const f32x4_t*)(w + n);
      f32x4_t add = (f32x4_t){0.f, 0.f, 0.f, 0.f};
      add += p[0];
#pragma unroll
      for (int s = 1; s < SP; ++s)
        if (s < splits) add += p[s];
      acc[i] = base + add;
      *(f32x4_t*)(hr + n) = acc[i];
      ss += acc[i][0] * acc[i][0] + acc[i][1] * acc[i][1] + acc[i][2] * acc[i][2] + acc[i][3] * acc[i][3];
    }
  }
  ss = block_sum_once<T>(ss, red);
  const float scale = rsqrtf(ss / (float)N + eps);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int n = (threadIdx.x + i * T) * 4;
    if (n < N)
      from_float4(out + (size_t)m * N + n, acc[i][0] * scale * wv[i][0], acc[i][1] * scale * wv[i][1], acc[i][2] * scale * wv[i][2],
                  acc[i][3] * scale * wv[i][3]);
  }
}

template <typename TO>
static void launch_splitk_add_rmsnorm(const float* partial, int splits, float* h, const float* w, float eps, void* out, int M, int N, hipStream_t s) {
#define SKN(SP_, T_, NV_) hipLaunchKernelGGL((splitk_add_rmsnorm_kernel<TO, SP_, T_, NV_>), dim3(M), dim3(T_), 0, s, partial, splits, h, w, eps, (TO*)out, M, N)
  if (N > 8192) SKN(16, 1024, 4);
  else if (N > 4096) SKN(16, 1024, 2);
  else if (N > 2048 && splits <= 2) SKN(2, 1024, 1);
  else if (N > 2048 && splits <= 4) SKN(4, 1024, 1);
  else if (N > 2048) SKN(16, 1024, 1);
  else if (splits <= 4) SKN(4, 512, 1);
  else SKN(16, 512, 1);
#undef SKN
}

extern "C" int tp_splitk_add_rmsnorm(const float* partial, int splits, float* h, const float* w, float eps, void* out,
                                     int out_dt, int M, int N, hipStream_t s) {
  TP_REQUIRE(M > 0 && N > 0 && splits >= 1 && splits <= 16, "splitk_add_rmsnorm: bad sizes");
  TP_REQUIRE(N % 4 == 0 && N <= 16384, "splitk_add_rmsnorm: width %d must be a multiple of 4, at most 16384", N);
  TP_REQUIRE(out_dt == TP_F32 || out_dt == TP_BF16, "splitk_add_rmsnorm: unknown dtype %d", out_dt);
  if (out_dt == TP_BF16)
    launch_splitk_add_rmsnorm<bf16_t>(partial, splits, h, w, eps, out, M, N, s);
  else
    launch_splitk_add_rmsnorm<float>(partial, splits, h, w, eps, out, M, N, s);
  TP_CHECK_LAUNCH("splitk_add_rmsnorm");
  return 0;
}

// In the few and skinny kernels x is the second operand, so the result lane holds weight rows
// (l / 16) * 4 + r and activation row l % 16; see the index arithmetic there.

static int g_tune_splits = 0, g_tune_mid = 0;                    // mid = 1: 17..64 rows stay on the skinny kernel
static int g_tune_order = 0;   // large products: 1 tiled kernel, plain block order; 2 tiled, XCD patches; 3 pipelined kernel

// Defined in gemm_pipe.hip; 0 when it took the product, -1 when the sizes are not its own.
int tp_linear_pipe(const bf16_t* x, const bf16_t* w, int w_tiled, void* out, int mode, int M, int N, int K, float* scratch,
                   size_t scratch_floats, int tune_splits, const RopeOut* rope, int defer, int* splits_out, GateAct gate,
                   hipStream_t s);

int tp_linear_pipe64(const bf16_t* x, const bf16_t* w, int w_tiled, void* out, int mode, int M, int N, int K, float* scratch,
                     size_t scratch_floats, int tune_splits, int defer, int* splits_out, GateAct gate, hipStream_t s);

extern int g_pipe_big;
// order: 1 tiled plain, 2 tiled XCD-aware, 3 pipelined; 5 / 6: pipelined with 256 x 256 tiles always / never;
// 7 / 8: with 256 x 192 tiles wherever N is a multiple of 192 / never; 9: with 192 x 256 tiles wherever N is a multiple of 256
extern "C" void tp_linear_tune_tile(int order) {
  g_pipe_big = order == 5 ? 1 : (order == 6 ? 2 : (order == 7 ? 3 : (order == 8 ? 4 : (order == 9 ? 5 : 0))));
  g_tune_order = order >= 5 ? 0 : order;
}

extern int g_pipe_mid;
// the pipelined product's 128 x 128 blocks: 0 chosen by shape, 1 for every product of more than 128 rows, 2 never
extern "C" void tp_linear_tune_mid_tile(int v) { g_pipe_mid = v; }

extern int g_pipe64_narrow;
// the 64-row pipeline's blocks: 0 chosen by shape, 1 always 64 columns wide, 2 always 128
extern "C" void tp_linear_tune_narrow(int v) { g_pipe64_narrow = v; }

extern "C" void tp_linear_tune_mid(int mid, int splits) {
  g_tune_mid = mid;
  g_tune_splits = splits;
}

static bool gate_has_constants(const GateAct& g) { return g.extra_slope != 0.f || g.limit > 0.f || g.offset != 0.f; }
// whether a product of a few rows takes the kernels of the split epilogue (see SPLIT)
static bool split_epilogue(int mode, const GateAct& g) { return mode == OUT_SPLIT || (mode == OUT_SWIGLU && gate_has_constants(g)); }

// whether a kernel's parameters are the members of FewArgs (whose offsets few_end() goes by)
template <typename... T>
constexpr bool few_args_are(void (*)(T...)) {
  FewArgs* a = nullptr;
  return std::is_same_v<std::tuple<T...>, std::tuple<decltype(a->x), decltype(a->w), decltype(a->out), decltype(a->M), decltype(a->N), decltype(a->K),
                                                     decltype(a->mode), decltype(a->layout), decltype(a->end)>>;
}

template <int P, int KIND, bool PRE, bool WT, bool DEEP = false>
static void launch_few3(const bf16_t* x, const bf16_t* w, void* out, int mode, int M, int N, int K, int layout, const RowScale& pre, const NormPrep& post,
                        const RopeOut& rp, hipStream_t s) {
  static_assert(few_args_are(&gemm_few_kernel<P, KIND, PRE, WT, DEEP>), "few_end() reads another structure than the kernel is given");
  // (DEEP: two blocks a CU, by their LDS; with more of them, 32,000 columns of one row, K 4,096 41.9 -> 42.1 us, K 8,192 78.6 -> 78.8)
  const size_t rows = P < 0 ? 2 * 16 * FEW_CHUNK_LD : P > 0 ? std::max((size_t)M * (K * 2 + 16), (size_t)(DEEP ? 56 << 10 : 0)) : 0;
  hipLaunchKernelGGL((gemm_few_kernel<P, KIND, PRE, WT, DEEP>), dim3((N + 15) / 16), dim3(FEW_WAVES * 64), rows, s, x, w, out, M, N, K, mode, layout, FewEnd{pre, post, rp});
}

template <int KIND, bool PRE>
static void launch_few2(const bf16_t* x, const bf16_t* w, void* out, int mode, int M, int N, int K, int layout, const RowScale& pre, const NormPrep& post,
                        const RopeOut& rp, hipStream_t s) {
#define FEW(P_, WT_) return launch_few3<P_, KIND, PRE, WT_>(x, w, out, mode, M, N, K, layout, pre, post, rp, s)
#define FEW_DEEP(P_) return launch_few3<P_, KIND, PRE, true, true>(x, w, out, mode, M, N, K, layout, pre, post, rp, s)
  const bool tiled = (layout & W_TILED) != 0, major = M > 1 && (layout & X_KBLOCKED) == 0;
  const int blocks = (N + 15) / 16, pieces = (M * (K / 8) + FEW_WAVES * 64 - 1) / (FEW_WAVES * 64);
  // Row-major rows of products with more column blocks than CUs go through LDS in chunks: read from memory as operands, 64-byte pieces of up to sixteen rows,
  // their way into the CU is as long as the weights' where blocks follow or share a CU.  From memory (to 32 KB through LDS) / in chunks, tiled weight, us; first
  // float32 results, then the sums added into the stream with the next norm prepared.  Sixteen rows: K 2,048, 272 blocks 7.5 / 7.4 and 8.1 / 7.7, 512 8.5 / 8.6 and
  // 9.5 / 9.2, 1,792 25.5 / 23.5; K 4,096, 272 13.6 / 12.8 and 13.7 / 12.9, 512 15.9 / 15.4 and 16.5 / 15.8, 896 27.5 / 25.3 and 28.6 / 25.9; K 8,192, 272 24.4 / 22.9
  // and 25.0 / 23.2, 512 27.9 / 26.9 and 29.0 / 27.1, 896 50.2 / 45.4 and 51.8 / 46.2, 1,792 88.0 / 81.2; but with a CU a block the latter K 2,048 6.0 / 6.1, K 4,096
  // 8.9 / 9.5, K 8,192 16.0 / 17.0.  Fourteen: K 2,048, 512 8.3 / 8.6 and 9.0 / 8.9; K 4,096, 384 13.8 / 14.1 and 14.6 / 14.6, 1,792 44.2 / 43.4 and 46.8 / 45.5; K 6,144,
  // 384 19.9 / 19.6 and 20.5 / 20.0, 768 30.0 / 30.8 and 30.9 / 31.2; K 8,192, 272 23.0 / 22.3 and 23.7 / 22.9, 512 26.4 / 26.4 and 27.2 / 26.7, 896 47.8 / 45.2 and 48.8 / 46.0.  Thirteen: K 8,192, 768 36.8 / 38.5 and 37.8 / 39.0, 896
  // 46.4 / 44.9 and 47.4 / 45.6, 1,792 80.5 / 81.5 and 84.4 / 83.8; K 5,120, 1,728 53.6 / 50.8 and 55.4 / 52.2; K 6,144, 1,792 62.9 / 63.6 and 65.3 / 65.8.  Twelve: K 3,072, 512
  // the latter 12.0 / 11.8, 1,792 32.7 / 32.3 and 34.6 / 33.2; K 2,048, 4,000 52.9 / 52.1; K 4,096, 1,280 32.3 / 33.0, 1,792 42.2 / 43.1; K 6,144, 1,792 61.9 / 62.7 and
  // 63.2 / 64.3; K 8,192, 896 45.5 / 43.9 and 46.4 / 45.0, 1,792 79.2 / 81.0.  Float32 results of 128,256 columns: K 3,072, two rows 117.0 / 115.4, eight 124.0 / 120.8,
  // sixteen 156.4 / 138.7; K 4,096, ten 171.3 / 177.3, twelve 183.9 / 180.4, sixteen 201.9 / 183.1.  A row-major weight takes that
  // way twice over: 4,096 x 128,256 eight rows 227 / 206, sixteen 270 / 230; 4,096 x 6,144 16.1 / 15.5 and 18.6 / 17.0; 2,048 x 8,192 9.6 / 9.5 and 10.9 / 10.5;
  // 8,192 x 4,096 six rows 18.2 / 19.2, eight 19.3 / 19.4, sixteen 21.4 / 20.7.  (Chunks are of use from two on, and to 8,192: 14,336 x 4,096 eight rows
  // 21.6 / 26.0.)
  if (major && K >= 2 * FEW_CHUNK && K <= 8 * FEW_CHUNK) {
    const bool short_k = K <= 3 * FEW_CHUNK;
    const int from = blocks <= 256 ? 17 : blocks < 896 ? (blocks <= 512 && K > 4 * FEW_CHUNK ? 14 : 15) : blocks < 4096 ? (short_k ? 12 : 13) : short_k ? 2 : 12;      // rows
    if (tiled && M >= from) FEW(-1, true);
    if (!tiled && (K <= 4 * FEW_CHUNK || M >= 8)) FEW(-1, false);
  }
  if (!tiled) FEW(0, false);
  // Row-major rows of several requests go through LDS whole while they are few enough (up to 32 KB: four rows 4,096 x 4,096 7.6 us, straight from memory
  // 8.3), and so does a single row of more blocks than there are CUs, up to 64 KB: blocks that follow or share a CU are bound by what it can pull, and the
  // row's own loads, four as wide as the weights' a run, are in their way; with up to one block a CU the wait for the copy is what counts.  From memory / through
  // LDS: K 4,096, 256 blocks 7.4 / 7.6 us, 257 9.7 / 8.6, 384 11.8 / 10.4, 512 13.0 / 12.5; K 2,048 4.7 / 5.0, 5.6 / 5.1, 6.6 / 6.1 and 7.5 / 7.1; K 8,192
  // 12.6 / 12.9, 17.8 / 16.0, 21.6 / 18.9 and 24.0 / 23.0.
  if (M > 1 ? !major || pieces > 4 : blocks <= 256 || pieces > 8) FEW(0, true);
  // From three blocks a CU on, or with more than 32 KB, a row of more than 4,096 also has two runs on their way and no more than two blocks a CU (56 KB of LDS).
  // One run from memory / two through LDS: K 8,192, 768 blocks 33.8 / 33.0 us, 1,792 72.5 / 71.1, 8,016 300.8 / 302.9; K 14,336, 576 48.6 / 45.7, 1,792
  // 123.9 / 120.7, 4,000 270.7 / 263.9; K 28,672, 512 75.9 / 72.1; six layers of the 70B shape, one row, 1,983 / 1,963.  Shorter rows gain alone what they lose
  // behind other kernels, where the wait for the copy counts: K 4,096, 576 blocks 15.4 / 14.6 and 1,024 22.7 / 22.5, but four layers with products of
  // 1,100 to 1,800 blocks 16,330 / 16,490 us for 24 steps; K 2,048, 1,280 blocks 14.7 / 15.3; K 3,072, 384 blocks, one and two through LDS 8.0 / 8.3.
  if (M == 1 && (blocks > 512 || pieces > 4)) {
    if (K <= 4 * FEW_CHUNK || (K <= 8 * FEW_CHUNK && blocks > 2048)) FEW(0, true);
    if (pieces <= 2) FEW_DEEP(2);
    if (pieces <= 4) FEW_DEEP(4);
    FEW_DEEP(8);
  }
  if (pieces <= 1) FEW(1, true);
  if (pieces <= 2) FEW(2, true);
  FEW(4, true);
#undef FEW
#undef FEW_DEEP
}

template <int KIND>
static void launch_few1(const bf16_t* x, const bf16_t* w, void* out, int mode, int M, int N, int K, int layout, const RowScale& pre, const NormPrep& post,
                        const RopeOut& rp, hipStream_t s) {
  if (pre.ss != nullptr) launch_few2<KIND, true>(x, w, out, mode, M, N, K, layout, pre, post, rp, s);
  else launch_few2<KIND, false>(x, w, out, mode, M, N, K, layout, pre, post, rp, s);
}

// at most 16 rows
static void launch_few(const bf16_t* x, const bf16_t* w, void* out, int mode, int M, int N, int K, int layout, const RowScale& pre, const NormPrep& post,
                       const RopeOut& rp, hipStream_t s) {
#define FEW(KIND_) return launch_few1<KIND_>(x, w, out, mode, M, N, K, layout, pre, post, rp, s)
  if (split_epilogue(mode, rp.gate)) FEW(FEW_SPLIT);
  if (mode == OUT_SWIGLU) FEW(FEW_SWIGLU);
  if (mode == OUT_ROPE) FEW(FEW_ROPE);
  if (post.w != nullptr) FEW(FEW_POST);
  FEW(FEW_STORE);
#undef FEW
}

template <int MT>
static void launch_skinny(const bf16_t* x, const bf16_t* w, void* out, int mode, int M, int N, int K, int w_tiled, const GateAct& gate, hipStream_t s) {
  // every wave should get at least one run of four steps
  const int runs = K / 128;
  const int waves = runs >= 8 ? 8 : (runs >= 4 ? 4 : 2);
  const int depth = runs >= 2 * waves && MT <= 2 ? 2 : 1;           // (more tiles: registers)
  const bool split = split_epilogue(mode, gate);
#define SKINNY(W_, D_, WT_, SPLIT_) \
  hipLaunchKernelGGL((gemm_skinny_mfma_kernel<MT, W_, D_, WT_, SPLIT_>), dim3((N + 15) / 16), dim3(W_ * 64), 0, s, x, w, out, mode, M, N, K, gate)
#define CASE(W_, D_)                                                  \
  if (waves == W_ && depth == D_) {                                   \
    if (split && w_tiled) SKINNY(W_, D_, true, true);                 \
    else if (split) SKINNY(W_, D_, false, true);                      \
    else if (w_tiled) SKINNY(W_, D_, true, false);                    \
    else SKINNY(W_, D_, false, false);                                \
    return;                                                           \
  }
  CASE(8, 1)
  CASE(4, 1)
  CASE(2, 1)
  if constexpr (MT <= 2) {
    CASE(8, 2)
    CASE(4, 2)
  }
#undef CASE
#undef SKINNY
}

// The q/k/v projection of at most 16 rows with rotation and cache write in its epilogue (see RopeOut).
// N = (n_heads + 2 n_kv) * head_dim.  Returns -1 for sizes this path does not take.
int tp_linear_rope_mfma(const void* x, const void* w, int w_tiled, int M, int N, int K, const float* pre_ss, int pre_count,
                        float pre_eps, const int* positions, const int* slots, const double* inv_freq, int rotary_dim,
                        float factor, int n_heads, int n_kv, int head_dim, void* q_out, void* k_cache, void* v_cache,
                        int page_size, const float* cos_sin, hipStream_t s) {
  if (M < 1 || (M > 16 && M <= 128) || K % 32 != 0 || head_dim % 16 != 0 || rotary_dim % 2 != 0 || rotary_dim > head_dim) return -1;
  if (N != (n_heads + 2 * n_kv) * head_dim || page_size < 1) return -1;
  if (((uintptr_t)x & 15) || ((uintptr_t)w & 15)) return -1;
  // w_tiled: bit 0, the weight is tiled; bit 1 (at most 16 rows), x is k-blocked [K / 8, M, 8]
  if ((w_tiled & 1) && (N % 16 != 0 || K % 64 != 0)) return -1;
  if ((w_tiled & 2) && M > 16) return -1;
  const RowScale pre = {pre_ss, pre_count, 1.0f / (float)K, pre_eps};
  const NormPrep post = {nullptr, nullptr, nullptr};
  const RopeOut rp = {positions, slots, inv_freq, (const float2*)cos_sin, factor, rotary_dim, n_heads, n_kv, head_dim, page_size,
                      0, (bf16_t*)q_out, (bf16_t*)k_cache, (bf16_t*)v_cache};
  if (M > 16) {
    // long steps: the pipelined kernels, whose wave tiles of 64 columns must each lie inside q, k or v (heads of a
    // multiple of 64; the wider tiles are left out unless the heads are multiples of 128), with the step's table
    // of cosines and sines
    if (head_dim % 64 != 0 || rotary_dim % 8 != 0 || cos_sin == nullptr || pre_ss != nullptr || page_size % 8 != 0) return -1;
    return tp_linear_pipe((const bf16_t*)x, (const bf16_t*)w, w_tiled & 1, nullptr, OUT_ROPE, M, N, K, nullptr, 0, 0, &rp, 0, nullptr, GateAct{}, s);
  }
  launch_few((const bf16_t*)x, (const bf16_t*)w, nullptr, OUT_ROPE, M, N, K, (w_tiled & 1 ? W_TILED : 0) | (w_tiled & 2 ? X_KBLOCKED : 0), pre, post, rp,
             s);
  return 0;
}

// accumulate: 0 store, 1 add into the float32 output, 2 gated-SiLU epilogue (see OUT_SWIGLU), 3 the squared-ReLU epilogue
// with side columns (see OUT_SPLIT; gate.act_cols, act_ld, side and side_ld are set).
// pre_ss / post_w: the split norm (RowScale / NormPrep above), at most 16 rows; nullptr without.
int tp_linear_mfma(const void* x, const void* w, void* out, int out_dt, int accumulate, int M, int N, int K,
                   float* scratch, size_t scratch_floats, const float* pre_ss, int pre_count, float pre_eps,
                   const void* post_w, void* post_xg, float* post_ss, int layout, int defer_reduce, int* splits_out,
                   GateAct gate, hipStream_t s) {
  if (splits_out) *splits_out = 1;
  if (K % 32 != 0) return -1;
  const int w_tiled = (layout & W_TILED) != 0;
  if (w_tiled && (N % 16 != 0 || K % 64 != 0)) return -1;
  if ((layout & (X_KBLOCKED | OUT_KBLOCKED | XG_KBLOCKED)) != 0 && M > 16) return -1;
  if ((layout & XG_KBLOCKED) && (post_w == nullptr || N % 8 != 0)) return -1;
  if ((layout & OUT_KBLOCKED) && accumulate != 2 && accumulate != 3) return -1;
  if (accumulate == 3 && (K % 64 != 0 || gate.act_cols % 128 != 0 || gate.act_cols <= 0 || gate.act_cols > N || out_dt != TP_BF16)) return -1;
  if ((pre_ss != nullptr || post_w != nullptr) && M > 16) return -1;
  if (post_w != nullptr && accumulate != 1) return -1;
  const RowScale pre = {pre_ss, pre_count, 1.0f / (float)K, pre_eps};
  const NormPrep post = {(const float*)post_w, (bf16_t*)post_xg, post_ss};
  if (((uintptr_t)x & 15) || ((uintptr_t)w & 15)) return -1;
  if (accumulate == 2 && (N % 16 != 0 || out_dt != TP_BF16)) return -1;
  const int mode = accumulate == 3 ? OUT_SPLIT : accumulate == 2 ? OUT_SWIGLU : (accumulate ? OUT_ACC_F32 : (out_dt == TP_F32 ? OUT_F32 : OUT_BF16));
  const bf16_t* xb = (const bf16_t*)x;
  const bf16_t* wb = (const bf16_t*)w;
  const bool mid_ok = scratch != nullptr && g_tune_mid != 1;
  RopeOut no_rope = {};
  no_rope.gate = gate;      // (the kernels read the gated epilogue's constants from here)
  if (M <= 16 || (M <= 64 && !mid_ok)) {
    if (M <= 16)
      launch_few(xb, wb, out, mode, M, N, K, layout, pre, post, no_rope, s);
    else if (M <= 32)
      launch_skinny<2>(xb, wb, out, mode, M, N, K, w_tiled, gate, s);
    else if (M <= 48)
      launch_skinny<3>(xb, wb, out, mode, M, N, K, w_tiled, gate, s);
    else
      launch_skinny<4>(xb, wb, out, mode, M, N, K, w_tiled, gate, s);
  } else {
    // large products: 128 x 128 tiles.  Between 17 and 128 rows the weights are still the traffic:
    // 64 x 128 tiles, and K split over blockIdx.z until there are blocks for every CU.
    // the pipelined kernels: from 65 rows on (their 128 x 128 blocks against two 64-row blocks that each fetch
    // the weights: 72 to 128 rows of the 8B shapes 26 -> 17..21 us, 43 -> 31..34 us, 21 -> 16 us, 52 -> 46 us)
    const bool pipe = g_tune_order ? g_tune_order == 3 : M > 64;
    const bool pipe64 = !pipe && M <= 128 && scratch != nullptr && g_tune_mid != 2;
    if (pipe && tp_linear_pipe(xb, wb, w_tiled, out, mode, M, N, K, scratch, scratch_floats, g_tune_splits, nullptr, defer_reduce,
                               splits_out, gate, s) == 0) {
      // taken by the pipelined kernel
    } else if (pipe64 && tp_linear_pipe64(xb, wb, w_tiled, out, mode, M, N, K, scratch, scratch_floats, g_tune_splits,
                                          defer_reduce, splits_out, gate, s) == 0) {
      // taken by the 64-row pipelined kernel
    } else if (w_tiled || mode == OUT_SPLIT) {
      return -1;   // the kernels below read row-major weights only, and have no columns that go elsewhere
    } else if (M > 128 || scratch == nullptr) {
      dim3 grid((N + 127) / 128, (M + 127) / 128);
      if (grid.y > 65535) return -1;
      const int xcd_order = g_tune_order != 1;
      if (xcd_order) {  // one-dimensional grid: 8 XCDs x patches of 64 blocks
        const int Q = ((int)grid.x + 7) / 8, MS = ((int)grid.y + 7) / 8, QS = (Q + 7) / 8;
        grid = dim3(8 * QS * MS * 64, 1);
      }
      if (K % 64 == 0)
        hipLaunchKernelGGL((gemm_tiled_mfma_kernel<64, 4, 4>), grid, dim3(256), 0, s, xb, wb, out, nullptr, mode, M, N, K,
                           xcd_order, gate);
      else
        hipLaunchKernelGGL((gemm_tiled_mfma_kernel<32, 4, 4>), grid, dim3(256), 0, s, xb, wb, out, nullptr, mode, M, N, K,
                           xcd_order, gate);
    } else {
      const int nb = (N + 127) / 128, mb = (M + 63) / 64;
      int splits = g_tune_splits ? g_tune_splits : (512 + nb * mb - 1) / (nb * mb);
      const int kt = K / (K % 64 == 0 ? 64 : 32);
      splits = max(1, min(splits, min(16, kt / 4)));
      while (splits > 1 && (size_t)splits * M * N > scratch_floats) --splits;
      const dim3 grid(nb, mb, splits);
      if (K % 64 == 0)
        hipLaunchKernelGGL((gemm_tiled_mfma_kernel<64, 2, 4>), grid, dim3(256), 0, s, xb, wb, out, scratch, mode, M, N, K, 0, gate);
      else
        hipLaunchKernelGGL((gemm_tiled_mfma_kernel<32, 2, 4>), grid, dim3(256), 0, s, xb, wb, out, scratch, mode, M, N, K, 0, gate);
      if (splits > 1 && defer_reduce && splits_out != nullptr && mode != OUT_SWIGLU) {
        *splits_out = splits;   // the caller's next kernel adds the partial sums [splits, M, N] in `scratch`
      } else if (splits > 1) {
        const size_t n_out = mode == OUT_SWIGLU ? (size_t)M * (N / 2) : (size_t)M * N;
        hipLaunchKernelGGL(gemm_splitk_reduce_kernel, dim3((unsigned)((n_out + 255) / 256)), dim3(256), 0, s, scratch, out,
                           mode, splits, M, N, gate);
      }
    }
  }
  TP_CHECK_LAUNCH("linear (mfma)");
  return 0;
}
