// Sums over the lanes of a wave: over neighbouring lanes by row permutes, for recurrences whose lanes share a state column, and of many
// values over all lanes at once.
#pragma once
#include "common.h"

// sum over KS neighbouring lanes (from a multiple of KS on); every lane gets it
template <int KS>
__device__ inline float column_sum(float v) {
#define DPP_ADD(ctrl) v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, 0xf, 0xf, false))
  if (KS >= 2) DPP_ADD(0xB1);    // quad_perm [1, 0, 3, 2]
  if (KS >= 4) DPP_ADD(0x4E);    // quad_perm [2, 3, 0, 1]
  if (KS >= 8) DPP_ADD(0x141);   // row_half_mirror
  if (KS >= 16) DPP_ADD(0x140);  // row_mirror
#undef DPP_ADD
  if (KS >= 32) v += __shfl_xor(v, 16, TP_WAVE);
  return v;
}

// Adds v[i] over the lanes of a wave for NV values at once: each step halves the values a lane still carries, NV - 1 exchanges
// (and single ones below NV lanes) instead of 6 NV.  The pairs added are those of an ordinary exchange tree from distance 32
// down, so a sum's bits do not depend on NV.  The lanes with equal lane / (64 / NV) then hold the sum of value lane / (64 / NV).
template <int N, int W>
__device__ inline void lanes_transpose_step(float* v, int lane) {
  if constexpr (N > 1) {
    const bool hi = lane & W;
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
      const float keep = hi ? v[i + N / 2] : v[i], send = hi ? v[i] : v[i + N / 2];
      v[i] = keep + __shfl_xor(send, W, TP_WAVE);
    }
  } else {
    v[0] += __shfl_xor(v[0], W, TP_WAVE);
  }
  if constexpr (W > 1) lanes_transpose_step<(N > 1 ? N / 2 : 1), W / 2>(v, lane);
}
template <int NV>
__device__ inline float lanes_transpose_sum(float (&v)[NV], int lane) {
  lanes_transpose_step<NV, TP_WAVE / 2>(v, lane);
  return v[0];
}
