// The router of a mixture of experts: one token's choice by one wave.
#pragma once
#include <math.h>

#include "common.h"

// logits [n, logit_stride] float32 (the first `experts` columns count).  s = softmax over the experts; the choice
// score of expert e is s[e] + correction[e]; experts form `groups` equal groups of neighbours, a group's score is
// its largest choice score, and only experts of the `keep` best groups can be chosen (groups <= 1: all); the `top`
// allowed experts with the largest choice scores are chosen (ties: the lower index), and a chosen expert's weight
// is s[e].  dense [n, experts] gets the weight of every chosen expert and 0 elsewhere; ids and weights [n, top]
// list the chosen experts in the order of choice.  One wave per token; lane l holds experts l, l + 64, ...
// (lane l holds experts l, l + 64, ...)
#define ROUTE_PER_LANE 8   // experts <= 64 * ROUTE_PER_LANE

__device__ inline void wave_arg_best(float& v, int& i) {
#pragma unroll
  for (int o = TP_WAVE / 2; o > 0; o >>= 1) {
    const float ov = __shfl_xor(v, o, TP_WAVE);
    const int oi = __shfl_xor(i, o, TP_WAVE);
    if (ov > v || (ov == v && oi < i)) {
      v = ov;
      i = oi;
    }
  }
}

// score_kind 0: s = softmax over the experts; 1: s = sigmoid of each logit by itself.  The choice score is s plus the
// correction (none: s).  A group is ranked by the sum of its `group_best` largest choice scores.  The weights are the
// chosen experts' s, with `normalize` divided by their sum plus sum_eps (added in the order of choice), times `scale`.
struct Route {
  const float *correction, *bias;   // [experts] or nullptr
  int experts, top, groups, keep, score_kind, group_best, normalize;
  float sum_eps, scale;
  float* dense;
  int* ids;
  float* weights;
};

// logits: the token's row (global memory or LDS); t: its row in the outputs; live false: nothing is stored; choice_l [experts] and
// group_l [groups] are the wave's own LDS.  Every wave of the block calls it the same number of times (it holds barriers).
template <int ROUTE_LANE>
__device__ inline void route_token(const Route& r, const float* logits, int t, bool live, float* choice_l, float* group_l) {
  const int lane = threadIdx.x % TP_WAVE;
  const int experts = r.experts, groups = r.groups;
  const float *correction = r.correction, *logit_bias = r.bias;
  float* dense = r.dense;
  float z[ROUTE_LANE], sc[ROUTE_LANE], ch[ROUTE_LANE];
  int won[ROUTE_LANE];
  float mx = -INFINITY;
#pragma unroll
  for (int k = 0; k < ROUTE_LANE; ++k) {
    const int e = lane + k * TP_WAVE;
    z[k] = e < experts ? logits[e] + (logit_bias != nullptr ? logit_bias[e] : 0.f) : -INFINITY;
    mx = fmaxf(mx, z[k]);
    won[k] = -1;
  }
  if (r.score_kind == 1) {
#pragma unroll
    for (int k = 0; k < ROUTE_LANE; ++k) sc[k] = lane + k * TP_WAVE < experts ? 1.0f / (1.0f + expf(-z[k])) : 0.f;
  } else {
    mx = wave_max(mx);
    float sum = 0.f;
#pragma unroll
    for (int k = 0; k < ROUTE_LANE; ++k) {
      sc[k] = lane + k * TP_WAVE < experts ? expf(z[k] - mx) : 0.f;
      sum += sc[k];
    }
    sum = wave_sum(sum);
    const float inv = 1.0f / sum;
#pragma unroll
    for (int k = 0; k < ROUTE_LANE; ++k) sc[k] *= inv;
  }
#pragma unroll
  for (int k = 0; k < ROUTE_LANE; ++k) {
    const int e = lane + k * TP_WAVE;
    ch[k] = e < experts ? (correction != nullptr ? sc[k] + correction[e] : sc[k]) : -INFINITY;
    if (e < experts) {
      choice_l[e] = ch[k];
      if (live) dense[(size_t)t * r.experts + e] = 0.f;
    }
  }
  if (groups > 1) {
    const int per = experts / groups;
    __syncthreads();
    for (int g = lane; g < groups; g += TP_WAVE) {
      // the group's largest scores one after the other (equal scores: the lower index first), added in that order
      float total = 0.f, pv = INFINITY;
      int pi = -1;
      for (int b = 0; b < r.group_best; ++b) {
        float best = -INFINITY;
        int bi = -1;
        for (int i = 0; i < per; ++i) {
          const float v = choice_l[g * per + i];
          if ((v < pv || (v == pv && i > pi)) && (bi < 0 || v > best)) {
            best = v;
            bi = i;
          }
        }
        if (bi < 0) break;
        total = b == 0 ? best : total + best;
        pv = best;
        pi = bi;
      }
      group_l[g] = total;
    }
    __syncthreads();
    // the `keep` best groups, one after the other; a kept group's score becomes +inf as its mark
    for (int it = 0; it < r.keep; ++it) {
      float bv = -INFINITY;
      int bi = 0x7fffffff;
      for (int g = lane; g < groups; g += TP_WAVE) {
        const float v = group_l[g];
        if (v != INFINITY && (v > bv || (v == bv && g < bi))) {
          bv = v;
          bi = g;
        }
      }
      wave_arg_best(bv, bi);
      __syncthreads();
      if (lane == 0 && bi != 0x7fffffff) group_l[bi] = INFINITY;
      __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < ROUTE_LANE; ++k) {
      const int e = lane + k * TP_WAVE;
      if (e < experts && group_l[e / per] != INFINITY) ch[k] = -INFINITY;
    }
  }
  float chosen_sum = 0.f;
  for (int it = 0; it < r.top; ++it) {
    float bv = -INFINITY, bs = 0.f;
    int bi = 0x7fffffff, bk = -1;
#pragma unroll
    for (int k = 0; k < ROUTE_LANE; ++k) {
      const int e = lane + k * TP_WAVE;
      if (e < experts && ch[k] > bv) {   // (ascending e within a lane: the lower index wins a tie)
        bv = ch[k];
        bi = e;
        bk = k;
        bs = sc[k];
      }
    }
    float v = bv;
    int i = bi;
    wave_arg_best(v, i);
    if (i == 0x7fffffff) break;   // fewer allowed experts than `top` (uniform over the wave)
    chosen_sum += __shfl(bs, i % TP_WAVE, TP_WAVE);   // (the winner's lane holds its score; every lane adds alike)
    if (i == bi && bk >= 0) {
      // this lane owns the winner
#pragma unroll
      for (int k = 0; k < ROUTE_LANE; ++k)
        if (k == bk) {
          ch[k] = -INFINITY;
          won[k] = it;
        }
    }
  }
  const float factor = r.normalize ? r.scale / (chosen_sum + r.sum_eps) : r.scale;
#pragma unroll
  for (int k = 0; k < ROUTE_LANE; ++k) {
    if (won[k] >= 0 && live) {
      const int e = lane + k * TP_WAVE;
      const float w = (r.normalize || r.scale != 1.0f) ? sc[k] * factor : sc[k];
      dense[(size_t)t * r.experts + e] = w;
      r.ids[(size_t)t * r.top + won[k]] = e;
      r.weights[(size_t)t * r.top + won[k]] = w;
    }
  }
}

// The same choice of up to 16 experts, bit for bit: lane l of a row of 16 lanes holds expert l, a wave works on four tokens.  The scores of a
// token are gathered once (sixteen loads from other lanes in flight together) and every lane counts the scores in front of its own; the
// choice one by one is a chain of reductions through LDS and barriers, some 5 us of a block that everything waits for.  Router and choice of
// eight experts in four groups at width 4,096 / 2,048, eight rows: 9.8 -> 6.4 and 8.6 -> 5.3 us; without groups 7.2 -> 4.8 and 6.5 -> 3.7; the
// choice alone of 1,803 rows 6.4 -> 4.2.
// Of scores that compare with nothing (NaN) none is chosen, and a group whose total is infinite is kept beside the others, as there.
#define ROUTE_FEW 16
__device__ inline void route_few(const Route& r, const float* logits, int t, bool live) {
  const int e = threadIdx.x % ROUTE_FEW, base = threadIdx.x % TP_WAVE - e, experts = r.experts;
  const bool mine = e < experts;
  const float correction = mine && r.correction != nullptr ? r.correction[e] : 0.f;
  const float z = mine ? logits[e] + (r.bias != nullptr ? r.bias[e] : 0.f) : -INFINITY;
  float sc;
  if (r.score_kind == 1) {
    sc = mine ? 1.0f / (1.0f + expf(-z)) : 0.f;
  } else {
    const float mx = row_max(z);
    sc = mine ? expf(z - mx) : 0.f;
    sc *= 1.0f / row_sum(sc);
  }
  float ch = mine ? (r.correction != nullptr ? sc + correction : sc) : -INFINITY;
  if (r.groups > 1) {
    const int per = experts / r.groups, first = e / per * per;   // (lanes past the last expert: a group of their own, never looked at)
    float all[ROUTE_FEW], totals[ROUTE_FEW];
#pragma unroll
    for (int j = 0; j < ROUTE_FEW; ++j) all[j] = __shfl(ch, base + j, TP_WAVE);
    // the group's largest scores one after the other (equal scores: the lower index first), added in that order
    float total = 0.f, pv = INFINITY;
    int pi = -1;
    for (int b = 0; b < r.group_best; ++b) {
      float best = -INFINITY;
      int bi = -1;
#pragma unroll
      for (int j = 0; j < ROUTE_FEW; ++j)
        if (j >= first && j < first + per && (all[j] < pv || (all[j] == pv && j > pi)) && (bi < 0 || all[j] > best)) {
          best = all[j];
          bi = j;
        }
      if (bi >= 0) total = b == 0 ? best : total + best;
      pv = bi >= 0 ? best : -INFINITY;
      pi = bi >= 0 ? bi : ROUTE_FEW;
    }
#pragma unroll
    for (int j = 0; j < ROUTE_FEW; ++j) totals[j] = __shfl(total, base + j, TP_WAVE);
    int in_front = 0;
#pragma unroll
    for (int j = 0; j < ROUTE_FEW; ++j)
      if (j < experts && (j < first || j >= first + per) && totals[j] != INFINITY && (totals[j] > total || (totals[j] == total && j < first))) ++in_front;
    // (counted member by member: per times the groups in front)
    if (!(total == INFINITY || (total == total && in_front < r.keep * per))) ch = -INFINITY;
  }
  float all[ROUTE_FEW];
#pragma unroll
  for (int j = 0; j < ROUTE_FEW; ++j) all[j] = __shfl(ch, base + j, TP_WAVE);
  int place = 0;
#pragma unroll
  for (int j = 0; j < ROUTE_FEW; ++j)
    if (all[j] > ch || (all[j] == ch && j < e)) ++place;
  const bool won = mine && ch > -INFINITY && place < r.top;
  float w = sc;
  if (r.normalize) {
    float chosen_sum = 0.f;      // (in the order of choice)
    for (int it = 0; it < r.top; ++it) {
      const unsigned there = (unsigned)(__ballot(won && place == it) >> base) & 0xffffu;
      const float s = __shfl(sc, base + (there != 0 ? __ffs(there) - 1 : 0), TP_WAVE);
      if (there != 0) chosen_sum += s;
    }
    w = sc * (r.scale / (chosen_sum + r.sum_eps));
  } else if (r.scale != 1.0f) {
    w = sc * r.scale;
  }
  if (!live || !mine) return;
  r.dense[(size_t)t * experts + e] = won ? w : 0.f;
  if (won) {
    r.ids[(size_t)t * r.top + place] = e;
    r.weights[(size_t)t * r.top + place] = w;
  }
}
