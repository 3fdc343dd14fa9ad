// From a token's router logits to the weights of its experts: what every kernel that makes the choice shares.
#pragma once

#include "common.h"

#define ROUTE_MAX_EXPERTS 1024

struct RouteCall {
  int dtype;                // element type of `h`: 0 float32, 1 bfloat16
  int tokens, width;
  int experts;              // router outputs: experts with tensors and identity experts together
  int top;
  int groups, keep;         // groups <= 1: every expert can be chosen
  const void* h;            // [tokens][ldh]
  int64_t ldh;
  const float* W;           // [experts][width] float32
  const float* correction;  // [experts] or null: added to the scores for the choice only
  const float* gate_w;      // [width] float32 or null
  float* weights;           // [tokens][experts]
  float* gate;              // [tokens]: sigmoid(gate_w . h), or null
  int score;                // 0: softmax over all experts; 1: each logit's sigmoid; 2: the logits, softmax over the chosen
  int group_rank;           // a group's score is the sum of its so many best (corrected) scores; 0 or 1: its best
  int normalize;            // 1: the chosen experts' scores over their sum; 0: the scores as they are
  const float* bias;        // [experts] or null: added to the logits
  unsigned long long* used; // [tokens] or null: bit e of a token's word is set where its weight of expert e < 64 is not zero
};

// The best (value, index) of a wave; among equal values the lowest index.  Every lane gets it.
__device__ __forceinline__ void wave_best(float& value, int& index) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float other = __shfl_xor(value, o, 64);
    const int other_index = __shfl_xor(index, o, 64);
    if (other > value || (other == value && other_index < index)) { value = other; index = other_index; }
  }
}

// Corrections and biases of a lane's first four experts.
struct RouteEarly {
  float correction[4], bias[4];
  __device__ __forceinline__ void load(const RouteCall& c) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      correction[j] = c.correction && lane + 64 * j < c.experts ? c.correction[lane + 64 * j] : 0.f;
      bias[j] = c.bias && lane + 64 * j < c.experts ? c.bias[lane + 64 * j] : 0.f;
    }
  }
};

// From a token's logits to its experts, by ONE wave: the experts dealt to its lanes, maxima and choices as wave
// reductions.  `score` holds the logits and afterwards the scores, `choice` afterwards the token's weight of every expert,
// zero where it was not chosen (both in LDS, written by the lane whose expert it is).  At most `top` experts are chosen whatever
// the values: a lane remembers which of its experts are taken, no value stands for it (a correction or logit may be infinite).
// Returns the weight of the lane's first expert.
__device__ __forceinline__ float route_choice(const RouteCall& c, const RouteEarly& early, float* score, float* choice) {
  const int lane = threadIdx.x & 63;
  if (c.bias)                                       // a lane keeps to its own experts
    for (int e = lane, j = 0; e < c.experts; e += 64, ++j) score[e] += j < 4 ? early.bias[j < 4 ? j : 0] : c.bias[e];
  float top_logit = -INFINITY;
  for (int e = lane; e < c.experts; e += 64) top_logit = fmaxf(top_logit, score[e]);
  top_logit = wave_max(top_logit);
  float total = 0.f;
  for (int e = lane; e < c.experts; e += 64) total += expf(score[e] - top_logit);
  total = wave_sum(total);
  for (int e = lane, j = 0; e < c.experts; e += 64, ++j) {     // a lane keeps to its own experts: no other lane reads them yet
    const float z = score[e];
    const float s = c.score == 1 ? 1.0f / (1.0f + expf(-z)) : c.score == 2 ? expf(z - top_logit) : expf(z - top_logit) / total;
    score[e] = s;
    choice[e] = (c.score == 2 ? z : s) + (c.correction ? (j < 4 ? early.correction[j < 4 ? j : 0] : c.correction[e]) : 0.f);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  if (c.groups > 1) {
    // a group's score is its best corrected score; the best `keep` groups stay open, the experts of
    // the others are shut out (minus infinity, since corrected scores may be negative).  Lane g
    // holds group g (at most 64 groups).
    const int per = c.experts / c.groups;
    float group_score = -INFINITY;
    if (lane < c.groups) {
      if (c.group_rank <= 1) {
        for (int i = 0; i < per; ++i) group_score = fmaxf(group_score, choice[lane * per + i]);
      } else {
        // the sum of the group's `group_rank` best: best after best, each below the one before it or
        // an equal one at a higher index
        float last = INFINITY;
        int last_index = -1;
        group_score = 0.f;
        for (int r = 0; r < c.group_rank && r < per; ++r) {
          float best = -INFINITY;
          int best_index = -1;
          for (int i = 0; i < per; ++i) {
            const float v = choice[lane * per + i];
            const bool left = v < last || (v == last && i > last_index);
            if (left && (best_index < 0 || v > best)) { best = v; best_index = i; }
          }
          group_score += best;
          last = best;
          last_index = best_index;
        }
      }
    }
    bool open = false;
    for (int kept = 0; kept < c.keep; ++kept) {
      float value = (lane < c.groups && !open) ? group_score : -INFINITY;
      int index = (lane < c.groups && !open) ? lane : 0x7fffffff;
      // (a group whose score is minus infinity itself still ranks before no group at all)
      unsigned long long candidates = __builtin_amdgcn_ballot_w64(lane < c.groups && !open);
      wave_best(value, index);
      if (index == 0x7fffffff) index = __builtin_ctzll(candidates);
      if (lane == index) open = true;
    }
    if (lane < c.groups && !open)
      for (int i = 0; i < per; ++i) choice[lane * per + i] = -INFINITY;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  float sum = 0.f;
  if (c.experts <= 64) {                           // (an expert a lane: nothing is read again while they are chosen)
    const float own = lane < c.experts ? score[lane] : 0.f, corrected = lane < c.experts ? choice[lane] : -INFINITY;
    bool taken = false;
    for (int k = 0; k < c.top; ++k) {
      const bool left = corrected > -INFINITY && !taken;
      float value = left ? corrected : -INFINITY;
      int index = left ? lane : 0x7fffffff;
      wave_best(value, index);
      if (index == 0x7fffffff) break;              // (nothing left above minus infinity, or what is left is not a number)
      if (lane == index) taken = true;
      sum += score[index];
    }
    const float weight = taken ? own * (c.normalize ? 1.0f / (sum + 1e-20f) : 1.0f) : 0.f;
    if (lane < c.experts) choice[lane] = weight;
    return weight;
  }
  unsigned taken = 0;                              // bit j: the lane's expert lane + 64 j (ROUTE_MAX_EXPERTS: sixteen of them)
  for (int k = 0; k < c.top; ++k) {
    float value = -INFINITY;
    int index = 0x7fffffff;
    for (int e = lane, j = 0; e < c.experts; e += 64, ++j) {
      const float v = choice[e];
      if (v > value && !(taken >> j & 1)) { value = v; index = e; }     // (ascending e: the lowest index among equals)
    }
    wave_best(value, index);
    if (index == 0x7fffffff) break;
    if (lane == (index & 63)) taken |= 1u << (index >> 6);
    sum += score[index];
  }
  const float inverse = c.normalize ? 1.0f / (sum + 1e-20f) : 1.0f;
  for (int e = lane, j = 0; e < c.experts; e += 64, ++j) choice[e] = taken >> j & 1 ? score[e] * inverse : 0.f;
  return choice[lane];
}

inline const char* route_refusal(const RouteCall* c) {
  if (c->experts <= 0 || c->experts > ROUTE_MAX_EXPERTS) return "1 to 1024 experts are possible";
  if (c->top <= 0 || c->top > c->experts || c->top > 64) return "a token uses 1 to 64 of the experts";
  if (c->groups > 1) {
    if (c->groups > 64 || c->experts % c->groups != 0 || c->keep <= 0 || c->keep > c->groups)
      return "the groups (at most 64) must divide the experts, and 1 to all of them stay open";
    if (c->keep * (c->experts / c->groups) < c->top) return "the open groups hold fewer experts than a token uses";
  }
  if (c->score < 0 || c->score > 2 || (c->score == 2 && c->normalize != 1) || c->group_rank < 0 || (c->normalize != 0 && c->normalize != 1))
    return "not a router these kernels know";
  return nullptr;
}

// Rows of a product that are still to be weighed: column e * ff + i of row t times the token's weight of expert e, made from its
// router's logits (route: dtype, experts, top, groups, keep, correction, score, group_rank, normalize, bias; nothing
// else is looked at); columns behind the experts as they are.
struct WeighedRows {
  RouteCall route;
  int ff;
  const float* logits;      // [rows][ld_logits]
  int64_t ld_logits;
};
#define WEIGHED_MAX_ROWS 16
#define WEIGHED_MAX_EXPERTS 64
