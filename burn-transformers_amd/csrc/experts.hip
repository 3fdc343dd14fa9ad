// Kernels of the routed feed-forward (a mixture of gated experts).
//   * route: per token the router's logits (32-bit, from 32-bit router weights), their softmax over
//     all experts, the choice of `top` experts by score + correction, restricted to the best `keep`
//     of `groups` equal groups of neighbouring experts (a group's score is its best corrected
//     score), and the chosen experts' softmax scores divided by their sum.  The result is a dense
//     row of weights per token, zero where an expert was not chosen.  Optionally the sigmoid gate
//     of an expert that every token uses (one number per token).
//   * gated activation: hidden = weight * silu(gate) * up for every expert side by side (and the
//     always-on expert with its sigmoid gate as weight), so that ONE product with the experts' down
//     matrices laid side by side gives the weighted sum of their outputs; experts whose output is
//     their input ("identity experts", the last router outputs) leave weight * h as 32-bit rows.
// A router may differ in three ways (`score`, `group_rank`, `normalize`): scores that are the
// logits' sigmoids instead of their softmax, a group's score that is the sum of its `group_rank` best
// instead of its best, and weights that are the chosen experts' scores as they are instead of over
// their sum.  The experts' activation (`act`) is silu(g) * u, or with a `limit`:
// g' = min(g, limit), u' = clamp(u, -limit, limit), g' * sigmoid(alpha * g') * (u' + 1).
// A third kind of score makes the choice by the logits themselves (with the correction) and weighs the chosen
// experts by the softmax over THEIR logits alone.  `bias` is added to the logits first.
// Ties between equal scores go to the lower index.
//   * weighed experts, for small steps: the router's logits come from the product that makes the experts' units (rows of
//     the same matrix, 32-bit results), and ONE kernel makes the choice and multiplies the units by their weights.
#include "host.h"
#include "tile.h"

#include <type_traits>

#define ROUTE_THREADS 1024
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

// Corrections and biases of a lane's first four experts.
struct RouteEarly {
  float correction[4], bias[4];
  __device__ __forceinline__ void load(const RouteCall& c) {
    const int lane = threadIdx.x & 63;
    correction[0] = c.correction && lane < c.experts ? c.correction[lane] : 0.f;
    bias[0] = c.bias && lane < c.experts ? c.bias[lane] : 0.f;
    if (c.experts <= 64) return;
#pragma unroll
    for (int j = 1; j < 4; ++j) {
      correction[j] = c.correction && lane + 64 * j < c.experts ? c.correction[lane + 64 * j] : 0.f;
      bias[j] = c.bias && lane + 64 * j < c.experts ? c.bias[lane + 64 * j] : 0.f;
    }
  }
};

// The groups that stay open, of lane g group g: the best `keep` by their scores.  `choice` holds the corrected scores in LDS.
__device__ __forceinline__ bool route_group_open(const RouteCall& c, const float* choice) {
  const int lane = threadIdx.x & 63;
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
  return open;
}

// From a token's logits to its experts, by ONE wave, for at most 64 experts: an expert a lane, `logit` its lane's.  What this takes is a chain of
// reductions and of trips to LDS behind a product that is itself 2 us, so values stay in lanes: an expert's rank is the number of
// lanes that go before it (their values read lane by lane, independent of each other), where choosing the best, `top` times over, is as many
// reductions one after the other; these stay where the experts are many beside the chosen.
// Measured (us, by reductions with everything in LDS / so): a decode step's weigh_experts of 4 and 8 tokens, 2 of 8 experts, 3.54 / 2.91.
// `choice`: LDS of the wave, used by groups.  Returns the token's weight of the lane's expert, zero where it was not chosen or there is none.
__device__ __forceinline__ float route_lanes(const RouteCall& c, const RouteEarly& early, float logit, float* choice) {
  const int lane = threadIdx.x & 63;
  const bool mine = lane < c.experts;
  const float z = c.bias ? logit + early.bias[0] : logit;
  float s;
  if (c.score == 1) {
    s = 1.0f / (1.0f + expf(-z));
  } else {
    const float top_logit = wave_max(mine ? fmaxf(-INFINITY, z) : -INFINITY);
    s = expf(z - top_logit);
    if (c.score == 0) s /= wave_sum(mine ? s : 0.f);
  }
  const float own = mine ? s : 0.f;
  float corrected = mine ? (c.score == 2 ? z : s) + early.correction[0] : -INFINITY;
  if (c.groups > 1) {
    if (mine) choice[lane] = corrected;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const unsigned long long open = __builtin_amdgcn_ballot_w64(route_group_open(c, choice));
    if (mine && !(open >> (lane / (c.experts / c.groups)) & 1)) corrected = -INFINITY;
  }
  const bool can = corrected > -INFINITY;          // (not minus infinity and a number: the others are never chosen)
  const float value = can ? corrected : -INFINITY;
  float sum = 0.f;
  bool taken = false;
  auto score_of = [&](int expert) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, own), expert)); };
  if (c.experts <= 16 * c.top) {
    int rank = 0;
    for (int j0 = 0; j0 < c.experts; j0 += 8)
#pragma unroll
      for (int j = j0; j < j0 + 8; ++j) {          // (lanes behind the experts hold minus infinity, which goes before nothing)
        const float other = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, value), j));
        rank += other > value || (other == value && j < lane) ? 1 : 0;
      }
    taken = can && rank < c.top;
    for (int k = 0; k < c.top; ++k) {
      const unsigned long long at = __builtin_amdgcn_ballot_w64(can && rank == k);
      if (at == 0) break;
      sum += score_of(__builtin_ctzll(at));
    }
  } else {
    for (int k = 0; k < c.top; ++k) {
      const bool left = can && !taken;
      float best = left ? value : -INFINITY;
      int index = left ? lane : 0x7fffffff;
      wave_best(best, index);
      index = __builtin_amdgcn_readfirstlane(index);
      if (index == 0x7fffffff) break;              // (nothing left)
      if (lane == index) taken = true;
      sum += score_of(index);
    }
  }
  return taken ? own * (c.normalize ? 1.0f / (sum + 1e-20f) : 1.0f) : 0.f;
}

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
    const int per = c.experts / c.groups;
    const bool open = route_group_open(c, choice);
    if (lane < c.groups && !open)
      for (int i = 0; i < per; ++i) choice[lane * per + i] = -INFINITY;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  float sum = 0.f;
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

// One work-group of sixteen waves per token.  Logits: a wave takes whole outputs (two at a time, the
// outputs dealt round the waves), its lanes the columns, sixteen a turn; nothing of a turn's loads stands
// behind a branch of its own, so all of them are in flight together, every wave's at once: the
// logits cost one round trip to memory and a wave reduction, and no sum crosses waves.  (Columns
// dealt to the threads and sixteen outputs' sums met through LDS, batch after batch, took 6 us a batch
// of sixteen outputs: a decode step has few tokens, and a kernel's time is the chain of its waits.)
// Everything after the logits is the first wave's alone, the experts dealt to its lanes, maxima and
// choices as wave reductions: no barrier, no serial scan.
#define ROUTE_OUTPUTS 2         // outputs whose sums a wave carries at once
#define ROUTE_COLUMNS 16        // columns of a lane and turn

template <typename T>
__global__ void __launch_bounds__(ROUTE_THREADS) route_kernel(RouteCall c) {
  __shared__ float score[ROUTE_MAX_EXPERTS];      // logits, then softmax scores
  __shared__ float choice[ROUTE_MAX_EXPERTS];     // scores with the correction, -inf where shut out; then the weights
  __shared__ float gate_sum;
  const int t = blockIdx.x, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const T* h = static_cast<const T*>(c.h) + (int64_t)t * c.ldh;
  const int outputs = c.experts + (c.gate_w ? 1 : 0);
  const int waves = blockDim.x >> 6;              // sixteen in steps of few tokens, four where tokens fill the chip anyway
  // the corrections and biases of this lane's first experts are asked for now, with the first loads
  RouteEarly early;
  if (wave == 0) early.load(c);
  for (int first = wave; first < outputs; first += waves * ROUTE_OUTPUTS) {
    float sums[ROUTE_OUTPUTS];
    const float* rows[ROUTE_OUTPUTS];               // an output beyond the last reads the last one's row and is dropped
#pragma unroll
    for (int j = 0; j < ROUTE_OUTPUTS; ++j) {
      sums[j] = 0.f;
      const int e = first + waves * j < outputs ? first + waves * j : outputs - 1;
      rows[j] = e < c.experts ? c.W + (int64_t)e * c.width : c.gate_w;
    }
    for (int col0 = lane; col0 < c.width; col0 += 64 * ROUTE_COLUMNS) {
      int cc[ROUTE_COLUMNS];
      float xs[ROUTE_COLUMNS];
#pragma unroll
      for (int u = 0; u < ROUTE_COLUMNS; ++u) {
        const int col = col0 + 64 * u;
        cc[u] = col < c.width ? col : 0;
        xs[u] = to_float(h[cc[u]]);
      }
      float ws[ROUTE_OUTPUTS][ROUTE_COLUMNS];
#pragma unroll
      for (int j = 0; j < ROUTE_OUTPUTS; ++j)
#pragma unroll
        for (int u = 0; u < ROUTE_COLUMNS; ++u) ws[j][u] = rows[j][cc[u]];
#pragma unroll
      for (int u = 0; u < ROUTE_COLUMNS; ++u) xs[u] = col0 + 64 * u < c.width ? xs[u] : 0.f;
#pragma unroll
      for (int j = 0; j < ROUTE_OUTPUTS; ++j)
#pragma unroll
        for (int u = 0; u < ROUTE_COLUMNS; ++u) sums[j] = fmaf(ws[j][u], xs[u], sums[j]);
    }
#pragma unroll
    for (int j = 0; j < ROUTE_OUTPUTS; ++j) {
      const float sum = wave_sum(sums[j]);
      const int e = first + waves * j;
      if (lane == 0 && e < outputs) {
        if (e < c.experts) score[e] = sum;
        else gate_sum = sum;                         // (stored at the end: nothing waits for a store meanwhile)
      }
    }
  }
  __syncthreads();
  if (wave != 0) return;
  const float first = c.experts <= 64 ? route_lanes(c, early, lane < c.experts ? score[lane] : 0.f, choice) : route_choice(c, early, score, choice);
  // the one store of a lane's experts: the chosen ones' scores over their sum, zero elsewhere
  float* weights = c.weights + (int64_t)t * c.experts;
  for (int e = lane; e < c.experts; e += 64) {
    const float w = e < 64 ? first : choice[e];
    weights[e] = w;
    if (e < 64 && c.used) {
      const unsigned long long used = __builtin_amdgcn_ballot_w64(w != 0.f);
      if (lane == 0) c.used[t] = used;
    }
  }
  if (c.gate_w && lane == 0) c.gate[t] = 1.0f / (1.0f + expf(-gate_sum));
}

// The same for steps of many tokens: a work-group takes sixteen tokens, whose logits are a product of 16 rows by the router's
// outputs on the matrix units (v_mfma_f32_16x16x4_f32: h widened, the router's 32 bits as they are), its sixteen waves a
// sixteenth of the columns each, so that the router is read once for sixteen tokens and not once a token; then every
// wave makes the choice of one of them.  Of an instruction's four K values step i takes column 4 g + i of a lane group's
// four, which are one read.  A work-group's own chain (two trips to memory, the sums' meeting, the choice) is 5 to
// 7 us for 512 and 1,024 columns whatever the step, so steps of fewer than ROUTE_ROWS_MIN tokens keep a work-group a token.  Measured (us, a
// work-group a token / sixteen; outputs of columns): 9 of 1,024 1,000 tokens 5.5 / 6.6, 1,200 6.5 / 6.6, 1,400 7.2 / 6.6, 1,530 7.4 / 6.6; 17 of 1,024 1,000
// 7.8 / 8.7, 1,200 9.1 / 8.7, 1,530 10.4 / 8.7; 8 of 512 1,000 4.6 / 4.8, 1,200 4.9 / 4.8, 1,530 5.5 / 4.8; 32 of 2,048 600 15.3 / 15.3, 1,530 25.9 / 15.4.  In a step of
// 1,809 tokens 9 outputs of 1,024 and a gate take 8.5.  From 1,280 tokens on sixteen would be the faster way; but the two add a logit's products
// in different orders, and a choice between experts that are nearly equal may fall the other way: the line stays where it is.
#define ROUTE_ROWS 16
#define ROUTE_ROWS_TILES 2      // (most outputs: 32)
#define ROUTE_ROWS_AHEAD 4      // chunks of 16 columns on their way

template <typename T, int TILES>
__global__ void __launch_bounds__(64 * ROUTE_ROWS) route_rows_kernel(RouteCall c) {
  typedef __attribute__((__vector_size__(4 * sizeof(T)))) T T4;
  __shared__ __attribute__((aligned(16))) floatx4 parts[ROUTE_ROWS][TILES][64];
  __shared__ float score[ROUTE_ROWS][16 * TILES], choice[ROUTE_ROWS][16 * TILES];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, n = lane & 15;
  const int t0 = blockIdx.x * ROUTE_ROWS, outputs = c.experts + (c.gate_w ? 1 : 0);
  const T* h = static_cast<const T*>(c.h) + (int64_t)min(t0 + n, c.tokens - 1) * c.ldh + 4 * g;
  const float* rows[TILES];                          // an output beyond the last reads the last one's row and is dropped
#pragma unroll
  for (int j = 0; j < TILES; ++j) {
    const int e = min(16 * j + n, outputs - 1);
    rows[j] = (e < c.experts ? c.W + (int64_t)e * c.width : c.gate_w) + 4 * g;
  }
  RouteEarly early;
  early.load(c);
  floatx4 sums[TILES];
#pragma unroll
  for (int j = 0; j < TILES; ++j) sums[j] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int chunks = c.width / 16;
  for (int k0 = wave; k0 < chunks; k0 += ROUTE_ROWS * ROUTE_ROWS_AHEAD) {
    T4 xs[ROUTE_ROWS_AHEAD];
    floatx4 ws[ROUTE_ROWS_AHEAD][TILES];
#pragma unroll
    for (int u = 0; u < ROUTE_ROWS_AHEAD; ++u) {
      const int col = 16 * min(k0 + ROUTE_ROWS * u, chunks - 1);
      xs[u] = *reinterpret_cast<const T4*>(h + col);
#pragma unroll
      for (int j = 0; j < TILES; ++j) ws[u][j] = *reinterpret_cast<const floatx4*>(rows[j] + col);
    }
#pragma unroll
    for (int u = 0; u < ROUTE_ROWS_AHEAD; ++u) {
      if (k0 + ROUTE_ROWS * u >= chunks) break;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < TILES; ++j) sums[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(to_float(xs[u][i]), ws[u][j][i], sums[j], 0, 0, 0);
    }
  }
#pragma unroll
  for (int j = 0; j < TILES; ++j) parts[wave][j][lane] = sums[j];        // lane holds tokens 4 g + i, output n
  __syncthreads();
  for (int k = tid; k < ROUTE_ROWS * 16 * TILES; k += 64 * ROUTE_ROWS) {
    const int t = k / (16 * TILES), e = k % (16 * TILES), from = 16 * (t >> 2) + (e & 15);
    float logit = 0.f;
#pragma unroll
    for (int w = 0; w < ROUTE_ROWS; ++w) logit += reinterpret_cast<const float*>(&parts[w][e >> 4][from])[t & 3];
    score[t][e] = logit;
  }
  __syncthreads();
  const int t = t0 + wave;
  if (t >= c.tokens) return;
  const float gate_sum = score[wave][c.gate_w ? c.experts : 0];
  const float w = route_lanes(c, early, lane < c.experts ? score[wave][lane] : 0.f, choice[wave]);
  if (lane < c.experts) c.weights[(int64_t)t * c.experts + lane] = w;
  const unsigned long long used = __builtin_amdgcn_ballot_w64(w != 0.f);
  if (lane == 0 && c.used) c.used[t] = used;
  if (lane == 0 && c.gate_w) c.gate[t] = 1.0f / (1.0f + expf(-gate_sum));
}

// (Few outputs of wide rows from 1,792 tokens on: 8 of 1,024 bfloat16 columns 1,530 tokens 5.5 / 6.2, 1,780 6.0 / 6.2; of 4,096 1,530 13.8 / 14.7, 1,780 15.6 /
// 14.8; of 4,096 float ones 13.3 / 14.9 and 14.5 / 14.8.)
#define ROUTE_ROWS_MIN 1536
#define ROUTE_ROWS_MIN_FEW 1792

template <typename T>
static bool launch_route_rows(hipStream_t stream, const RouteCall& c) {
  const int outputs = c.experts + (c.gate_w ? 1 : 0), tiles = (outputs + 15) / 16;
  if (c.tokens < (outputs <= 8 && c.width >= 1024 ? ROUTE_ROWS_MIN_FEW : ROUTE_ROWS_MIN) || tiles > ROUTE_ROWS_TILES || c.width % 16 != 0 || c.ldh % 4 != 0 || ((uintptr_t)c.h & (4 * sizeof(T) - 1)) ||
      (((uintptr_t)c.W | (uintptr_t)c.gate_w) & 15))
    return false;
  dim3 grid((c.tokens + ROUTE_ROWS - 1) / ROUTE_ROWS), block(64 * ROUTE_ROWS);
  if (tiles == 1) hipLaunchKernelGGL((route_rows_kernel<T, 1>), grid, block, 0, stream, c);
  else hipLaunchKernelGGL((route_rows_kernel<T, 2>), grid, block, 0, stream, c);
  return true;
}

static const char* route_refusal(const RouteCall* c) {
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

BT_EXPORT int bt_route_call(void* stream, const RouteCall* c) {
  if (c->tokens <= 0) return BT_OK;
  if (const char* wrong = route_refusal(c))
    BT_REFUSE("route: %d of %d experts a token, %d of %d groups, score %d: %s", c->top, c->experts, c->keep, c->groups, c->score, wrong);
  if (c->width <= 0) BT_REFUSE("route: width %d must be positive", c->width);
  if (!c->h || !c->W || !c->weights || (c->gate_w && !c->gate)) BT_REFUSE("route: missing operand");
  if (c->dtype == 0 ? launch_route_rows<float>((hipStream_t)stream, *c) : launch_route_rows<bf16_t>((hipStream_t)stream, *c))
    return bt_check_launch("route");
  // (measured at 2,048 tokens of width 2,048: 32 us with sixteen waves a token, 18 with four)
  dim3 grid(c->tokens), block(c->tokens <= 256 ? ROUTE_THREADS : 256);
  if (c->dtype == 0)
    hipLaunchKernelGGL(route_kernel<float>, grid, block, 0, (hipStream_t)stream, *c);
  else
    hipLaunchKernelGGL(route_kernel<bf16_t>, grid, block, 0, (hipStream_t)stream, *c);
  return bt_check_launch("route");
}

struct GatedExpertsCall {
  int dtype;                // element type of `gu`, `hidden` and `h`
  int tokens;
  int experts;              // experts with tensors, each `ff` wide
  int ff;
  int shared_ff;            // width of the expert every token uses; 0: none
  int identity;             // identity experts: router outputs experts .. experts + identity - 1
  int hidden_cols;          // columns of `hidden` written: experts * ff + shared_ff, then zeros
  int width;
  const void* gu;           // [tokens][ld_gu]: per expert its gate rows (ff) then its up rows (ff); then the shared expert's
  int64_t ld_gu;
  const float* weights;     // [tokens][experts + identity]
  const float* gate;        // [tokens]: the shared expert's weight, or null
  void* hidden;             // [tokens][ld_hidden]
  int64_t ld_hidden;
  const void* h;            // [tokens][ldh]: the experts' input (read for identity experts only)
  int64_t ldh;
  float* identity_out;      // [tokens][width] float32: (sum of the identity experts' weights) * h; or null
  int act;                  // 0: silu(g) * u; 1: min(g, limit) * sigmoid(alpha * min(g, limit)) * (clamp(u, -limit, limit) + 1);
                            // 2, 3, 4: units WITHOUT a gate, gelu(u) in its exact (erf) form, silu(u) and max(u, 0)^2: `gu`
                            // then holds per expert its ff up rows only, the shared expert's behind them
  float limit;
  float alpha;
};

template <int ACT>
__device__ __forceinline__ float plain_unit_as(float u) {
  if constexpr (ACT == 4) return u > 0.f ? u * u : 0.f;
  else if constexpr (ACT == 2) return 0.5f * u * (1.0f + erff(u * 0.70710678118654752f));
  else return u / (1.0f + expf(-u));
}
template <int ACT>
__device__ __forceinline__ float gated_unit_as(float limit, float alpha, float g, float u) {
  if constexpr (ACT == 1) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return g / (1.0f + expf(-alpha * g)) * (u + 1.0f);
  }
  return g / (1.0f + expf(-g)) * u;
}
__device__ __forceinline__ float plain_unit(const GatedExpertsCall& c, float u) {
  return c.act == 4 ? plain_unit_as<4>(u) : c.act == 2 ? plain_unit_as<2>(u) : plain_unit_as<3>(u);
}
__device__ __forceinline__ float gated_unit(const GatedExpertsCall& c, float g, float u) {
  return c.act == 1 ? gated_unit_as<1>(c.limit, c.alpha, g, u) : gated_unit_as<0>(c.limit, c.alpha, g, u);
}

template <typename T>
__global__ void __launch_bounds__(256) gated_experts_kernel(GatedExpertsCall c) {
  const int t = blockIdx.x;
  const T* gu = static_cast<const T*>(c.gu) + (int64_t)t * c.ld_gu;
  T* hidden = static_cast<T*>(c.hidden) + (int64_t)t * c.ld_hidden;
  const float* weights = c.weights + (int64_t)t * (c.experts + c.identity);
  const int routed = c.experts * c.ff;
  const bool gated = c.act < 2;
  // a token's columns are dealt to the work-groups of its row of the grid (a decode step has few tokens)
  for (int col = blockIdx.y * blockDim.x + threadIdx.x; col < c.hidden_cols; col += gridDim.y * blockDim.x) {
    float out = 0.f;
    if (col < routed) {
      const int e = col / c.ff, i = col - e * c.ff;
      const float w = weights[e];
      if (w != 0.f && gated) {
        const float g = to_float(gu[(int64_t)e * 2 * c.ff + i]), u = to_float(gu[(int64_t)e * 2 * c.ff + c.ff + i]);
        out = w * gated_unit(c, g, u);
      } else if (w != 0.f) {
        out = w * plain_unit(c, to_float(gu[col]));
      }
    } else if (col < routed + c.shared_ff) {
      const int i = col - routed;
      const float share = c.gate ? c.gate[t] : 1.0f;
      if (gated) {
        const float g = to_float(gu[(int64_t)2 * routed + i]), u = to_float(gu[(int64_t)2 * routed + c.shared_ff + i]);
        out = share * gated_unit(c, g, u);
      } else {
        out = share * plain_unit(c, to_float(gu[col]));
      }
    }
    hidden[col] = from_float<T>(out);
  }
  if (c.identity_out) {
    float w = 0.f;
    for (int i = 0; i < c.identity; ++i) w += weights[c.experts + i];
    const T* h = static_cast<const T*>(c.h) + (int64_t)t * c.ldh;
    for (int col = blockIdx.y * blockDim.x + threadIdx.x; col < c.width; col += gridDim.y * blockDim.x)
      c.identity_out[(int64_t)t * c.width + col] = w != 0.f ? w * to_float(h[col]) : 0.f;
  }
}

// The same for units without a gate whose columns can be taken 16 bytes at a time: no piece lies in two experts.
template <typename T>
__global__ void __launch_bounds__(256) plain_experts_kernel(GatedExpertsCall c) {
  constexpr int PER = 16 / sizeof(T);
  const int t = blockIdx.x, routed = c.experts * c.ff / PER, pieces = c.hidden_cols / PER;
  const int4v* up = reinterpret_cast<const int4v*>(static_cast<const T*>(c.gu) + (int64_t)t * c.ld_gu);
  int4v* hidden = reinterpret_cast<int4v*>(static_cast<T*>(c.hidden) + (int64_t)t * c.ld_hidden);
  const float* weights = c.weights + (int64_t)t * (c.experts + c.identity);
  const float share = c.gate ? c.gate[t] : 1.0f;
  const int all = (c.experts * c.ff + c.shared_ff) / PER;
  for (int piece = blockIdx.y * blockDim.x + threadIdx.x; piece < pieces; piece += gridDim.y * blockDim.x) {
    const float w = piece < routed ? weights[piece * PER / c.ff] : piece < all ? share : 0.f;
    int4v v = {0, 0, 0, 0};
    if (w != 0.f) {
      v = up[piece];
      T* values = reinterpret_cast<T*>(&v);
#pragma unroll
      for (int i = 0; i < PER; ++i) values[i] = from_float<T>(w * plain_unit(c, to_float(values[i])));
    }
    hidden[piece] = v;
  }
}

BT_EXPORT int bt_gated_experts_call(void* stream, const GatedExpertsCall* c) {
  if (c->tokens <= 0) return BT_OK;
  if (c->experts < 0 || c->ff <= 0 || c->shared_ff < 0 || c->identity < 0)
    BT_REFUSE("gated_experts: %d experts of %d, a shared one of %d and %d identity experts", c->experts, c->ff, c->shared_ff, c->identity);
  const int64_t columns = (int64_t)c->experts * c->ff + c->shared_ff;
  if (c->act < 0 || c->act > 4) BT_REFUSE("gated_experts: unknown activation %d", c->act);
  if (c->hidden_cols < columns || c->ld_hidden < c->hidden_cols || c->ld_gu < (c->act < 2 ? 2 : 1) * columns)
    BT_REFUSE("gated_experts: the rows do not hold the experts");
  if (!c->gu || (!c->weights && c->experts + c->identity > 0) || !c->hidden || (c->identity_out && (!c->h || c->width <= 0)))
    BT_REFUSE("gated_experts: missing operand");
  // about 1,024 columns a work-group, fewer work-groups a token where there are many tokens
  int per_token = (c->hidden_cols + 1023) / 1024;
  if (per_token > 64) per_token = 64;
  dim3 grid(c->tokens, per_token), block(256);
  const int per = c->dtype == 0 ? 4 : 8;
  if (c->act >= 2 && !c->identity_out && c->ff % per == 0 && c->shared_ff % per == 0 && c->hidden_cols % per == 0 && c->ld_gu % per == 0 &&
      c->ld_hidden % per == 0 && ((uintptr_t)c->gu & 15) == 0 && ((uintptr_t)c->hidden & 15) == 0 && c->ld_gu >= c->hidden_cols) {
    grid.y = (c->hidden_cols / per + 255) / 256;
    if (grid.y > 64) grid.y = 64;
    if (c->dtype == 0)
      hipLaunchKernelGGL(plain_experts_kernel<float>, grid, block, 0, (hipStream_t)stream, *c);
    else
      hipLaunchKernelGGL(plain_experts_kernel<bf16_t>, grid, block, 0, (hipStream_t)stream, *c);
    return bt_check_launch("gated_experts");
  }
  if (c->dtype == 0)
    hipLaunchKernelGGL(gated_experts_kernel<float>, grid, block, 0, (hipStream_t)stream, *c);
  else
    hipLaunchKernelGGL(gated_experts_kernel<bf16_t>, grid, block, 0, (hipStream_t)stream, *c);
  return bt_check_launch("gated_experts");
}

// --- experts by rows -----------------------------------------------------------------------------
//
// In a step of many tokens every expert would multiply every token, though a token uses `top` of them.  Here the tokens
// that chose an expert are listed (group_experts), one kernel makes the units of the listed rows only, the rows gathered
// by the loads that bring them into LDS and the activation and the token's weight applied to the sums while they are in
// registers, and one kernel multiplies them with the experts' down matrices and lays every (token, choice)'s output into
// a plane of its own; the norm behind adds the planes as it adds any partial sums.  The expert that every token uses is
// one more group whose list is all tokens.  Which expert and rows a work-group takes follows from the counts, which are
// on the GPU: the grid is the most tiles there can be, and work-groups beyond the counted ones leave at once.
// The tiles are TilePipe's (tile.h): 128 columns and BM rows on four waves.  Where units have a gate, the two 32-wide blocks of a wave's columns are 32 gate rows and the up rows beside them.
#define GROUP_PLACE_BITS 24        // a list's entry: the token, and behind it which of the token's choices the expert is
#define GROUP_MAX_EXPERTS 64       // (a lane an expert)

// Tiles of 128 rows (two stages, two work-groups to a compute unit) from this many rows an expert on average, tiles of 64
// (three stages, two work-groups) below and for float.  Measured with the router (us, every expert on every row / tiles of 64 /
// of 128; 8 experts of the width, two a token): width 1,024 with gates, 128 tokens 37 / 33 / 42, 512 61 / 40 / 48, 1,024 97 / 58 / 57, 2,048
// 157 / 91 / 88, 4,096 289 / 154 / 142; width 2,048 without gates and a shared expert, 200 tokens 98 / 51 / 69, 773 250 / 102 / 101, 2,048
// 378 / 221 / 192.  One work-group to a unit with more stages loses (128 rows in four: 106 us at 2,048 tokens).  Float: width
// 1,024 with gates, 128 tokens 104 / 92 / 150, 2,048 908 / 310 / 353.  65 tokens of 1,024 without gates draw (36.6 / 37.2);
// where the experts have less to do every expert on every row is the cheaper way, and the caller takes it.  Those figures are of a loop that waited for
// its operands behind every barrier and stored rows 8 bytes at a time; with TilePipe and the shared expert's tiles dealt over the XCDs, at 1,809 tokens of
// width 1,024 with a shared expert of 2,048: units 53.7 -> 48.3 us, outputs 43.0 -> 34.4; 2,048 tokens without one 43.9 -> 40.8 and 24.7 -> 22.1.
// What bounds them: two rounds of tiles of sixteen turns each, 5 us of launch, first loads and last stores beside 17 us of LDS traffic.
#define EXPERT_TALL_ROWS 192

struct GroupExpertsCall {
  int dtype;                // element type of `h`
  int tokens;
  int experts, identity;    // experts with tensors and identity experts, as in GatedExpertsCall
  int top;
  int width;
  const float* weights;     // [tokens][experts + identity]
  const unsigned long long* used;   // [tokens], as route leaves it
  int* rows;                // [experts][pitch]: the tokens that use an expert, in order
  int64_t pitch;
  int* counts;              // [experts]
  const void* h;            // [tokens][ldh]
  int64_t ldh;
  float* out;               // [top][..][ld_out]: rows of planes that no expert writes are written here: the identity experts'
  int64_t plane;            // weights * h, or zeros
  int64_t ld_out;
};

template <typename T>
__global__ void __launch_bounds__(1024) group_experts_kernel(GroupExpertsCall c) {
  __shared__ int found[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, outputs = c.experts + c.identity;
  if ((int)blockIdx.x < c.experts) {
    const int e = blockIdx.x;
    int base = 0;
    for (int t0 = 0; t0 < c.tokens; t0 += 1024) {
      const int t = t0 + threadIdx.x;
      const unsigned long long word = t < c.tokens ? c.used[t] : 0;
      const int place = __builtin_popcountll(word & ((1ull << e) - 1));
      const bool mine = (word >> e & 1) && place < c.top;             // (there is room for `top` choices of a token)
      const unsigned long long all = __builtin_amdgcn_ballot_w64(mine);
      if (lane == 0) found[wave] = __builtin_popcountll(all);
      __syncthreads();
      int before = base + __builtin_popcountll(all & ((1ull << lane) - 1)), total = 0;
      for (int i = 0; i < 16; ++i) {
        before += i < wave ? found[i] : 0;
        total += found[i];
      }
      if (mine) c.rows[e * c.pitch + before] = (place << GROUP_PLACE_BITS) | t;
      base += total;
      __syncthreads();
    }
    if (threadIdx.x == 0) c.counts[e] = base;
    return;
  }
  const int t = ((int)blockIdx.x - c.experts) * 16 + wave;              // a wave a token
  if (t >= c.tokens) return;
  const int used = __builtin_popcountll(c.used[t] & (~0ull >> (64 - c.experts)));
  if (used >= c.top) return;
  const float* w = c.weights + (int64_t)t * outputs;
  float own = 0.f;
  for (int i = 0; i < c.identity; ++i) own += w[c.experts + i];
  const T* h = static_cast<const T*>(c.h) + (int64_t)t * c.ldh;
  for (int p = used; p < c.top; ++p) {
    float* out = c.out + p * c.plane + (int64_t)t * c.ld_out;
    for (int col = lane; col < c.width; col += 64) out[col] = p == used && own != 0.f ? own * to_float(h[col]) : 0.f;
  }
}

BT_EXPORT int bt_group_experts_call(void* stream, const GroupExpertsCall* c) {
  if (c->tokens <= 0) return BT_OK;
  if (c->experts <= 0 || c->experts > GROUP_MAX_EXPERTS || c->identity < 0 || c->top <= 0 || c->top > 64 || c->width <= 0)
    BT_REFUSE("group_experts: %d experts (1..%d), %d identity experts, %d a token", c->experts, GROUP_MAX_EXPERTS, c->identity, c->top);
  if (c->tokens >= 1 << GROUP_PLACE_BITS) BT_REFUSE("group_experts: %d tokens are too many", c->tokens);
  if (!c->weights || !c->used || !c->rows || !c->counts || !c->h || !c->out || c->pitch < c->tokens || c->ldh < c->width || c->ld_out < c->width)
    BT_REFUSE("group_experts: missing operand or rows too short");
  dim3 grid(c->experts + (c->tokens + 15) / 16), block(1024);
  if (c->dtype == 0)
    hipLaunchKernelGGL(group_experts_kernel<float>, grid, block, 0, (hipStream_t)stream, *c);
  else
    hipLaunchKernelGGL(group_experts_kernel<bf16_t>, grid, block, 0, (hipStream_t)stream, *c);
  return bt_check_launch("group_experts");
}

struct ExpertProductsCall {
  int dtype;                // element type of `a`, `w` and, of the first product, `hidden`
  int second;               // 0: units of the listed rows of `a` = h; 1: `a` = the units, outputs into planes
  int tokens;
  int experts, identity, top;
  int ff, shared_ff, width; // shared_ff 0: no expert that every token uses
  const int* rows;          // as group_experts leaves them
  int64_t pitch;
  const int* counts;
  const void* h;            // [tokens][ldh]
  int64_t ldh;
  const void* w;            // first: [rows][ld_w], rows as `gu` of GatedExpertsCall has columns; second: [width][ld_w], an
  int64_t ld_w;             // expert's ff columns behind the other's, the shared expert's behind them
  const float* weights;     // [tokens][experts + identity]
  const float* gate;        // [tokens] or null
  void* hidden;             // [tokens * top][ff]: the listed rows one expert behind the other
  void* shared_hidden;      // [tokens][shared_ff]
  float* out;               // second: [top (+ 1: the shared expert's)][..][ld_out]
  int64_t plane;
  int64_t ld_out;
  int act;                  // as in GatedExpertsCall
  float limit, alpha;
};

// Which tile a work-group takes: of which expert (-1: the shared one), its first row in the expert's list and column tile.
struct GroupTile {
  int expert, first, count, column;
  int slot;                 // where the expert's rows start in `hidden`
};

template <int BM>
__device__ __forceinline__ bool group_tile(const ExpertProductsCall& c, int columns, int shared_columns, GroupTile& tile) {
  const int lane = threadIdx.x & 63;
  const int count = lane < c.experts ? c.counts[lane] : 0, tiles = (count + BM - 1) / BM;
  int rows_to = count, tiles_to = tiles;                                // sums up to and with this lane's expert
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int r = __shfl_up(rows_to, o, 64), t = __shfl_up(tiles_to, o, 64);
    if (lane >= o) { rows_to += r; tiles_to += t; }
  }
  const int routed = __builtin_amdgcn_readlane(tiles_to, 63) * columns, to_all = (c.tokens + BM - 1) / BM * shared_columns;
  const int all = routed + to_all;
  if ((int)blockIdx.x >= all) return false;
  // Every XCD takes its run of the shared expert's tiles first and of the others behind: in the second product they have their own K,
  // and numbered in one line some XCDs had the long ones alone (43 us where the others were done after 28).
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  auto start = [&](int n) { return xcd * (n >> 3) + (xcd < (n & 7) ? xcd : n & 7); };
  const int own = (to_all >> 3) + (xcd < (to_all & 7) ? 1 : 0);
  if (local < own) {
    const int id = start(to_all) + local;
    tile.expert = -1;
    tile.first = id / shared_columns * BM;
    tile.column = id % shared_columns;
    tile.count = c.tokens;
    tile.slot = 0;
    return true;
  }
  const int id = start(all) - start(to_all) + local - own;
  const int row_tile = id / columns;
  tile.column = id % columns;
  tile.expert = __builtin_ctzll(__builtin_amdgcn_ballot_w64(tiles_to > row_tile));
  tile.count = __builtin_amdgcn_readlane(count, tile.expert);
  tile.first = (row_tile - (__builtin_amdgcn_readlane(tiles_to, tile.expert) - __builtin_amdgcn_readlane(tiles, tile.expert))) * BM;
  tile.slot = __builtin_amdgcn_readlane(rows_to, tile.expert) - tile.count;
  return true;
}

template <typename T, int BM, int STAGES, bool SECOND, bool GATED>
__global__ void __launch_bounds__(256, 2) expert_products_kernel(ExpertProductsCall c) {
  constexpr int ELEMS = Mma<T>::ELEMS, ROW_K = 8 * ELEMS, BN = 128;
  typedef TilePipe<T, BM, BN, 2, 2, STAGES> Pipe;
  constexpr int TM = BM / 64;
  constexpr int HELD = !SECOND && GATED ? 64 : 128;                     // output columns of a tile
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];   // [STAGES][BM + BN][128 bytes]
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int wm = wave & 1, wn = wave >> 1, l32 = lane & 31, g = lane >> 5;
  GroupTile tile;
  const int columns = SECOND ? (c.width + HELD - 1) / HELD : (c.ff + HELD - 1) / HELD;
  const int shared_columns = c.shared_ff == 0 ? 0 : SECOND ? columns : (c.shared_ff + HELD - 1) / HELD;
  if (!group_tile<BM>(c, columns, shared_columns, tile)) return;        // (the whole work-group)
  const bool shared = tile.expert < 0;
  const int ff = shared ? c.shared_ff : c.ff, n_base = tile.column * HELD, n_end = SECOND ? c.width : ff;
  const int* list = c.rows + (int64_t)(shared ? 0 : tile.expert) * c.pitch;
  auto entry = [&](int m) { return shared ? m : list[m]; };
  auto token = [&](int m) { return entry(m) & ((1 << GROUP_PLACE_BITS) - 1); };

  // operands: a stage's rows are BM of A, then BN of W; the addresses' first parts are the same for the whole work-group
  const T *a, *w;
  if (SECOND) {
    a = shared ? static_cast<const T*>(c.shared_hidden) : static_cast<const T*>(c.hidden) + (int64_t)tile.slot * c.ff;
    w = static_cast<const T*>(c.w) + (int64_t)(shared ? c.experts : tile.expert) * c.ff;
  } else {
    a = static_cast<const T*>(c.h);
    w = static_cast<const T*>(c.w) + (int64_t)(shared ? c.experts : tile.expert) * c.ff * (GATED ? 2 : 1) * c.ld_w;
  }
  const int64_t ld_a = SECOND ? ff : c.ldh;
  // the rows' tokens and weights are asked for before the operands
  int held[TM];
  float weight[TM];
#pragma unroll
  for (int bm = 0; bm < TM; ++bm) {
    const int m = tile.first + wm * (BM / 2) + bm * 32 + l32;
    held[bm] = m < tile.count ? entry(m) : -1;
    weight[bm] = 1.f;
    if (!SECOND && held[bm] >= 0) {
      const int t = held[bm] & ((1 << GROUP_PLACE_BITS) - 1);
      if (!shared) weight[bm] = c.weights[(int64_t)t * (c.experts + c.identity) + tile.expert];
      else if (c.gate) weight[bm] = c.gate[t];
    }
  }
  floatx16 acc[2][TM];
#pragma unroll
  for (int bn = 0; bn < 2; ++bn)
#pragma unroll
    for (int bm = 0; bm < TM; ++bm)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[bn][bm][r] = 0.f;
  Pipe::template multiply<int64_t>(
      lds, reinterpret_cast<const unsigned char*>(a), reinterpret_cast<const unsigned char*>(w), (SECOND ? ff : c.width) / ROW_K,
      [&](int stage_row, bool from_w) {
        if (!from_w) {
          const int m = tile.first + stage_row < tile.count ? tile.first + stage_row : tile.count - 1;
          return (SECOND ? m : token(m)) * ld_a * (int64_t)sizeof(T);
        }
        const int r = stage_row - BM;
        int n = !SECOND && GATED ? n_base + (r >> 6) * 32 + (r & 31) : n_base + r;
        n = n < n_end ? n : n_end - 1;
        return ((!SECOND && GATED && (r & 32) ? ff : 0) + n) * c.ld_w * (int64_t)sizeof(T);
      },
      acc);
  __syncthreads();

  // lane holds D[i][j]: i = 8 * (r / 4) + 4 * g + r % 4 (column n), j = lane % 32 (row m); its rows go through LDS, so that memory
  // sees 16-byte pieces of whole rows
  typedef typename std::conditional<SECOND, float, T>::type Out;
  constexpr int COLUMNS = HELD / 2, PIECE = 16 / (int)sizeof(Out), LANES = COLUMNS / PIECE, PITCH = COLUMNS * (int)sizeof(Out) + 16;
  unsigned char* scratch = lds + wave * (BM / 2 * PITCH);
  auto units = [&](auto act) {
    constexpr int ACT = decltype(act)::value;
#pragma unroll
    for (int bm = 0; bm < TM; ++bm)
#pragma unroll
      for (int bn = 0; bn < COLUMNS / 32; ++bn)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          typedef __attribute__((__vector_size__(4 * sizeof(Out)))) Out Out4;
          Out4 v;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            if constexpr (SECOND) v[i] = acc[bn][bm][4 * q + i];
            else if constexpr (GATED) v[i] = from_float<T>(weight[bm] * gated_unit_as<ACT>(c.limit, c.alpha, acc[0][bm][4 * q + i], acc[1][bm][4 * q + i]));
            else v[i] = from_float<T>(weight[bm] * plain_unit_as<ACT>(acc[bn][bm][4 * q + i]));
          }
          *reinterpret_cast<Out4*>(scratch + (bm * 32 + l32) * PITCH + (bn * 32 + q * 8 + g * 4) * (int)sizeof(Out)) = v;
        }
  };
  // (one choice for all values: with the choice at every value all units' code lay between each two of them)
  if constexpr (SECOND) {
    units(Constant<0>());
  } else if constexpr (GATED) {
    if (c.act == 1) units(Constant<1>());
    else units(Constant<0>());
  } else {
    if (c.act == 4) units(Constant<4>());
    else if (c.act == 2) units(Constant<2>());
    else units(Constant<3>());
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");       // (a wave's accesses of LDS are served in order)
  const int n = n_base + wn * COLUMNS + lane % LANES * PIECE;
  constexpr int TURNS = BM / 2 * LANES / 64;
  int row[TURNS];
#pragma unroll
  for (int t = 0; t < TURNS; ++t) {
    const int m = tile.first + wm * (BM / 2) + (64 / LANES) * t + lane / LANES;
    row[t] = m < tile.count ? (SECOND ? entry(m) : m) : -1;
  }
#pragma unroll
  for (int t = 0; t < TURNS; ++t) {
    const int4v v = *reinterpret_cast<const int4v*>(scratch + ((64 / LANES) * t + lane / LANES) * PITCH + lane % LANES * 16);
    if (row[t] < 0 || n >= n_end) continue;
    Out* out;
    if constexpr (SECOND)
      out = c.out + (shared ? c.top : row[t] >> GROUP_PLACE_BITS) * c.plane + (int64_t)(row[t] & ((1 << GROUP_PLACE_BITS) - 1)) * c.ld_out;
    else
      out = shared ? static_cast<T*>(c.shared_hidden) + (int64_t)row[t] * ff : static_cast<T*>(c.hidden) + (int64_t)(tile.slot + row[t]) * ff;
    *reinterpret_cast<int4v*>(out + n) = v;
  }
}

template <typename T, int BM, int STAGES, bool SECOND, bool GATED>
static int launch_expert_products(hipStream_t s, const ExpertProductsCall& c) {
  auto kernel = expert_products_kernel<T, BM, STAGES, SECOND, GATED>;
  // (a wave leaves BM / 2 rows of its half of the columns there in the end, 16 bytes between them)
  const size_t stages = (size_t)STAGES * (BM + 128) * TILE_ROW_BYTES, rows = (size_t)2 * BM * ((SECOND ? 256 : 64 * sizeof(T)) + 16);
  const size_t lds = stages > rows ? stages : rows;
  static bool raised = false;
  if (!raised) {
    hipError_t err = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err != hipSuccess) BT_REFUSE("expert_products: cannot get %zu bytes of LDS: %s", lds, hipGetErrorString(err));
    raised = true;
  }
  const int held = !SECOND && GATED ? 64 : 128;
  const int64_t columns = ((SECOND ? c.width : c.ff) + held - 1) / held;
  const int64_t shared_columns = c.shared_ff == 0 ? 0 : SECOND ? columns : (c.shared_ff + held - 1) / held;
  const int64_t most = ((int64_t)c.tokens * c.top / BM + c.experts) * columns + (int64_t)((c.tokens + BM - 1) / BM) * shared_columns;
  if (most > 0x7fffffff) BT_REFUSE("expert_products: %lld tiles are too many", (long long)most);
  hipLaunchKernelGGL(kernel, dim3((unsigned)most), dim3(256), lds, s, c);
  return bt_check_launch("expert_products");
}

template <typename T, int BM, int STAGES>
static int launch_expert_form(hipStream_t s, const ExpertProductsCall& c) {
  if (c.second) return launch_expert_products<T, BM, STAGES, true, false>(s, c);
  return c.act < 2 ? launch_expert_products<T, BM, STAGES, false, true>(s, c) : launch_expert_products<T, BM, STAGES, false, false>(s, c);
}

BT_EXPORT int bt_expert_products_call(void* stream, const ExpertProductsCall* c) {
  if (c->tokens <= 0) return BT_OK;
  const int row_k = c->dtype == 0 ? 32 : 64, elems = c->dtype == 0 ? 4 : 8;
  if (c->dtype != 0 && c->dtype != 1) BT_REFUSE("expert_products: element type %d is neither float nor bfloat16", c->dtype);
  if (c->experts <= 0 || c->experts > GROUP_MAX_EXPERTS || c->identity < 0 || c->top <= 0 || c->ff <= 0 || c->shared_ff < 0 || c->act < 0 || c->act > 4)
    BT_REFUSE("expert_products: %d experts (1..%d) of %d, %d a token, activation %d", c->experts, GROUP_MAX_EXPERTS, c->ff, c->top, c->act);
  if (c->width % row_k || c->ff % row_k || c->shared_ff % row_k)
    BT_REFUSE("expert_products: width %d and experts of %d and %d must be multiples of %d", c->width, c->ff, c->shared_ff, row_k);
  const int64_t inner = (int64_t)c->experts * c->ff + c->shared_ff;
  if (c->ld_w % elems || c->ldh % elems || c->ld_out % 4 || c->plane % 4 || c->ld_w < (c->second ? inner : c->width) || c->ldh < c->width || c->ld_out < c->width ||
      c->pitch < c->tokens || c->tokens >= 1 << GROUP_PLACE_BITS)
    BT_REFUSE("expert_products: rows too short or not of whole 16 bytes");
  if (!c->rows || !c->counts || !c->h || !c->w || !c->weights || !c->hidden || (c->shared_ff && !c->shared_hidden) || (c->second && !c->out) ||
      (((uintptr_t)c->h | (uintptr_t)c->w | (uintptr_t)c->hidden | (uintptr_t)c->shared_hidden | (uintptr_t)c->out) & 15))
    BT_REFUSE("expert_products: missing operand, or one that is not aligned to 16 bytes");
  hipStream_t s = (hipStream_t)stream;
  if (c->dtype == 0) return launch_expert_form<float, 64, 3>(s, *c);
  return (int64_t)c->tokens * c->top >= (int64_t)EXPERT_TALL_ROWS * c->experts ? launch_expert_form<bf16_t, 128, 2>(s, *c)
                                                                              : launch_expert_form<bf16_t, 64, 3>(s, *c);
}

// hidden[t][e * ff + i] *= the token's weight of expert e, for `experts` experts side by side, from the router's logits of
// the token; columns behind them (an expert every token uses) stay.  A work-group makes the token's whole choice (of up to
// 64 experts every wave for itself, by ranks in lanes; of more its first wave, a few reductions over the experts) and multiplies its share of the columns.
struct WeighExpertsCall {
  RouteCall route;          // dtype: element type of `hidden`; tokens, experts, top, groups, keep, correction, score, group_rank,
                            // normalize, bias; nothing else is looked at
  int ff;
  const float* logits;      // [tokens][ld_logits]
  int64_t ld_logits;
  void* hidden;             // [tokens][ld_hidden]
  int64_t ld_hidden;
};

template <typename T>
__global__ void __launch_bounds__(256) weigh_experts_kernel(WeighExpertsCall w) {
  __shared__ float score[ROUTE_MAX_EXPERTS], choice[ROUTE_MAX_EXPERTS];
  constexpr int PER = 16 / sizeof(T);
  const RouteCall& c = w.route;
  const int t = blockIdx.x, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  T* hidden = static_cast<T*>(w.hidden) + (int64_t)t * w.ld_hidden;
  const int columns = c.experts * w.ff;
  const int pieces = (columns + PER - 1) / PER;
  // (16 bytes at a time where no piece lies in two experts)
  const bool whole = w.ff % PER == 0 && (w.ld_hidden % PER) == 0 && ((uintptr_t)w.hidden & 15) == 0;
  int piece = blockIdx.y * blockDim.x + threadIdx.x;
  int4v held = {0, 0, 0, 0};
  if (whole && piece < pieces) held = *reinterpret_cast<const int4v*>(hidden + (int64_t)piece * PER);      // on its way during the choice
  int expert = min(piece, pieces - 1) * PER / w.ff;   // (the division, too)
  const float* logits = w.logits + (int64_t)t * w.ld_logits;
  RouteEarly early;
  early.load(c);
  const float* weights = choice;
  if (c.experts <= 64) {                           // (every wave for itself: none waits for another)
    float* own = choice + 64 * wave;
    const float weight = route_lanes(c, early, lane < c.experts ? logits[lane] : 0.f, own);
    if (lane < c.experts) own[lane] = weight;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    weights = own;
  } else {
    if (wave == 0) {
      for (int e = lane; e < c.experts; e += 64) score[e] = logits[e];
      route_choice(c, early, score, choice);
    }
    __syncthreads();
  }
  if (!whole) {
    for (int col = piece; col < columns; col += gridDim.y * blockDim.x) {
      const float f = weights[col / w.ff];
      hidden[col] = from_float<T>(f != 0.f ? f * to_float(hidden[col]) : 0.f);
    }
    return;
  }
  for (; piece < pieces; piece += gridDim.y * blockDim.x) {
    const float f = weights[expert];
    T* values = reinterpret_cast<T*>(&held);
#pragma unroll
    for (int i = 0; i < PER; ++i) values[i] = from_float<T>(f != 0.f ? f * to_float(values[i]) : 0.f);
    *reinterpret_cast<int4v*>(hidden + (int64_t)piece * PER) = held;
    const int next = piece + gridDim.y * blockDim.x;
    if (next < pieces) {
      held = *reinterpret_cast<const int4v*>(hidden + (int64_t)next * PER);
      expert = next * PER / w.ff;
    }
  }
}

BT_EXPORT int bt_weigh_experts_call(void* stream, const WeighExpertsCall* w) {
  const RouteCall* c = &w->route;
  if (c->tokens <= 0) return BT_OK;
  if (const char* wrong = route_refusal(c))
    BT_REFUSE("weigh_experts: %d of %d experts a token, %d of %d groups, score %d: %s", c->top, c->experts, c->keep, c->groups, c->score, wrong);
  if (w->ff <= 0 || w->ld_logits < c->experts || w->ld_hidden < (int64_t)c->experts * w->ff || (int64_t)c->experts * w->ff > 0x7fffffff)
    BT_REFUSE("weigh_experts: the rows do not hold %d experts of %d", c->experts, w->ff);
  if (!w->logits || !w->hidden) BT_REFUSE("weigh_experts: missing operand");
  const int per = c->dtype == 0 ? 4 : 8;
  int per_token = (c->experts * w->ff + 256 * per - 1) / (256 * per);
  if (per_token > 64) per_token = 64;
  dim3 grid(c->tokens, per_token), block(256);
  if (c->dtype == 0)
    hipLaunchKernelGGL(weigh_experts_kernel<float>, grid, block, 0, (hipStream_t)stream, *w);
  else
    hipLaunchKernelGGL(weigh_experts_kernel<bf16_t>, grid, block, 0, (hipStream_t)stream, *w);
  return bt_check_launch("weigh_experts");
}
