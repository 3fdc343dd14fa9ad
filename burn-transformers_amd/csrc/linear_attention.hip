// Kernels of mixers that are linear attention with a matrix state per head (no softmax, no cache of
// keys): per head a state S [dim][vdim] in 32-bit that every token first lets decay per key channel
// and then writes a rank-one update into, token after token.
//   * keyed scan: per token and head, with a decay g [dim], a key k [dim], a value v [vdim], a query q [dim]:
//         S <- diag(g) S;   u = v                              (plain write)
//                           u = beta (v - S^T k)               (delta rule: what S already answers for k is taken off)
//         S <- S + k u^T;   o = S^T q                          (the read-out sees the token's own write)
//     How g, k and q come about is the kernel's `form`:
//       form 0 (gated delta rule): q and k are rows of their own (heads may share them), optionally made unit
//           vectors per head here, x / sqrt(sum x^2 + unit_eps), q times q_scale; g = exp(-exp(A_log[head]) * dt)
//           from step sizes dt per head and key channel, or one per head for all its key channels (`decay_span` 1);
//           with `dt_bias` the step sizes come raw and dt = softplus(raw + dt_bias); beta = sigmoid(beta logit of the head)
//       form 1 (forget gate that also decides what is written): f = lower + (1 - lower) * sigmoid(f_raw + f_bias)
//           per head and key channel; g = f, k = 1 - f, q = silu(q_raw); no beta
//   * head norm with a gate: every head's read-out over its root mean square over vdim, times a scale of
//     vdim entries that the heads share, times the sigmoid of a gate's logits where there are any
// A sequence's state lives in its slot's row of the cache's per-sequence state area; a step may bring any
// number of a sequence's tokens, which are walked in order from the state the last step left.
#include "host.h"
#include "scan.h"

struct KeyedScanCall {
  int tokens, n_seqs;
  int heads;              // heads of v, g, beta and of the state
  int kv_heads;           // heads of q and k (form 0); head h uses h / (heads / kv_heads)
  int dim, vdim;
  int form;               // 0: delta rule; 1: forget gate with complement keys
  int unit;               // form 0: 1 if q and k are made unit vectors per head here
  float unit_eps;
  float q_scale;          // form 0: factor on q (after the unit norm)
  const float* q;         // [tokens][ld_q]: form 0: head j at columns j * dim; form 1: raw, head h at h * dim
  int64_t ld_q;
  const float* k;         // [tokens][ld_k] (form 0)
  int64_t ld_k;
  const float* v;         // [tokens][ld_v]: head h at columns h * vdim
  int64_t ld_v;
  const float* g;         // [tokens][ld_g]: head h at columns h * dim: step sizes (form 0), gate logits (form 1);
  int64_t ld_g;           // with decay_span 1 head h at column h

  const float* beta;      // [tokens][ld_beta]: one logit a head (form 0)
  int64_t ld_beta;
  const float* A_log;     // [heads] (form 0)
  const float* g_bias;    // [heads * dim] (form 1), or null
  const float* lower;     // [heads * dim] (form 1)
  float* out;             // [tokens][ld_out] float32: head h at columns h * vdim
  int64_t ld_out;
  float* S;               // slot s: [heads][vdim / 4 rounded up][dim][4] at S + s * state_stride
  int64_t state_stride;
  const int* seq_off;     // [n_seqs + 1]
  const int* slots;       // [n_seqs]
  // form 1 only: long sequences are cut into spans of at least `span` tokens that are scanned side by side (see
  // "Spans" in scan.h; the forget gate's step is a diagonal decay and a write, which is linear in S; the delta
  // rule's is not diagonal and walks its sequences in order).  0: never; max_count is the most tokens a sequence
  // of the step brings, carry the room for the spans' states: (tokens / span + 2 n_seqs + 1) blocks of a slot's
  // state and heads * dim products of decays
  int span;
  int max_count;
  float* carry;
  int decay_span;         // form 0: 0 a step size per head and key channel, 1 one per head
  const float* dt_bias;   // form 0: null, or [heads * dim] ([heads] with decay_span 1): g holds raw sums, dt = softplus(g + dt_bias)
  // null, or room for what blocks of 16 tokens leave: (tokens / 16 + n_seqs + 1) * heads * (16 (3 dim + vdim) + dim) floats,
  // aligned to 16 bytes; with it long sequences go in blocks on the matrix units (max_count as above)
  float* blocks;
};

// One wave per (4 value channels of a head, sequence): sixteen lanes share a channel, each owns R key channels
// of its column of S in registers.  A work-group is four waves with four channels each of the same head: they
// share the run of decays, queries and keys in LDS.
// A run is up to 2048 / NP tokens (NP = 16 R key channels, padded), so that a thread stages KS_LOADS entries
// of it: every load of a run is issued before the first is used (a loop of single loads is waited for once
// per trip), and the NEXT run's loads are issued before this run's tokens are walked, so memory's latency
// hides behind the recurrence.
#define KS_WAVES 4
#define KS_THREADS (64 * KS_WAVES)
#define KS_LOADS 8

template <int R>
struct KsRun {
  static constexpr int NP = 16 * R;
  static constexpr int V = R < 4 ? R : 4;                          // floats a lane reads at a time
  static constexpr int MOST = 2048 / NP > 64 ? 64 : 2048 / NP;     // tokens of a run
  static constexpr int TOK_LOADS = (MOST * 4 + 63) / 64;           // (v, beta) pairs a lane stages
};

// Decays, queries and keys of a run lie in LDS as planes of [tokens][NP] floats (the forget gate's keys are
// 1 - decay and have no plane: every wave reads a token's whole row of every plane, and with several waves to a
// SIMD those reads are what bounds a token's time).  Lane j of the sixteen that share a value channel owns the
// key channels j + 16 r, r < R (so the lanes' loads of a register's worth of state are neighbours in memory); in
// a plane's row channel j + 16 r lies at (16 (r / V) + j) V + r % V, so that a lane reads V neighbouring floats
// at a time and neighbouring lanes read neighbouring vectors.
template <int R, int V>
__device__ __forceinline__ int ks_place(int sub, int r) { return (16 * (r / V) + sub) * V + r % V; }

template <int R, int V>
__device__ __forceinline__ void ks_read(const float* row, int sub, float* out) {
#pragma unroll
  for (int i = 0; i < R / V; ++i) {
    const float* at = row + (16 * i + sub) * V;
    if (V == 4) {
      const float4 x = *reinterpret_cast<const float4*>(at);
      out[4 * i] = x.x; out[4 * i + 1] = x.y; out[4 * i + 2] = x.z; out[4 * i + 3] = x.w;
    } else if (V == 2) {
      const float2 x = *reinterpret_cast<const float2*>(at);
      out[2 * i] = x.x; out[2 * i + 1] = x.y;
    } else {
      out[i] = at[0];
    }
  }
}

// phase 0: whole sequences, from and to the slot's state.  1: spans from zero, leaving their end states and the
// products of their decays, no read-outs.  3: spans from the carried states, writing read-outs, leaving no state.
template <int R, int FORM, int PHASE>
__global__ void __launch_bounds__(KS_THREADS) keyed_scan_kernel(KeyedScanCall c, int chunk, int tiles) {
  constexpr int phase = PHASE;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  constexpr int NP = KsRun<R>::NP, V = KsRun<R>::V, TOK_LOADS = KsRun<R>::TOK_LOADS;
  constexpr int ROWS_A_TURN = KS_THREADS / NP;                                // tokens that the threads' entries of one turn span
  constexpr int PLANES = FORM == 0 ? 3 : 2;
  float* G = lds;                                                             // [chunk][NP] decays
  float* Q = lds + (size_t)chunk * NP;                                        // [chunk][NP] queries
  float* Kp = lds + (size_t)2 * chunk * NP;                                   // [chunk][NP] keys (delta rule)
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, sub = lane & 15, pl = lane >> 4;
  float2* tok = reinterpret_cast<float2*>(lds + (size_t)PLANES * chunk * NP) + (size_t)wave * chunk * 4;   // [waves][chunk][4]: v, beta
  // one decay a head: a run's decays are worked out once a token (thread i takes token i), not once a key channel
  float* dec = lds + (size_t)PLANES * chunk * NP + (size_t)KS_WAVES * chunk * 8;                          // [chunk]
  const bool per_head = FORM == 0 && c.decay_span == 1;
  const int tile = min((int)blockIdx.x * KS_WAVES + wave, tiles - 1), head = blockIdx.y;
  const int seq = blockIdx.z % c.n_seqs, part = blockIdx.z / c.n_seqs;
  const bool works = (int)blockIdx.x * KS_WAVES + wave < tiles;
  const int p = tile * 4 + pl;
  const bool live = works && p < c.vdim;
  const int shared = FORM == 0 ? head / (c.heads / c.kv_heads) : head;
  int first = c.seq_off[seq], last = c.seq_off[seq + 1];
  const int64_t in_slot = ((int64_t)head * tiles + tile) * c.dim * 4 + pl;        // where this lane's column of S starts
  float* held = c.S + (int64_t)c.slots[seq] * c.state_stride + in_slot;
  float* products = nullptr;                              // phase 1: where this span's products of decays go
  if (phase) {
    first += part * c.span;
    if (first >= last) return;                            // (the whole work-group: no barrier has been met)
    last = min(first + c.span, last);
    const int64_t state_floats = (int64_t)c.heads * tiles * c.dim * 4, per_span = state_floats + (int64_t)c.heads * c.dim;
    float* mine = c.carry + span_block(c.seq_off, seq, c.span, part) * per_span;
    held = (phase == 1 ? mine : mine - per_span) + in_slot;
    products = mine + state_floats + (int64_t)head * c.dim;
  }
  float S[R], P[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int n = sub + 16 * r;
    S[r] = n < c.dim && phase != 1 ? held[(int64_t)n * 4] : 0.f;
    P[r] = 1.0f;
  }
  const float rate = FORM == 0 ? -expf(c.A_log[head]) : 0.f;
  float* ocol = c.out + head * c.vdim + (live ? p : 0);
  // a thread's entries of a run are key channel `n` of the tokens row0, row0 + ROWS_A_TURN, ...
  const int n = threadIdx.x % NP, row0 = threadIdx.x / NP;
  const int place = ks_place<R, V>(n % 16, n / 16);       // where channel n lies in a plane's row
  const bool in_head = n < c.dim;
  const int nc = in_head ? n : 0;
  const int col_g = FORM == 0 && c.decay_span == 1 ? head : head * c.dim + nc, col_k = shared * c.dim + nc;
  float low = 0.f, bias = 0.f;
  if (FORM == 1) {
    low = c.lower[col_g];
    bias = c.g_bias ? c.g_bias[col_g] : 0.f;
  }
  const bool raw_steps = FORM == 0 && c.dt_bias != nullptr;
  if (raw_steps) bias = c.dt_bias[col_g];
  const int ch = tile * 4 + (lane & 3);                   // the value channel of a lane's (v, beta) pairs
  const int chc = ch < c.vdim ? ch : 0;
  float rg[KS_LOADS], rk[KS_LOADS], rq[KS_LOADS], rv[TOK_LOADS], rb[TOK_LOADS], rh = 0.f;
  // issues the loads of the run that starts at token t0 (rows beyond the run read its last token and are dropped)
  auto fetch = [&](int t0, int count) {
#pragma unroll
    for (int j = 0; j < KS_LOADS; ++j) {
      const int i = min(row0 + j * ROWS_A_TURN, count - 1);
      const int64_t t = t0 + i;
      rg[j] = per_head ? 0.f : c.g[t * c.ld_g + col_g];
      rq[j] = PHASE == 1 ? 0.f : c.q[t * c.ld_q + (FORM == 0 ? col_k : col_g)];
      rk[j] = FORM == 0 ? c.k[t * c.ld_k + col_k] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < TOK_LOADS; ++j) {
      const int i = min((lane >> 2) + 16 * j, count - 1);
      const int64_t t = t0 + i;
      rv[j] = c.v[t * c.ld_v + head * c.vdim + chc];
      rb[j] = FORM == 0 ? c.beta[t * c.ld_beta + head] : 0.f;
    }
    if (per_head) rh = c.g[(int64_t)(t0 + min((int)threadIdx.x, count - 1)) * c.ld_g + head];
  };
  if (first < last) fetch(first, min(chunk, last - first));
  for (int t0 = first; t0 < last; t0 += chunk) {
    const int count = min(chunk, last - t0);
    __syncthreads();                                       // the run before has been walked
    if (per_head) {
      if ((int)threadIdx.x < count) dec[threadIdx.x] = expf(rate * (raw_steps ? softplus_f(rh + bias) : rh));
      __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < KS_LOADS; ++j) {
      const int i = row0 + j * ROWS_A_TURN;
      if (i < count) {
        float decay = 0.f, query = 0.f;
        if (in_head) {
          if (FORM == 0) {
            decay = per_head ? dec[i] : expf(rate * (raw_steps ? softplus_f(rg[j] + bias) : rg[j]));
            query = rq[j];
          } else {
            decay = low + (1.0f - low) / (1.0f + expf(-(rg[j] + bias)));
            query = PHASE == 1 ? 0.f : silu_f(rq[j]);
          }
        }
        G[i * NP + place] = decay;
        if (PHASE != 1) Q[i * NP + place] = query;
        if (FORM == 0) Kp[i * NP + place] = in_head ? rk[j] : 0.f;
      }
    }
#pragma unroll
    for (int j = 0; j < TOK_LOADS; ++j) {
      const int i = (lane >> 2) + 16 * j;
      if (i < count)
        tok[i * 4 + (lane & 3)] = make_float2(ch < c.vdim ? rv[j] : 0.f, FORM == 0 ? 1.0f / (1.0f + expf(-rb[j])) : 1.0f);
    }
    __syncthreads();
    if (t0 + chunk < last) fetch(t0 + chunk, min(chunk, last - t0 - chunk));      // in flight while this run is walked
    if (FORM == 0 && c.unit) {          // q and k as unit vectors: sixteen lanes take a token
      for (int i = threadIdx.x >> 4; i < count; i += 4 * KS_WAVES) {
        float kk[R], qq[R], sk = 0.f, sq = 0.f;
        ks_read<R, V>(Kp + i * NP, sub, kk);
        ks_read<R, V>(Q + i * NP, sub, qq);
#pragma unroll
        for (int r = 0; r < R; ++r) {
          sk = fmaf(kk[r], kk[r], sk);
          sq = fmaf(qq[r], qq[r], sq);
        }
        const float rk_ = 1.0f / sqrtf(sum_of_16_lanes(sk) + c.unit_eps);
        const float rq_ = c.q_scale / sqrtf(sum_of_16_lanes(sq) + c.unit_eps);
#pragma unroll
        for (int r = 0; r < R; ++r) {
          Kp[i * NP + ks_place<R, V>(sub, r)] = kk[r] * rk_;
          Q[i * NP + ks_place<R, V>(sub, r)] = qq[r] * rq_;
        }
      }
      __syncthreads();
    }
    if (!works) continue;
    // a token's inputs are read from LDS while the token before it is worked on: a wave is alone on its SIMD,
    // so nothing else hides that latency
    float g[R], k[R], q[R];
    float2 vb = tok[pl];
    ks_read<R, V>(G, sub, g);
    if (PHASE != 1) ks_read<R, V>(Q, sub, q);
    if (FORM == 0) ks_read<R, V>(Kp, sub, k);
#pragma unroll 4
    for (int i = 0; i < count; ++i) {
      const int ahead = min(i + 1, count - 1);
      float g_next[R], k_next[R], q_next[R];
      const float2 vb_next = tok[ahead * 4 + pl];
      ks_read<R, V>(G + ahead * NP, sub, g_next);
      if (PHASE != 1) ks_read<R, V>(Q + ahead * NP, sub, q_next);
      if (FORM == 0) ks_read<R, V>(Kp + ahead * NP, sub, k_next);
      float u = vb.x;
      if (FORM == 0) {
        float answered = 0.f, answered_odd = 0.f;          // (two sums: half as long a chain of dependent adds)
#pragma unroll
        for (int r = 0; r < R; ++r) {
          S[r] *= g[r];
          if (r & 1) answered_odd = fmaf(S[r], k[r], answered_odd);
          else answered = fmaf(S[r], k[r], answered);
        }
        u = vb.y * (vb.x - sum_of_16_lanes(answered + answered_odd));
      } else {
#pragma unroll
        for (int r = 0; r < R; ++r) {
          k[r] = 1.0f - g[r];
          S[r] *= g[r];
          if (PHASE == 1) P[r] *= g[r];
        }
      }
      if (PHASE == 1) {                                     // a span from zero leaves its state only: no read-out
#pragma unroll
        for (int r = 0; r < R; ++r) S[r] = fmaf(k[r], u, S[r]);
      } else {
        float acc = 0.f, acc_odd = 0.f;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          S[r] = fmaf(k[r], u, S[r]);
          if (r & 1) acc_odd = fmaf(S[r], q[r], acc_odd);
          else acc = fmaf(S[r], q[r], acc);
        }
        const float o = sum_of_16_lanes(acc + acc_odd);
        if (live && sub == 0) ocol[(int64_t)(t0 + i) * c.ld_out] = o;
      }
      vb = vb_next;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        g[r] = g_next[r];
        if (PHASE != 1) q[r] = q_next[r];
        if (FORM == 0) k[r] = k_next[r];
      }
    }
  }
  if (!works || phase == 3) return;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int nn = sub + 16 * r;
    if (nn < c.dim) held[(int64_t)nn * 4] = S[r];
    if (nn < c.dim && phase == 1 && blockIdx.x == 0 && wave == 0 && pl == 0) products[nn] = P[r];
  }
}

// C_k = P_k C_(k-1) + E_k along every sequence, in place; C_(-1), the state the sequence came with, is kept in
// front of its spans, and the last C goes into the slot.
__global__ void __launch_bounds__(256) keyed_carry_kernel(KeyedScanCall c, int tiles) {
  const int seq = blockIdx.y;
  const int64_t index = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, size = (int64_t)c.heads * tiles * c.dim * 4;
  if (index >= size) return;
  const int count = c.seq_off[seq + 1] - c.seq_off[seq];
  const int spans = (count + c.span - 1) / c.span;
  const int64_t per_span = size + (int64_t)c.heads * c.dim;
  float* block = c.carry + span_block(c.seq_off, seq, c.span, 0) * per_span;
  float* slot = c.S + (int64_t)c.slots[seq] * c.state_stride;
  float state = slot[index];
  (block - per_span)[index] = state;
  const int64_t decay = size + (index / ((int64_t)4 * c.dim * tiles)) * c.dim + (index / 4) % c.dim;
  for (int k = 0; k < spans; ++k, block += per_span) {
    state = block[decay] * state + block[index];
    block[index] = state;
  }
  slot[index] = state;
}

// Into spans of how many tokens the forget gate's long sequences are cut, 0 for not at all.
static int keyed_span(const KeyedScanCall& c) {
  const int tiles = (c.vdim + 3) / 4, groups = (tiles + KS_WAVES - 1) / KS_WAVES;
  const int span = c.form == 1 ? span_tokens(c.span, c.max_count, c.carry, (int64_t)groups * KS_WAVES * c.heads * c.n_seqs, 1) : 0;
  return span > 0 && (int64_t)c.n_seqs * ((c.max_count + span - 1) / span) <= 65535 ? span : 0;
}

template <int R>
static void launch_keyed_scan(hipStream_t stream, const KeyedScanCall& c) {
  const int per_token = (c.form == 0 ? 3 : 2) * 16 * R + 8 * KS_WAVES + 1;      // planes, (v, beta) pairs, a decay
  const int tiles = (c.vdim + 3) / 4, groups = (tiles + KS_WAVES - 1) / KS_WAVES;
  dim3 block(KS_THREADS);
  const int span = keyed_span(c);
  if (span > 0) {
    KeyedScanCall cut = c;
    cut.span = span;
    const int chunk = span < KsRun<R>::MOST ? span : KsRun<R>::MOST;
    const int spans = (c.max_count + span - 1) / span;
    dim3 grid(groups, c.heads, c.n_seqs * spans);
    const size_t lds = (size_t)chunk * per_token * sizeof(float);
    const int64_t state_floats = (int64_t)c.heads * tiles * c.dim * 4;
    hipLaunchKernelGGL((keyed_scan_kernel<R, 1, 1>), grid, block, lds, stream, cut, chunk, tiles);
    hipLaunchKernelGGL(keyed_carry_kernel, dim3((unsigned)((state_floats + 255) / 256), c.n_seqs), dim3(256), 0, stream, cut, tiles);
    hipLaunchKernelGGL((keyed_scan_kernel<R, 1, 3>), grid, block, lds, stream, cut, chunk, tiles);
    return;
  }
  const int chunk = c.tokens < KsRun<R>::MOST ? c.tokens : KsRun<R>::MOST;
  dim3 grid(groups, c.heads, c.n_seqs);
  const size_t lds = (size_t)chunk * per_token * sizeof(float);
  if (c.form == 0)
    hipLaunchKernelGGL((keyed_scan_kernel<R, 0, 0>), grid, block, lds, stream, c, chunk, tiles);
  else
    hipLaunchKernelGGL((keyed_scan_kernel<R, 1, 0>), grid, block, lds, stream, c, chunk, tiles);
}

// --- blocks of sixteen tokens on the matrix units ----------------------------------------------
//
// A token of the walk above costs 0.25 to 0.5 us (delta rule) however idle the chip is.  What a block of B = 16 tokens does to the
// state can be written down before the state is known.  With a_t the product of the block's decays up to and with
// token t (per key channel), b_s that of the decays behind token s, kd = a k, qd = a q, ku = b k:
//     A[t][s] = beta_t sum_d k_t k_s g_(s+1) .. g_t   (s < t),   P[t][s] the same with q_t, without beta, and s <= t
//     T = (I + A)^-1 diag(beta),  M = P T
//     u = T v - (T kd) S0,   o = M v + (qd - M kd) S0,   S = diag(a_B) S0 + ku^T u
// so W = T kd, R = qd - M kd, T v and M v are left by one kernel, all blocks side by side, and a second one walks
// the blocks in order with the state in registers: two products with S0 and one into it a block, on
// v_mfma_f32_16x16x4_f32 (32-bit multiply and add throughout).  Decays are only ever multiplied with each other, never
// divided and never taken to logarithms, so a decay of nearly nothing is as exact as in the walk.  The forget gate
// writes plain values: T v is v and W is not there.
//
// Operands lie in the workspace as the lanes of a wave want them (a lane's four values of a 16 x 16 tile side by side,
// lanes one after the other).  Of an instruction's four K values step i takes number 4 g + i in lane group g = lane / 16:
// the registers in which a product's result lands are then the B operand of the next one, and nothing moves between
// lanes.  Measured, token by token / in blocks (us; 8 heads of 128 x 128, 2 x 1,024 tokens): delta rule with one decay
// a head 386 / 78, one a key channel 522 / 82, forget gate (there in spans) 139 / 57; 2 x 128 tokens 52 / 24, 69 / 26,
// 45 / 18.  The operands take 25 us (18 without T) of the long ones; the walk takes 0.87 us a block (0.63), of which the
// matrix units are busy for 0.32 (0.21).  Since then (see KB_AHEAD) the walk takes 0.66 us a block (0.45), and 2 x 1,024 tokens 65 us (46).
#define KB_TOKENS 16

// Floats of one block and head: W, R and ku [tiles of 16 channels][64 lanes][4], T v [tiles of 16 values][64][4], a_B [dim].
__host__ __device__ __forceinline__ int64_t kb_floats(int dim, int vdim) { return (int64_t)KB_TOKENS * (3 * dim + vdim) + dim; }

// Where block `block` of sequence `seq` and a head keeps them: ranges of different sequences do not meet.
__device__ __forceinline__ float* kb_place(const KeyedScanCall& c, int seq, int block, int head) {
  return c.blocks + ((int64_t)(c.seq_off[seq] / KB_TOKENS + seq + block) * c.heads + head) * kb_floats(c.dim, c.vdim);
}

template <int FORM, int DT>
__global__ void __launch_bounds__(256, 4) keyed_blocks_kernel(KeyedScanCall c) {
  constexpr int DIM = 16 * DT, PITCH = DIM + 4;
  __shared__ __attribute__((aligned(16))) float K[KB_TOKENS][PITCH], Q[KB_TOKENS][PITCH], G[KB_TOKENS][PITCH];
  __shared__ __attribute__((aligned(16))) float A[KB_TOKENS][KB_TOKENS], P[KB_TOKENS][KB_TOKENS], T[KB_TOKENS][20], M[KB_TOKENS][20];
  __shared__ float strength[KB_TOKENS], one[KB_TOKENS];                  // beta, and a decay the whole head shares
  const int head = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int part;
  const int seq = piece_sequence(c.seq_off, c.n_seqs, c.tokens, c.max_count, KB_TOKENS, blockIdx.y, part);
  if (seq < 0) return;                                                   // (the whole work-group)
  const int first = c.seq_off[seq] + part * KB_TOKENS;
  const int count = min(KB_TOKENS, c.seq_off[seq + 1] - first);
  const int shared = FORM == 0 ? head / (c.heads / c.kv_heads) : head;
  float* place = kb_place(c, seq, part, head);
  const float rate = FORM == 0 ? -expf(c.A_log[head]) : 0.f;
  const bool per_head = FORM == 0 && c.decay_span == 1;
  if (FORM == 0 && tid < KB_TOKENS) {
    const int64_t t = first + min(tid, count - 1);
    strength[tid] = tid < count ? 1.0f / (1.0f + expf(-c.beta[t * c.ld_beta + head])) : 0.f;
    if (per_head) {
      const float raw = c.g[t * c.ld_g + head];
      one[tid] = expf(rate * (c.dt_bias ? softplus_f(raw + c.dt_bias[head]) : raw));
    }
  }
  if (per_head) __syncthreads();
  // rows behind the sequence's end decay by one and hold zeros: they change nothing
#pragma unroll
  for (int j = 0; j < DT; ++j) {
    const int i = (tid + 256 * j) / DIM, d = (tid + 256 * j) % DIM;
    const int64_t t = first + min(i, count - 1);
    const float raw = per_head ? 0.f : c.g[t * c.ld_g + head * DIM + d];
    float q = c.q[t * c.ld_q + shared * DIM + d], k, decay;
    if (FORM == 0) {
      k = c.k[t * c.ld_k + shared * DIM + d];
      decay = per_head ? one[i] : expf(rate * (c.dt_bias ? softplus_f(raw + c.dt_bias[head * DIM + d]) : raw));
    } else {
      const float low = c.lower[head * DIM + d];
      decay = low + (1.0f - low) / (1.0f + expf(-(raw + (c.g_bias ? c.g_bias[head * DIM + d] : 0.f))));
      k = 1.0f - decay;
      q = silu_f(q);
    }
    const bool there = i < count;
    K[i][d] = there ? k : 0.f;
    Q[i][d] = there ? q : 0.f;
    G[i][d] = there ? decay : 1.f;
  }
  __syncthreads();
  const int sub = tid & 15, s = tid >> 4;
  if (FORM == 0 && c.unit) {                                             // sixteen lanes make a token's vectors unit vectors
    float sk = 0.f, sq = 0.f;
#pragma unroll
    for (int r = 0; r < DT; ++r) {
      sk = fmaf(K[s][sub + 16 * r], K[s][sub + 16 * r], sk);
      sq = fmaf(Q[s][sub + 16 * r], Q[s][sub + 16 * r], sq);
    }
    sk = 1.0f / sqrtf(sum_of_16_lanes(sk) + c.unit_eps);
    sq = c.q_scale / sqrtf(sum_of_16_lanes(sq) + c.unit_eps);
#pragma unroll
    for (int r = 0; r < DT; ++r) {
      K[s][sub + 16 * r] *= sk;
      Q[s][sub + 16 * r] *= sq;
    }
    __syncthreads();
  }
  // pairs: sixteen lanes carry token s's key through the decays behind it and meet every later key and query; a lane
  // owns channels 4 sub .. 4 sub + 3 of every 64, so that a row is read 16 bytes at a time
  {
    constexpr int R = (DT + 3) / 4;
    floatx4 w[R];
    auto row = [&](const float* at, int r) {
      const int d = 64 * r + 4 * sub;
      return DT % 4 == 0 || d < DIM ? *reinterpret_cast<const floatx4*>(at + d) : floatx4{0.f, 0.f, 0.f, 0.f};
    };
#pragma unroll
    for (int r = 0; r < R; ++r) w[r] = row(K[s], r);
    const int begin = __builtin_amdgcn_readfirstlane(tid >> 6) * 4;      // the first s of the wave
#pragma unroll 2
    for (int t = begin; t < KB_TOKENS; ++t) {
      floatx4 ak = {0.f, 0.f, 0.f, 0.f}, aq = ak;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const floatx4 g = row(G[t], r), q = row(Q[t], r);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          w[r][i] = t > s ? w[r][i] * g[i] : w[r][i];
          aq[i] = fmaf(w[r][i], q[i], aq[i]);
        }
        if (FORM == 0) {
          const floatx4 k = row(K[t], r);
#pragma unroll
          for (int i = 0; i < 4; ++i) ak[i] = fmaf(w[r][i], k[i], ak[i]);
        }
      }
      const float pair_q = sum_of_16_lanes((aq[0] + aq[1]) + (aq[2] + aq[3]));
      if (FORM == 0) {
        const float pair_k = sum_of_16_lanes((ak[0] + ak[1]) + (ak[2] + ak[3]));
        if (sub == 0) {
          P[t][s] = t >= s ? pair_q : 0.f;
          A[t][s] = t > s ? strength[t] * pair_k : 0.f;
        }
      } else if (sub == 0) {
        M[t][s] = t >= s ? pair_q : 0.f;
      }
    }
    if (FORM == 1 && sub == 0)
      for (int t = 0; t < begin; ++t) M[t][s] = 0.f;
  }
  __syncthreads();
  if (FORM == 0 && wave == 0) {                                          // T, a column a lane (four lanes share one), and M
    float col[KB_TOKENS];
#pragma unroll
    for (int t = 0; t < KB_TOKENS; ++t) {
      floatx4 v = {t == sub ? 1.f : 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int e = 0; e < t; ++e) v[e & 3] = fmaf(-A[t][e], col[e], v[e & 3]);
      col[t] = (v[0] + v[1]) + (v[2] + v[3]);
    }
#pragma unroll
    for (int t = 0; t < KB_TOKENS; ++t) col[t] = t >= sub ? col[t] * strength[sub] : 0.f;
#pragma unroll
    for (int t = 0; t < KB_TOKENS; ++t)
      if ((lane >> 4) == (t & 3)) T[t][sub] = col[t];
#pragma unroll
    for (int i = 0; i < 4; ++i) {                                        // rows 4 i + g; P holds nothing behind the diagonal
      const int t = 4 * i + (lane >> 4);
      float m = 0.f;
#pragma unroll
      for (int e = 0; e < 4 * i + 4; ++e) m = e <= t ? fmaf(P[t][e], col[e], m) : m;
      M[t][sub] = m;
    }
  }
  if (wave >= 2) {                                                       // k -> kd, q -> qd, decays -> ku, a channel a thread
    const int d = tid - 128;
    if (d < DIM) {
      float k[KB_TOKENS], g[KB_TOKENS], run = 1.f;
#pragma unroll
      for (int t = 0; t < KB_TOKENS; ++t) {
        k[t] = K[t][d];
        g[t] = G[t][d];
        run *= g[t];
        K[t][d] = k[t] * run;
        Q[t][d] *= run;
      }
      place[KB_TOKENS * (3 * DIM + c.vdim) + d] = run;
      run = 1.f;
#pragma unroll
      for (int t = KB_TOKENS - 1; t >= 0; --t) {
        G[t][d] = k[t] * run;
        run *= g[t];
      }
    }
  }
  __syncthreads();
  const int g = lane >> 4, n = lane & 15;
  floatx4 tb, mb = *reinterpret_cast<const floatx4*>(&M[n][4 * g]);
  if (FORM == 0) tb = *reinterpret_cast<const floatx4*>(&T[n][4 * g]);
  floatx4* frag = reinterpret_cast<floatx4*>(place);
  // T and M hold zeros for the tokens behind a row's own, and the products take them: a value there that is not finite
  // would make this row's not a number.  Where a result is not finite it is summed again, over the row's own tokens only.
  auto finite = [](floatx4 v) { return fabsf((v[0] + v[1]) + (v[2] + v[3])) < INFINITY; };
  auto own = [](const float* row, int t, auto value) {
    float sum = 0.f;
#pragma unroll 1
    for (int s = 0; s <= t; ++s) sum = fmaf(row[s], value(s), sum);
    return sum;
  };
  for (int tile = wave; tile < DT; tile += 4) {
    const int d = 16 * tile + n;
    floatx4 r = *reinterpret_cast<const floatx4*>(&Q[n][16 * tile + 4 * g]), u;
    if (FORM == 0) {
      floatx4 w = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float kd = K[4 * g + i][d];
        w = __builtin_amdgcn_mfma_f32_16x16x4f32(kd, tb[i], w, 0, 0, 0);
        r = __builtin_amdgcn_mfma_f32_16x16x4f32(kd, -mb[i], r, 0, 0, 0);
      }
      if (__builtin_expect(!(finite(w) && finite(r)), 0))
        for (int i = 0; i < 4; ++i) {
          const int from = 16 * tile + 4 * g + i;
          auto kd = [&](int s) { return K[s][from]; };
          w[i] = own(T[n], n, kd);
          r[i] = Q[n][from] - own(M[n], n, kd);
        }
      frag[64 * tile + lane] = w;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) u[i] = G[4 * g + i][d];
    frag[64 * (DT + tile) + lane] = r;
    frag[64 * (2 * DT + tile) + lane] = u;
  }
  const float* v_rows = c.v + (int64_t)first * c.ld_v + head * c.vdim;
  float* out = c.out + (int64_t)first * c.ld_out + head * c.vdim;
  for (int tile = wave; 16 * tile < c.vdim; tile += 4) {
    floatx4 v, u = {0.f, 0.f, 0.f, 0.f}, o = u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float value = v_rows[(int64_t)min(4 * g + i, count - 1) * c.ld_v + 16 * tile + n];
      v[i] = 4 * g + i < count ? value : 0.f;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (FORM == 0) u = __builtin_amdgcn_mfma_f32_16x16x4f32(tb[i], v[i], u, 0, 0, 0);
      o = __builtin_amdgcn_mfma_f32_16x16x4f32(mb[i], v[i], o, 0, 0, 0);
    }
    if (__builtin_expect(!(finite(o) && (FORM == 1 || finite(u))), 0))
      for (int i = 0; i < 4; ++i) {
        const int t = min(4 * g + i, count - 1);                         // (rows behind the sequence's end are not used)
        auto value = [&](int s) { return v_rows[(int64_t)s * c.ld_v + 16 * tile + n]; };
        if (FORM == 0) u[i] = own(T[t], t, value);
        o[i] = own(M[t], t, value);
      }
    frag[64 * (3 * DT + tile) + lane] = FORM == 0 ? u : v;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (4 * g + i < count) out[(int64_t)(4 * g + i) * c.ld_out + 16 * tile + n] = o[i];
  }
}

// One work-group per 16 value channels of a head and sequence: four waves share the key channels (TW tiles of 16 each),
// every wave's part of W S0 and R S0 meets in LDS.  The operands of the next KB_AHEAD - 1 blocks are on their way.
// What bounds a block is one wave's chain on each SIMD: 24 matrix instructions (16 without W) of 32 cycles, the exchange, and the address unit,
// which four waves' loads take 450 cycles (so: no load of what another wave has, a decay a lane and not four of which a quad's lanes all have
// the same; a load behind each matrix instruction, the exchange while R S0 runs).  How far ahead they are asked for makes no difference (2, 4
// and 6 blocks alike).  The loop takes whole turns of KB_AHEAD and the rest stands behind it: with a way out between two blocks the
// compiler's waits in front of a turn are those of every way into it, and all loads are waited for.  Measured (us, 8 heads of 128 x 128, 2 x
// 1,024 tokens, the walk alone): delta rule 56.9 -> 42.1, forget gate 40 -> 28.7.
#define KB_AHEAD 4

template <int FORM, int TW>
struct KbStage {
  floatx4 w[FORM == 0 ? TW : 1], r[TW], ku[TW];
  float a[TW], o;
  typename std::conditional<FORM == 0, float, floatx4>::type u;   // of T v the wave's quarter, or all of v
};

// Spans of blocks (the forget gate).  A walk of few columns leaves compute units idle and the others with one wave to a SIMD, whose
// chain from block to block is what the time is.  Its step is linear in S, so long sequences are cut into spans of c.span
// tokens ("Spans" in scan.h): keyed_spans_kernel leaves the state behind every span but a sequence's last, the first one's from the
// slot's state and the others' from zero, and their products of decays; the walk then takes every span side by side, from
// the state that those add up to.  A span from zero is one product a block (u is v), without barriers.
// Measured with the blocks' operands (us, whole sequences / in spans; 8 heads of 128 x 128): 2 x 1,024 tokens 45.5 / 45.1, 2,048 67.8 / 43.6,
// 1,000 37.6 / 30.5, 640 28.2 / 26.4; 16 heads, 2,000 tokens 75.9 / 65.4; 8 heads of 64 x 64, 2,048 42.8 / 25.7.
__device__ __forceinline__ int64_t kb_span_floats(const KeyedScanCall& c) { return (int64_t)c.heads * c.dim * c.vdim + (int64_t)c.heads * c.dim; }

// The operands of a wave's TW tiles of key channels of a block that the state's update takes.
template <int TW>
struct KbUpdate {
  floatx4 ku[TW], u;
  float a[TW];
};

// Four channels' rows of S times their decays, of which a quad's four lanes hold one each.
__device__ __forceinline__ void decay(floatx4& s, float a) {
  s[0] *= dpp_move<0x00>(a);
  s[1] *= dpp_move<0x55>(a);
  s[2] *= dpp_move<0xAA>(a);
  s[3] *= dpp_move<0xFF>(a);
}

template <int DT>
__global__ void __launch_bounds__(256, 2) keyed_spans_kernel(KeyedScanCall c) {
  constexpr int TW = (DT + 3) / 4, DIM = 16 * DT;
  const int columns = c.vdim / 16, pair = blockIdx.x / (8 * columns) * 8 + blockIdx.x % 8;
  const int column = blockIdx.x / 8 % columns, head = pair % c.heads;
  int part;
  const int seq = piece_sequence(c.seq_off, c.n_seqs, c.tokens, c.max_count, c.span, pair / c.heads, part);
  if (seq < 0 || (part + 1) * c.span >= c.seq_off[seq + 1] - c.seq_off[seq]) return;   // nothing stands behind a sequence's last span
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, n = lane & 15;
  const int blocks = c.span / KB_TOKENS, vtiles = c.vdim / 4, p = 16 * column + n;
  const int64_t stride = (int64_t)c.heads * kb_floats(DIM, c.vdim) * 4, of_head = ((int64_t)head * vtiles + p / 4) * DIM * 4 + p % 4;
  const char* at = reinterpret_cast<const char*>(kb_place(c, seq, part * blocks, head));
  float* const end = c.carry + span_block(c.seq_off, seq, c.span, part) * kb_span_floats(c);
  uint32_t from_tile[TW], from_decay[TW];
#pragma unroll
  for (int j = 0; j < TW; ++j) {
    const int tile = min(wave * TW + j, DT - 1);
    from_tile[j] = (KB_TOKENS * 2 * DIM + 256 * tile + 4 * lane) * 4;
    from_decay[j] = (KB_TOKENS * (3 * DIM + c.vdim) + 16 * tile + 4 * g + (n & 3)) * 4;
  }
  uint32_t from_u = (KB_TOKENS * 3 * DIM + 256 * column + 4 * lane) * 4;
  KbUpdate<TW> stages[KB_AHEAD];
  int fetched = 0;
  auto load = [&](uint32_t& from) {                        // (as in the walk)
    asm volatile("" : "+v"(from));
    return (const __attribute__((address_space(1))) char*)at + from;
  };
  auto fetch = [&](KbUpdate<TW>& st) {
#pragma unroll
    for (int j = 0; j < TW; ++j) {
      st.ku[j] = *reinterpret_cast<const __attribute__((address_space(1))) floatx4*>(load(from_tile[j]));
      st.a[j] = *reinterpret_cast<const __attribute__((address_space(1))) float*>(load(from_decay[j]));
    }
    st.u = *reinterpret_cast<const __attribute__((address_space(1))) floatx4*>(load(from_u));
    at += ++fetched < blocks ? stride : 0;                 // (at the end the last block's again, not used)
  };
  auto mine = [&](int j) { return DT % 4 == 0 || wave * TW + j < DT; };
  floatx4 S[TW];
  float P[TW];                                             // of channel 4 g + n % 4
#pragma unroll
  for (int i = 0; i < KB_AHEAD - 1; ++i) {
    fetch(stages[i]);
    __builtin_amdgcn_sched_barrier(0);
  }
  auto row = [&](int j, int i) { return of_head + (int64_t)(16 * (wave * TW + j) + 4 * g + i) * 4; };
#pragma unroll
  for (int j = 0; j < TW; ++j) {
    P[j] = 1.f;
    S[j] = floatx4{0.f, 0.f, 0.f, 0.f};
  }
  if (part == 0) {                                         // the slot's state, kept for the walk (whose last span writes the slot)
    const float* slot = c.S + (int64_t)c.slots[seq] * c.state_stride;
    float* const kept = end - kb_span_floats(c);
#pragma unroll
    for (int j = 0; j < TW; ++j)
      if (mine(j))
#pragma unroll
        for (int i = 0; i < 4; ++i) S[j][i] = slot[row(j, i)];
#pragma unroll
    for (int j = 0; j < TW; ++j)
      if (mine(j))
#pragma unroll
        for (int i = 0; i < 4; ++i) kept[row(j, i)] = S[j][i];
  }
  landed(S);
  auto step = [&](const KbUpdate<TW>& st) {
#pragma unroll
    for (int j = 0; j < TW; ++j) {
      decay(S[j], st.a[j]);
      P[j] *= st.a[j];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < TW; ++j)
        if (mine(j)) S[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(st.ku[j][i], st.u[i], S[j], 0, 0, 0);
  };
  int block = 0;
  for (; block + KB_AHEAD <= blocks; block += KB_AHEAD) {
#pragma unroll
    for (int i = 0; i < KB_AHEAD; ++i) {
      fetch(stages[(i + KB_AHEAD - 1) % KB_AHEAD]);
      __builtin_amdgcn_sched_barrier(0);
      step(stages[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < KB_AHEAD - 1; ++i)
    if (block + i < blocks) step(stages[i]);
#pragma unroll
  for (int j = 0; j < TW; ++j)
    if (mine(j))
#pragma unroll
      for (int i = 0; i < 4; ++i) end[row(j, i)] = S[j][i];
  if (column == 0 && n < 4) {
#pragma unroll
    for (int j = 0; j < TW; ++j)
      if (mine(j)) end[(int64_t)c.heads * DIM * c.vdim + head * DIM + 16 * (wave * TW + j) + 4 * g + n] = P[j];
  }
}

// SPANS: c.span tokens of a sequence a work-group, behind keyed_spans_kernel; otherwise whole sequences.
template <int FORM, int DT, bool SPANS>
__global__ void __launch_bounds__(256, 2) keyed_blocks_walk_kernel(KeyedScanCall c) {
  constexpr int TW = (DT + 3) / 4, DIM = 16 * DT;
  __shared__ __attribute__((aligned(16))) floatx4 parts[2][2][4][64];   // [turn][W S0, R S0][wave][lane]
  // the columns of a head and sequence read the same operands: they are numbered onto one XCD (work-groups are dealt to
  // eight of them in turn), which reads them from memory once
  const int columns = c.vdim / 16, pair = blockIdx.x / (8 * columns) * 8 + blockIdx.x % 8;
  const int column = blockIdx.x / 8 % columns, head = pair % c.heads;
  int seq = pair / c.heads, part = 0;
  if constexpr (SPANS) seq = piece_sequence(c.seq_off, c.n_seqs, c.tokens, c.max_count, c.span, seq, part);
  else if (seq >= c.n_seqs) return;
  if (SPANS && seq < 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, n = lane & 15;
  int first = c.seq_off[seq], count = c.seq_off[seq + 1] - first;
  if (count <= 0) return;
  const bool cut = SPANS && count > c.span, last = !cut || (part + 1) * c.span >= count;
  if constexpr (SPANS) {
    first += part * c.span;
    count = last ? count - part * c.span : c.span;
  }
  const int blocks = (count + KB_TOKENS - 1) / KB_TOKENS;
  const int64_t stride = (int64_t)c.heads * kb_floats(DIM, c.vdim);
  const float* place = kb_place(c, seq, SPANS ? part * (c.span / KB_TOKENS) : 0, head);
  const int vtiles = (c.vdim + 3) / 4, p = 16 * column + n;
  const int64_t of_head = ((int64_t)head * vtiles + p / 4) * DIM * 4 + p % 4;
  float* slot = c.S + (int64_t)c.slots[seq] * c.state_stride + of_head;
  // tiles of key channels are dealt in turn; a wave has all its TW tiles unless DT is no multiple of four
  auto mine = [&](int j) { return DT % 4 == 0 || wave * TW + j < DT; };
  floatx4 S[TW];
  auto read = [&](const float* from, floatx4 (&to)[TW], int apart) {
#pragma unroll
    for (int j = 0; j < TW; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) to[j][i] = mine(j) ? from[(int64_t)(16 * (wave * TW + j) + 4 * g + i) * apart] : 0.f;
  };
  KbStage<FORM, TW> stages[KB_AHEAD];
  // a block's operands: one address that all lanes share, and every lane's distances from it
  uint32_t from_tile[TW], from_decay[TW];
#pragma unroll
  for (int j = 0; j < TW; ++j) {
    const int tile = min(wave * TW + j, DT - 1);
    from_tile[j] = (256 * tile + 4 * lane) * 4;
    from_decay[j] = (KB_TOKENS * (3 * DIM + c.vdim) + 16 * tile + 4 * g + (n & 3)) * 4;
  }
  uint32_t from_u = (KB_TOKENS * 3 * DIM + 256 * column + 4 * lane + (FORM == 0 ? wave : 0)) * 4;
  uint32_t from_o = (uint32_t)((4 * g + wave) * c.ld_out + n) * 4;
  const uint32_t from_last = (uint32_t)(min(4 * g + wave, count - (blocks - 1) * KB_TOKENS - 1) * c.ld_out + n) * 4;
  const char* at = reinterpret_cast<const char*>(place);
  float* const outs = c.out + (int64_t)first * c.ld_out + head * c.vdim + 16 * column;
  const char* out_at = reinterpret_cast<const char*>(outs);
  int row = 4 * g + wave, fetched = 0;                     // a wave finishes every fourth token's read-out
  float* out = outs + (int64_t)min(row, count - 1) * c.ld_out + n;
  const int64_t out_step = KB_TOKENS * c.ld_out;
  // (a distance is taken as a new number each time: widened once for all it would be added to the address in 64 bits at every load)
  auto load4 = [&](uint32_t& from, int further) {
    const char* base = at + further;
    asm volatile("" : "+v"(from), "+s"(base));
    return *reinterpret_cast<const __attribute__((address_space(1))) floatx4*>((const __attribute__((address_space(1))) char*)base + from);
  };
  auto load1 = [&](const char* base, uint32_t& from) {
    asm volatile("" : "+v"(from));
    return *reinterpret_cast<const float*>(base + from);
  };
  constexpr int LOADS = (FORM == 0 ? 4 : 3) * TW + 2;
  auto fetch = [&](KbStage<FORM, TW>& st, auto number) {   // one of a block's LOADS, in order
    constexpr int load = decltype(number)::value, j = load % TW, kind = load / TW + (FORM == 0 ? 0 : 1);
    if constexpr (load >= LOADS) {
      return;
    } else if constexpr (load == LOADS - 1) {
      if (fetched >= blocks - 1) from_o = from_last;
      st.o = load1(out_at, from_o);
      // on to the next block; at the end the last one's operands are asked for again and not used
      const bool more = ++fetched < blocks;
      at += more ? stride * 4 : 0;
      out_at += more ? out_step * 4 : 0;
    } else if constexpr (load == LOADS - 2) {
      if constexpr (FORM == 0) st.u = load1(at, from_u);
      else st.u = load4(from_u, 0);
    } else if constexpr (kind == 0) {
      st.w[j] = load4(from_tile[j], 0);
    } else if constexpr (kind == 1) {
      st.r[j] = load4(from_tile[j], KB_TOKENS * DIM * 4);
    } else if constexpr (kind == 2) {
      st.ku[j] = load4(from_tile[j], 2 * KB_TOKENS * DIM * 4);
    } else {
      st.a[j] = load1(at, from_decay[j]);
    }
  };
  // A block's read-out is added up from LDS behind the next block's barrier.
  float pending = 0.f;
  auto finish = [&](const float (&r)[4]) {
    const float o = pending + ((r[0] + r[1]) + (r[2] + r[3]));
    if (row < count) *out = o;
    row += KB_TOKENS;
    out += out_step;
  };
  auto read_outs = [&](int turn, float (&r)[4]) {
    const float* at = reinterpret_cast<const float*>(&parts[turn][1][0][lane]) + wave;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = at[256 * i];
  };
  auto walk = [&](KbStage<FORM, TW>& st, int turn, bool behind, auto asks, KbStage<FORM, TW>& next) {
    floatx4 ws[TW], rs[TW];
#pragma unroll
    for (int j = 0; j < TW; ++j) ws[j] = rs[j] = floatx4{0.f, 0.f, 0.f, 0.f};
    if constexpr (FORM == 0) {                             // a quarter of T v is in every wave's part
#pragma unroll
      for (int i = 0; i < 4; ++i) ws[0][i] = i == wave ? -st.u : 0.f;
    }
    // The products with S0, a load of the next block's operands behind each: one of 16 bytes a lane takes the address unit, which the
    // four waves share, 16 cycles, and a wave that asks for all its ten at once waits for them.
    auto ask = [&](auto number) {
      if constexpr (decltype(asks)::value) fetch(next, number);
      __builtin_amdgcn_sched_barrier(0);
    };
    auto step = [&](floatx4 (&sum)[TW], const floatx4* op, auto number) {
      constexpr int j = decltype(number)::value % TW, i = decltype(number)::value / TW;
      if (mine(j)) sum[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(op[j][i], S[j][i], sum[j], 0, 0, 0);
    };
    constexpr int FIRST = FORM == 0 ? 4 * TW : 0;          // loads behind W's steps
    if constexpr (FORM == 0) {
      each<4 * TW>([&](auto x) { step(ws, st.w, x); ask(x); });
      if (TW > 1) ws[0] += ws[TW - 1];
      parts[turn][0][wave][lane] = ws[0];
      __builtin_amdgcn_sched_barrier(0);
    }
    each<2 * TW>([&](auto x) { step(rs, st.r, x); ask(Number<FIRST + decltype(x)::value>()); });
    lds_barrier();
    floatx4 others[4];
    float r[4];
    if (FORM == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) others[i] = parts[turn][0][i][lane];
    }
    read_outs(turn ^ 1, r);
    __builtin_amdgcn_sched_barrier(0);
    each<2 * TW>([&](auto x) { step(rs, st.r, Number<2 * TW + decltype(x)::value>()); ask(Number<FIRST + 2 * TW + decltype(x)::value>()); });
    ask(Number<FIRST + 4 * TW>());
    static_assert(FIRST + 4 * TW + 1 >= LOADS, "every load has its place");
    floatx4 u;
    if constexpr (FORM == 0) u = -((others[0] + others[1]) + (others[2] + others[3]));
    else u = st.u;
#pragma unroll
    for (int j = 0; j < TW; ++j) decay(S[j], st.a[j]);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < TW; ++j)
        if (mine(j)) S[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(st.ku[j][i], u[i], S[j], 0, 0, 0);
    if (behind) finish(r);
    if (TW > 1) rs[0] += rs[TW - 1];
    parts[turn][1][wave][lane] = rs[0];
    pending = st.o;
  };
#pragma unroll
  for (int i = 0; i < KB_AHEAD - 1; ++i) {
    each<LOADS>([&](auto load) { fetch(stages[i], load); });
    __builtin_amdgcn_sched_barrier(0);                     // (in order: a stage is waited for by the loads behind it)
  }
  if (!cut) {
    read(slot, S, 4);
  } else {                                                 // C(-1), or C(0) carried on: C(k) = P(k) C(k - 1) + E(k)
    const int64_t span = kb_span_floats(c), products = (int64_t)c.heads * DIM * c.vdim + head * DIM;
    const float* held = c.carry + span_block(c.seq_off, seq, c.span, part == 0 ? -1 : 0) * span;
    read(held + of_head, S, 4);
    if (part > 1) {
      floatx4 E[TW], P[TW], E_next[TW], P_next[TW];
      held += span;
      read(held + of_head, E, 4);
      read(held + products, P, 1);
      for (int k = 1; k < part; ++k) {
        if (k + 1 < part) held += span;                    // (the last one's again, not used)
        read(held + of_head, E_next, 4);
        read(held + products, P_next, 1);
#pragma unroll
        for (int j = 0; j < TW; ++j) {
          S[j] = P[j] * S[j] + E[j];
          E[j] = E_next[j];
          P[j] = P_next[j];
        }
      }
    }
  }
  landed(S);
  int block = 0;
  for (; block + KB_AHEAD <= blocks; block += KB_AHEAD) {  // (whole turns: see KB_AHEAD)
#pragma unroll
    for (int i = 0; i < KB_AHEAD; ++i) {
      walk(stages[i], i & 1, block + i > 0, Number<1>(), stages[(i + KB_AHEAD - 1) % KB_AHEAD]);
    }
  }
#pragma unroll
  for (int i = 0; i < KB_AHEAD - 1; ++i)
    if (block + i < blocks) walk(stages[i], i & 1, block + i > 0, Number<0>(), stages[i]);  // (the same for all four waves)
  lds_barrier();
  float r[4];
  read_outs((blocks - 1) & 1, r);
  finish(r);
  if (!last) return;
#pragma unroll
  for (int j = 0; j < TW; ++j)
    if (mine(j))
#pragma unroll
      for (int i = 0; i < 4; ++i) slot[(int64_t)(16 * (wave * TW + j) + 4 * g + i) * 4] = S[j][i];
}

// Steps whose longest sequence brings at least this many tokens may go in blocks (blocks_pay).  Below, two launches cost what walking
// does (us, token by token / in blocks; one decay a head, one a key channel, forget gate): 2 x 32 tokens 16.0 / 17.2,
// 19.9 / 19.5, 13.8 / 13.0; 16 x 40 tokens 42.8 / 37.0, 56.3 / 39.3, 32.8 / 28.4; 4 x 48 tokens 22.9 / 19.6, 29.2 / 22.1, 20.0 / 15.0.
#define KB_MIN_TOKENS 40

// From there on the cheaper way is taken, by what was measured of both (us; a state of R tiles of 16 key channels): token by token a
// launch and a token's chain for every token of the longest sequence, in spans the chain of one span twice and a step of the
// carry for every span; in blocks two launches and a block's chain, and for every sequence that is short beside the longest one
// the work-groups that bring its state in and out (they hold a compute unit's registers, two to a unit).  Measured (start
// to end, token by token or in spans / in blocks): forget gate, 2 heads of 16 x 16, 4,000 tokens 36 / 90, 4 of 64 x 64 68 / 106, 8 of 128 x 128
// 246 / 167; delta rule with one decay a head, 8 heads of 128 x 128, 40 tokens and 63 single ones 33 / 54, 100 and 63 46 / 55, 500 and 63
// 192 / 61, 1,000 and 200 375 / 149; 16 heads, 64 and 31 36 / 55; 2 heads of 16 x 16, 40 tokens 11 / 15.  With the walk as it is
// now the forget gate in blocks, 4 heads of 64 x 64, 1,000 tokens 33 / 25; 2 of 16 x 16, 4,000 35 / 82.  (Of blocks that would be cut into spans the
// time of whole sequences is weighed, which is more than they take: small states with long sequences stay token by token in spans, 4 heads of 64 x
// 64, 4,000 tokens 64, where the blocks were not measured in spans.)
static bool blocks_pay(const KeyedScanCall& c) {
  const float r = c.dim / 16, longest = c.max_count;
  const int span = keyed_span(c);
  const float token = c.form == 1 ? 0.11f + 0.0275f * r : c.decay_span == 1 ? 0.17f + 0.026f * r : 0.165f + 0.043f * r;
  const float start = c.form == 1 ? 3.5f : 3.f + 0.4f * r;
  const float walk = span == 0 ? start + token * longest
                               : 2.f + 2.f * token * span * span_crowding((int64_t)c.heads * (c.vdim / 4), c.tokens, span) +
                                     (0.3f + 2e-5f * c.heads * c.dim * c.vdim) * (longest / span);
  const float others = short_sequences(c.tokens, c.n_seqs, c.max_count) * (c.heads * (c.vdim / 16)) * (0.003f + 4e-5f * c.dim);
  const float blocks = (c.form == 1 ? 8.f + 0.6f * r + (0.0165f + 0.0011f * r) * longest : 13.f + 0.5f * r + (0.028f + 0.0033f * r) * longest) + others;
  return blocks < walk;
}

// Into spans of how many tokens the walk over blocks cuts the forget gate's sequences, 0 for not at all: as many as give every compute
// unit the two work-groups it holds, where that makes at least three of the longest sequence.  Below 640 tokens the second kernel costs
// what it gains, below 832 where several sequences give half the units and more a work-group (us, whole / in spans, 8 heads of 128 x 128: 256
// tokens 19.1 / 18.5, 640 27.8 / 26.0, 1,000 37.6 / 30.5; 2 x 300 22.6 / 26.4, 2 x 512 31.9 / 33.2, 2 x 640 33.5 / 34.9, 2 x 768 36.7 / 37.3, 2 x 896 40.7 /
// 40.0, 2 x 1,536 59.5 / 53.4; 4 heads 4 x 640 33.2 / 35.4, 4 x 1,024 44.0 / 43.0; 16 heads 640 32.6 / 32.7, 1,000 43.0 / 39.9; 12 heads 2 x 800 40.5 / 40.3).
#define KB_UNITS 256
#define KB_SPAN_MIN 640
#define KB_SPAN_MIN_OF_MANY 832
static int keyed_block_span(const KeyedScanCall& c) {
  if (c.form != 1 || c.span <= 0 || !c.carry) return 0;
  const int64_t per_token = (int64_t)c.heads * (c.vdim / 16);
  if (per_token * c.n_seqs >= 2 * KB_UNITS) return 0;
  int64_t tokens = (c.tokens * per_token + 2 * KB_UNITS - 1) / (2 * KB_UNITS);
  if (tokens < c.span) tokens = c.span;
  tokens = (tokens + KB_TOKENS - 1) / KB_TOKENS * KB_TOKENS;
  const int least = c.n_seqs > 1 && 2 * per_token * c.n_seqs >= KB_UNITS ? KB_SPAN_MIN_OF_MANY : KB_SPAN_MIN;
  return c.max_count >= least && c.max_count >= 3 * tokens ? (int)tokens : 0;
}

template <int DT>
static void launch_keyed_blocks(hipStream_t stream, const KeyedScanCall& c) {
  dim3 side(c.heads, c.tokens / KB_TOKENS + c.n_seqs), block(256);      // (the heads of a piece side by side: they share rows)
  auto walks = [&](int64_t pieces) { return dim3((unsigned)((c.heads * pieces + 7) / 8 * 8 * (c.vdim / 16))); };
  if (c.form == 0) {
    hipLaunchKernelGGL((keyed_blocks_kernel<0, DT>), side, block, 0, stream, c);
    hipLaunchKernelGGL((keyed_blocks_walk_kernel<0, DT, false>), walks(c.n_seqs), block, 0, stream, c);
    return;
  }
  hipLaunchKernelGGL((keyed_blocks_kernel<1, DT>), side, block, 0, stream, c);
  if (const int span = keyed_block_span(c)) {
    KeyedScanCall cut = c;
    cut.span = span;
    const dim3 grid = walks(c.tokens / span + c.n_seqs);
    hipLaunchKernelGGL(keyed_spans_kernel<DT>, grid, block, 0, stream, cut);
    hipLaunchKernelGGL((keyed_blocks_walk_kernel<1, DT, true>), grid, block, 0, stream, cut);
  } else {
    hipLaunchKernelGGL((keyed_blocks_walk_kernel<1, DT, false>), walks(c.n_seqs), block, 0, stream, c);
  }
}

// True if the call went in blocks: it brings the room, tiles of 16 and enough tokens.
static bool keyed_blocks(hipStream_t stream, const KeyedScanCall& c) {
  if (!c.blocks || c.max_count < KB_MIN_TOKENS || c.dim % 16 != 0 || c.dim > 128 || c.vdim % 16 != 0 ||
      c.tokens / KB_TOKENS + c.n_seqs > 65535 || (int64_t)c.heads * c.n_seqs * (c.vdim / 16) > 1 << 30 || !blocks_pay(c))
    return false;
  switch (c.dim / 16) {
    case 1: launch_keyed_blocks<1>(stream, c); break;
    case 2: launch_keyed_blocks<2>(stream, c); break;
    case 3: launch_keyed_blocks<3>(stream, c); break;
    case 4: launch_keyed_blocks<4>(stream, c); break;
    case 5: launch_keyed_blocks<5>(stream, c); break;
    case 6: launch_keyed_blocks<6>(stream, c); break;
    case 7: launch_keyed_blocks<7>(stream, c); break;
    default: launch_keyed_blocks<8>(stream, c); break;
  }
  return true;
}

BT_EXPORT int bt_keyed_scan_call(void* stream, const KeyedScanCall* c) {
  if (c->tokens <= 0 || c->n_seqs <= 0) return BT_OK;
  if (c->heads <= 0 || c->dim <= 0 || c->dim > 256 || c->vdim <= 0)
    BT_REFUSE("keyed_scan: %d heads with keys of %d (1..256) and values of %d", c->heads, c->dim, c->vdim);
  if (c->form != 0 && c->form != 1) BT_REFUSE("keyed_scan: unknown form %d", c->form);
  if (c->form == 0 && (c->kv_heads <= 0 || c->heads % c->kv_heads != 0))
    BT_REFUSE("keyed_scan: %d heads cannot share %d heads of queries and keys", c->heads, c->kv_heads);
  if (!c->q || !c->v || !c->g || !c->out || !c->S || !c->seq_off || !c->slots)
    BT_REFUSE("keyed_scan: missing operand");
  if (c->form == 0 && (!c->k || !c->beta || !c->A_log)) BT_REFUSE("keyed_scan: the delta rule lacks keys, beta or A_log");
  if (c->form == 1 && !c->lower) BT_REFUSE("keyed_scan: the forget gate lacks its lower bound");
  const int64_t qk = (int64_t)(c->form == 0 ? c->kv_heads : c->heads) * c->dim;
  if (c->decay_span != 0 && (c->decay_span != 1 || c->form != 0)) BT_REFUSE("keyed_scan: a decay per head goes with the delta rule");
  if (c->ld_q < qk || (c->form == 0 && c->ld_k < qk) || c->ld_g < (int64_t)c->heads * (c->decay_span == 1 ? 1 : c->dim) ||
      c->ld_v < (int64_t)c->heads * c->vdim || c->ld_out < (int64_t)c->heads * c->vdim ||
      (c->form == 0 && c->ld_beta < c->heads))
    BT_REFUSE("keyed_scan: rows too short for %d heads of %d and %d", c->heads, c->dim, c->vdim);
  if (c->state_stride < (int64_t)c->heads * ((c->vdim + 3) / 4) * c->dim * 4)
    BT_REFUSE("keyed_scan: a slot's state of %lld elements does not hold %d heads of %d x %d", (long long)c->state_stride,
              c->heads, c->dim, c->vdim);
  if (c->heads > 65535 || c->n_seqs > 65535) BT_REFUSE("keyed_scan: %d heads of %d sequences are too many", c->heads, c->n_seqs);
  if ((uintptr_t)c->blocks % 16 != 0) BT_REFUSE("keyed_scan: the room for blocks is not aligned to 16 bytes");
  hipStream_t s = (hipStream_t)stream;
  if (keyed_blocks(s, *c)) return bt_check_launch("keyed_scan");
  const int per = (c->dim + 15) / 16;
  if (per <= 1) launch_keyed_scan<1>(s, *c);
  else if (per <= 2) launch_keyed_scan<2>(s, *c);
  else if (per <= 4) launch_keyed_scan<4>(s, *c);
  else if (per <= 8) launch_keyed_scan<8>(s, *c);
  else launch_keyed_scan<16>(s, *c);
  return bt_check_launch("keyed_scan");
}

// out[t][h * vdim + i] = y / sqrt(mean_i(y^2) + eps) * weight[i] * sigmoid(gate[t][h * vdim + i]), y = the
// head's read-out; without `gate` no last factor.  Columns of `out` behind the heads are set to zero.
struct HeadNormGateCall {
  int out_dtype;          // 0 float32, 1 bfloat16
  int tokens, heads, vdim;
  int out_cols;           // columns of out written: heads * vdim, then zeros
  float eps;
  float mult;             // one more factor on the result
  const float* y;         // [tokens][ld_y]
  int64_t ld_y;
  const float* gate;      // [tokens][ld_gate] logits, or null
  int64_t ld_gate;
  const float* weight;    // [vdim]
  void* out;              // [tokens][ld_out]
  int64_t ld_out;
  int gate_act;           // what the gate's logits z become: 0 sigmoid(z), 1 silu(z) = z sigmoid(z)
};

template <typename T>
__global__ void __launch_bounds__(256) head_norm_gate_kernel(HeadNormGateCall c) {
  const int t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  T* out = static_cast<T*>(c.out) + (int64_t)t * c.ld_out;
  for (int head = blockIdx.y * 4 + wave; head < c.heads; head += gridDim.y * 4) {
    const float* y = c.y + (int64_t)t * c.ld_y + head * c.vdim;
    float squares = 0.f;
    for (int i = lane; i < c.vdim; i += 64) squares = fmaf(y[i], y[i], squares);
    const float scale = c.mult / sqrtf(wave_sum(squares) / (float)c.vdim + c.eps);
    for (int i = lane; i < c.vdim; i += 64) {
      float v = y[i] * scale * c.weight[i];
      if (c.gate) {
        const float z = c.gate[(int64_t)t * c.ld_gate + head * c.vdim + i];
        v *= (c.gate_act == 1 ? z : 1.0f) / (1.0f + expf(-z));
      }
      out[head * c.vdim + i] = from_float<T>(v);
    }
  }
  if (blockIdx.y == 0)
    for (int col = c.heads * c.vdim + threadIdx.x; col < c.out_cols; col += blockDim.x) out[col] = from_float<T>(0.f);
}

BT_EXPORT int bt_head_norm_gate_call(void* stream, const HeadNormGateCall* c) {
  if (c->tokens <= 0) return BT_OK;
  if (c->heads <= 0 || c->vdim <= 0) BT_REFUSE("head_norm_gate: %d heads of %d", c->heads, c->vdim);
  const int64_t columns = (int64_t)c->heads * c->vdim;
  if (!c->y || !c->weight || !c->out || c->ld_y < columns || c->out_cols < columns || c->ld_out < c->out_cols ||
      (c->gate && c->ld_gate < columns))
    BT_REFUSE("head_norm_gate: missing operand or rows too short");
  if (c->gate_act != 0 && c->gate_act != 1) BT_REFUSE("head_norm_gate: unknown activation %d of the gate", c->gate_act);
  int per_token = (c->heads + 3) / 4;
  if (per_token > 64) per_token = 64;
  dim3 grid(c->tokens, per_token), block(256);
  if (c->out_dtype == 0)
    hipLaunchKernelGGL(head_norm_gate_kernel<float>, grid, block, 0, (hipStream_t)stream, *c);
  else
    hipLaunchKernelGGL(head_norm_gate_kernel<bf16_t>, grid, block, 0, (hipStream_t)stream, *c);
  return bt_check_launch("head_norm_gate");
}
