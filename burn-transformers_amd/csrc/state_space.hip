// Kernels of the recurrent (state-space) mixers.  Everything that enters a recurrence is 32-bit:
// step sizes, decays, states, the sums over the state.  A sequence's state lives in its slot's row
// of the cache's per-sequence state area and is carried from step to step; a step may bring any
// number of a sequence's tokens, which are walked in order.
//   * causal convolution per channel with bias and silu; its last taps - 1 inputs are state
//   * dt projection: softplus(W low + b)
//   * selective scan (one state row per channel, one decay per state element), with the output gate
//   * scan with one decay per head and a state of [state, head size] (state-space duality form)
//   * gate, then RMS norm in equal parts
#include <type_traits>

#include "host.h"
#include "scan.h"


// Brings rows t0 .. t0 + count - 1 of B and C (`state` columns each, row pitch `ld`, 32-bit offsets) into LDS
// as pairs, [count][NP] with zeros behind `state`; NP is a power of two.  A pass of the wave covers
// whole rows (64 / NP of them, or 1 / (NP / 64) of one), a lane keeps its column, and thirty-two passes'
// loads are issued before the first is stored: a loop of single loads would wait for memory once per
// element, and one that works its row and column out of a running index spends more instructions on
// that than the recurrence spends on a token.  `lane` numbers the THREADS threads that share the work.
template <int NP, int LOADS, int THREADS>
__device__ __forceinline__ void fill_pairs_ahead(float2* BC, const float* B, const float* C, int ld, int t0, int count,
                                                 int state, int lane) {
  constexpr int ROWS = NP >= THREADS ? 1 : THREADS / NP;     // rows a pass covers
  constexpr int COLS = NP >= THREADS ? NP / THREADS : 1;     // passes a row takes
  constexpr int AHEAD = COLS >= LOADS ? 1 : LOADS / COLS;    // row passes whose loads are in flight together
  const int lane_row = NP >= THREADS ? 0 : lane / NP, lane_col = NP >= THREADS ? lane : lane % NP;
  for (int r0 = 0; r0 < count; r0 += ROWS * AHEAD) {
    float2 got[AHEAD][COLS];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      const int row = r0 + u * ROWS + lane_row;
      const int at = (t0 + min(row, count - 1)) * ld;
#pragma unroll
      for (int k = 0; k < COLS; ++k) {
        const int n = lane_col + THREADS * k;
        got[u][k] = (row < count && n < state) ? make_float2(B[at + n], C[at + n]) : make_float2(0.f, 0.f);
      }
    }
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      const int row = r0 + u * ROWS + lane_row;
#pragma unroll
      for (int k = 0; k < COLS; ++k)
        if (row < count) BC[row * NP + lane_col + THREADS * k] = got[u][k];
    }
  }
}

// (a step of single tokens has one row to bring: the short form spares it the long one's idle passes)
template <int NP, int THREADS>
__device__ __forceinline__ void fill_pairs(float2* BC, const float* B, const float* C, int ld, int t0, int count,
                                           int state, int lane) {
  constexpr int ROWS = NP >= THREADS ? 1 : THREADS / NP;
  if (count <= 2 * ROWS)
    fill_pairs_ahead<NP, 2, THREADS>(BC, B, C, ld, t0, count, state, lane);
  else
    fill_pairs_ahead<NP, 2048 / THREADS, THREADS>(BC, B, C, ld, t0, count, state, lane);
}

// ---------------------------------------------------------------------------------------------
struct CausalConvCall {
  int cast_dtype;         // element type of `cast`
  int tokens, n_seqs, channels, taps;
  int cast_cols;          // columns of `cast` written: the channels, then zeros
  const float* in;        // [tokens][ld_in]
  int64_t ld_in;
  const float* weight;    // [channels][taps]; the last tap meets the current token
  const float* bias;      // [channels], or null: none
  float* out;             // [tokens][ld_out] float32
  int64_t ld_out;
  void* cast;             // [tokens][ld_cast] the same in the products' type, or null
  int64_t ld_cast;
  float* state;           // slot s: [taps - 1][channels] at state + s * state_stride, oldest first
  int64_t state_stride;
  const int* tok_seq;
  const int* seq_off;     // [n_seqs + 1]
  const int* slots;       // [n_seqs]
  int act;                // what follows the sum: 0 silu, 1 nothing
};

// SHIFT: every sequence of the step brings one token (a decode step), so a (sequence, channel) pair
// belongs to one thread, which can also move the state on: no second kernel.
template <typename T, bool SHIFT>
__global__ void __launch_bounds__(256) causal_conv_kernel(CausalConvCall c) {
  const int t = blockIdx.x;
  const int ch = blockIdx.y * blockDim.x + threadIdx.x;
  T* cast = static_cast<T*>(c.cast);
  if (ch >= c.channels) {
    if (cast && ch < c.cast_cols) cast[(int64_t)t * c.ld_cast + ch] = from_float<T>(0.f);
    return;
  }
  const int seq = c.tok_seq[t];
  const int local = t - c.seq_off[seq];
  float* held = c.state + (int64_t)c.slots[seq] * c.state_stride;
  float sum = c.bias ? c.bias[ch] : 0.f;
  for (int j = 0; j < c.taps; ++j) {
    const int back = c.taps - 1 - j;
    const int src = local - back;
    const float u = src >= 0 ? c.in[(int64_t)(t - back) * c.ld_in + ch]
                             : held[(int64_t)(c.taps - 1 + src) * c.channels + ch];
    sum = fmaf(c.weight[(int64_t)ch * c.taps + j], u, sum);
  }
  const float y = c.act == 0 ? silu_f(sum) : sum;
  c.out[(int64_t)t * c.ld_out + ch] = y;
  if (cast) cast[(int64_t)t * c.ld_cast + ch] = from_float<T>(y);
  if (SHIFT) {
    for (int r = 0; r + 2 < c.taps; ++r) held[(int64_t)r * c.channels + ch] = held[(int64_t)(r + 1) * c.channels + ch];
    if (c.taps > 1) held[(int64_t)(c.taps - 2) * c.channels + ch] = c.in[(int64_t)t * c.ld_in + ch];
  }
}

// The same for steps of many tokens: a thread takes a channel of CONV_RUN tokens one after the other, so that an input is read
// once and not once a tap, the taps stay in registers and all of a run's inputs are on their way together; a run that
// begins a sequence takes its window's front from the state, one that straddles two reads the tables for every token.  Sums are
// taken in the same order as above.  Measured with the state's kernel (us, a token a thread / in runs; channels of 4 taps): 2,048 tokens of 2,048
// 28.4 / 12.4 (the bytes: 6.9), 2 x 256 of 2,048 9.3 / 5.9, 16 x 40 11.2 / 6.8, 3 x 100 of 1,536 6.6 / 7.4; runs of 16 17.2.  A run that
// straddles has one trip to memory more, which few values do not hide: 500 and 63 x 1 tokens of 300 channels 6.7 / 7.6, of 2,048 11.3 / 9.2,
// 100 x 16 of 300 7.9 / 7.6 (token after token within the run 9.4, 10.9, 8.0).
#define CONV_RUN 8
#define CONV_MIN_TOKENS 384
#define CONV_MIN_VALUES 350000
// ... and where several sequences may straddle runs, of which few taps gain less (300 and 100 x 1 tokens: of 1,024 channels 2 taps 5.6 / 6.4, 3 6.1 /
// 6.8, 4 6.8 / 7.3, of 2,048 2 taps 6.9 / 7.3, 4 9.6 / 8.8; 120 x 5 of 900 2 taps 6.2 / 6.9, 4 8.6 / 8.2).
#define CONV_MIN_VALUES_MANY 500000
#define CONV_MIN_VALUES_MANY_FEW_TAPS 1000000

template <typename T, int TAPS>
__global__ void __launch_bounds__(256) causal_conv_run_kernel(CausalConvCall c) {
  const int t0 = blockIdx.x * CONV_RUN, ch = blockIdx.y * blockDim.x + threadIdx.x;
  const int count = min(CONV_RUN, c.tokens - t0);
  T* cast = static_cast<T*>(c.cast);
  if (ch >= c.channels) {
    if (cast && ch < c.cast_cols)
      for (int i = 0; i < count; ++i) cast[(int64_t)(t0 + i) * c.ld_cast + ch] = from_float<T>(0.f);
    return;
  }
  float w[TAPS];
#pragma unroll
  for (int j = 0; j < TAPS; ++j) w[j] = c.weight[(int64_t)ch * TAPS + j];
  const float bias = c.bias ? c.bias[ch] : 0.f;
  const float* in = c.in + (int64_t)t0 * c.ld_in + ch;
  float* out = c.out + (int64_t)t0 * c.ld_out + ch;
  // most runs are whole and lie in one sequence: no token of theirs asks where it stands
  const int seq0 = c.tok_seq[t0];
  if (count == CONV_RUN && seq0 == c.tok_seq[t0 + CONV_RUN - 1]) {
    const int before = t0 - c.seq_off[seq0];                // tokens of the sequence in front of the run
    const float* held = c.state + (int64_t)c.slots[seq0] * c.state_stride + ch;
    float u[CONV_RUN + TAPS - 1];
#pragma unroll
    for (int i = 0; i < CONV_RUN + TAPS - 1; ++i) {
      const int src = before + i - (TAPS - 1);
      u[i] = *(i >= TAPS - 1 || src >= 0 ? in + (int64_t)(i - (TAPS - 1)) * c.ld_in : held + (int64_t)(TAPS - 1 + src) * c.channels);
    }
#pragma unroll
    for (int i = 0; i < CONV_RUN; ++i) {
      float sum = bias;
#pragma unroll
      for (int j = 0; j < TAPS; ++j) sum = fmaf(w[j], u[i + j], sum);
      const float y = c.act == 0 ? silu_f(sum) : sum;
      out[(int64_t)i * c.ld_out] = y;
      if (cast) cast[(int64_t)(t0 + i) * c.ld_cast + ch] = from_float<T>(y);
    }
    return;
  }
  // (all tokens' table reads, then all their inputs on their way together; behind the step's end the last token again)
  float u[CONV_RUN][TAPS];
#pragma unroll
  for (int i = 0; i < CONV_RUN; ++i) {
    const int k = min(i, count - 1), seq = c.tok_seq[t0 + k], local = t0 + k - c.seq_off[seq];
    const float* held = c.state + (int64_t)c.slots[seq] * c.state_stride + ch;
#pragma unroll
    for (int j = 0; j < TAPS; ++j) {
      const int back = TAPS - 1 - j, src = local - back;
      u[i][j] = *(src >= 0 ? in + (int64_t)(k - back) * c.ld_in : held + (int64_t)(TAPS - 1 + src) * c.channels);
    }
  }
#pragma unroll
  for (int i = 0; i < CONV_RUN; ++i) {
    float sum = bias;
#pragma unroll
    for (int j = 0; j < TAPS; ++j) sum = fmaf(w[j], u[i][j], sum);
    const float y = c.act == 0 ? silu_f(sum) : sum;
    if (i < count) {
      out[(int64_t)i * c.ld_out] = y;
      if (cast) cast[(int64_t)(t0 + i) * c.ld_cast + ch] = from_float<T>(y);
    }
  }
}

template <typename T>
static bool launch_conv_run(hipStream_t stream, const CausalConvCall& c, int cols) {
  dim3 grid((c.tokens + CONV_RUN - 1) / CONV_RUN, (cols + 255) / 256), block(256);
  switch (c.taps) {
    case 2: hipLaunchKernelGGL((causal_conv_run_kernel<T, 2>), grid, block, 0, stream, c); return true;
    case 3: hipLaunchKernelGGL((causal_conv_run_kernel<T, 3>), grid, block, 0, stream, c); return true;
    case 4: hipLaunchKernelGGL((causal_conv_run_kernel<T, 4>), grid, block, 0, stream, c); return true;
  }
  return false;
}

// After the convolution: the state becomes the last taps - 1 inputs of each sequence.
__global__ void __launch_bounds__(256) conv_state_kernel(CausalConvCall c) {
  const int seq = blockIdx.x;
  const int ch = blockIdx.y * blockDim.x + threadIdx.x;
  if (ch >= c.channels) return;
  const int first = c.seq_off[seq], count = c.seq_off[seq + 1] - first;
  float* held = c.state + (int64_t)c.slots[seq] * c.state_stride;
  for (int r = 0; r < c.taps - 1; ++r) {
    const int src = count - (c.taps - 1) + r;
    // (an older input moves up: row r + count lies behind row r, and is read before it is written)
    held[(int64_t)r * c.channels + ch] = src >= 0 ? c.in[(int64_t)(first + src) * c.ld_in + ch]
                                                  : held[(int64_t)(r + count) * c.channels + ch];
  }
}

BT_EXPORT int bt_causal_conv_call(void* stream, const CausalConvCall* c) {
  if (c->tokens <= 0) return BT_OK;
  if (c->channels <= 0 || c->taps <= 0 || c->n_seqs <= 0)
    BT_REFUSE("causal_conv: %d channels, %d taps, %d sequences: all must be positive", c->channels, c->taps, c->n_seqs);
  if (!c->in || !c->weight || !c->out || !c->tok_seq || !c->seq_off || !c->slots || (c->taps > 1 && !c->state))
    BT_REFUSE("causal_conv: missing operand");
  if (c->act != 0 && c->act != 1) BT_REFUSE("causal_conv: unknown activation %d", c->act);
  if (c->ld_in < c->channels || c->ld_out < c->channels || (c->cast && (c->cast_cols < c->channels || c->ld_cast < c->cast_cols)))
    BT_REFUSE("causal_conv: the rows do not hold %d channels", c->channels);
  if (c->taps > 1 && c->state_stride < (int64_t)(c->taps - 1) * c->channels)
    BT_REFUSE("causal_conv: a slot's state of %lld elements does not hold %d inputs of %d channels",
              (long long)c->state_stride, c->taps - 1, c->channels);
  const int cols = c->cast && c->cast_cols > c->channels ? c->cast_cols : c->channels;
  dim3 grid(c->tokens, (cols + 255) / 256), block(256);
  if (c->tokens == c->n_seqs) {        // one token of every sequence
    if (c->cast_dtype == 0)
      hipLaunchKernelGGL((causal_conv_kernel<float, true>), grid, block, 0, (hipStream_t)stream, *c);
    else
      hipLaunchKernelGGL((causal_conv_kernel<bf16_t, true>), grid, block, 0, (hipStream_t)stream, *c);
    return bt_check_launch("causal_conv");
  }
  const int least = c->n_seqs == 1 ? CONV_MIN_VALUES : c->taps >= 4 ? CONV_MIN_VALUES_MANY : CONV_MIN_VALUES_MANY_FEW_TAPS;
  const bool run = c->tokens >= CONV_MIN_TOKENS && (int64_t)c->tokens * c->channels >= least &&
                   (c->cast_dtype == 0 ? launch_conv_run<float>((hipStream_t)stream, *c, cols) : launch_conv_run<bf16_t>((hipStream_t)stream, *c, cols));
  if (run) {
  } else if (c->cast_dtype == 0)
    hipLaunchKernelGGL((causal_conv_kernel<float, false>), grid, block, 0, (hipStream_t)stream, *c);
  else
    hipLaunchKernelGGL((causal_conv_kernel<bf16_t, false>), grid, block, 0, (hipStream_t)stream, *c);
  int rc = bt_check_launch("causal_conv");
  if (rc || c->taps == 1) return rc;
  hipLaunchKernelGGL(conv_state_kernel, dim3(c->n_seqs, (c->channels + 255) / 256), block, 0, (hipStream_t)stream, *c);
  return bt_check_launch("causal_conv state");
}

// ---------------------------------------------------------------------------------------------
// out[t][c] = act(sum_r W[c][r] * low[t][r] + bias[c]), act the softplus (`act` 0), the sigmoid (1) or
// nothing (2); the rank is small.
struct DtProjectCall {
  int dtype;              // element type of W
  int tokens, channels, rank;
  const float* low;       // [tokens][ld_low]
  int64_t ld_low;
  const void* W;          // [channels][rank]
  const float* bias;      // [channels], or null: none
  float* out;             // [tokens][ld_out]
  int64_t ld_out;
  int act;                // 0: softplus, 1: sigmoid, 2: none
};

// TOKENS tokens share a work-group (their rows of `low` wait in LDS, every weight is read once for
// all of them); steps of few tokens take one token a work-group, which is more work-groups and a
// shorter chain in each.
template <typename T, int TOKENS>
__global__ void __launch_bounds__(256) dt_project_kernel(DtProjectCall c) {
  extern __shared__ float rows[];      // [TOKENS][rank]
  const int t0 = blockIdx.x * TOKENS;
  for (int e = threadIdx.x; e < TOKENS * c.rank; e += blockDim.x) {
    const int i = e / c.rank, r = e % c.rank;
    rows[e] = t0 + i < c.tokens ? c.low[(int64_t)(t0 + i) * c.ld_low + r] : 0.f;
  }
  __syncthreads();
  const int ch = blockIdx.y * blockDim.x + threadIdx.x;
  if (ch >= c.channels) return;
  const T* w = static_cast<const T*>(c.W) + (int64_t)ch * c.rank;
  float acc[TOKENS];
#pragma unroll
  for (int i = 0; i < TOKENS; ++i) acc[i] = 0.f;
#pragma unroll 8      // (eight of a thread's weights on their way at once)
  for (int r = 0; r < c.rank; ++r) {
    const float wv = to_float(w[r]);
#pragma unroll
    for (int i = 0; i < TOKENS; ++i) acc[i] = fmaf(wv, rows[i * c.rank + r], acc[i]);
  }
  const float b = c.bias ? c.bias[ch] : 0.f;
#pragma unroll
  for (int i = 0; i < TOKENS; ++i)
    if (t0 + i < c.tokens) {
      const float z = acc[i] + b;
      c.out[(int64_t)(t0 + i) * c.ld_out + ch] = c.act == 0 ? softplus_f(z) : (c.act == 1 ? 1.0f / (1.0f + expf(-z)) : z);
    }
}

template <typename T, int TOKENS>
static void launch_dt_project(hipStream_t stream, const DtProjectCall& c) {
  dim3 grid((c.tokens + TOKENS - 1) / TOKENS, (c.channels + 255) / 256), block(256);
  hipLaunchKernelGGL((dt_project_kernel<T, TOKENS>), grid, block, (size_t)TOKENS * c.rank * sizeof(float), stream, c);
}

BT_EXPORT int bt_dt_project_call(void* stream, const DtProjectCall* c) {
  if (c->tokens <= 0) return BT_OK;
  if (c->channels <= 0 || c->rank <= 0 || c->rank > 1024)
    BT_REFUSE("dt_project: %d channels from rank %d (1..1024)", c->channels, c->rank);
  if (!c->low || !c->W || !c->out || c->ld_low < c->rank || c->ld_out < c->channels)
    BT_REFUSE("dt_project: missing operand or rows too short");
  if (c->act < 0 || c->act > 2) BT_REFUSE("dt_project: unknown activation %d", c->act);
  hipStream_t s = (hipStream_t)stream;
  if (c->tokens <= 16) {
    if (c->dtype == 0) launch_dt_project<float, 1>(s, *c);
    else launch_dt_project<bf16_t, 1>(s, *c);
  } else {
    if (c->dtype == 0) launch_dt_project<float, 8>(s, *c);
    else launch_dt_project<bf16_t, 8>(s, *c);
  }
  return bt_check_launch("dt_project");
}

// ---------------------------------------------------------------------------------------------
// Selective scan.  Per channel c and state element n, token after token of a sequence:
//   S[c][n] <- exp(dt_c * A[c][n]) * S[c][n] + dt_c * x_c * B_n,   A = -exp(A_log)
//   y_c = sum_n S[c][n] * C_n + D_c * x_c;   out_c = y_c * silu(z_c)
// One wave per (8 channels, sequence): eight lanes share a channel, lane j of them owns the state
// elements j, j + 8, ... in registers (R of them).
struct SelectiveScanCall {
  int out_dtype;
  int tokens, n_seqs, channels, state;
  int out_cols;           // columns of out written: the channels, then zeros
  const float* x;         // [tokens][ld_x] after convolution and silu
  int64_t ld_x;
  const float* z;         // [tokens][ld_z] gate, pre-activation
  int64_t ld_z;
  const float* dt;        // [tokens][ld_dt] after softplus
  int64_t ld_dt;
  const float* B;         // [tokens][ld_bc]
  const float* C;         // [tokens][ld_bc]
  int64_t ld_bc;
  const float* A_log;     // [channels][state]
  const float* D;         // [channels]
  void* out;              // [tokens][ld_out]
  int64_t ld_out;
  float* S;               // slot s: [channels][state] at S + s * state_stride
  int64_t state_stride;
  const int* seq_off;
  const int* slots;
  // span > 0: long sequences are cut into spans of that many tokens which are scanned side by side
  // (see "Spans" below); max_count is the most tokens a sequence of the step brings, carry the room
  // for the spans' states: (tokens / span + 2 n_seqs + 1) blocks of channels * state + channels floats
  int span;
  int max_count;
  float* carry;
};

// LDS holds a run of `chunk` tokens' inputs (B and C rows padded to 8 R with zeros, and the wave's eight
// channels' dt, x and z), brought in with loads that are all in flight together: one round trip to
// memory per run of tokens instead of one per token, which is what bounds a recurrence.
// phase 0: whole sequences, from and to the slot's state.  1: spans from zero, leaving E_k and the sum
// of dt.  3: spans from the carried states, writing outputs.
template <typename T, int R>
__global__ void __launch_bounds__(64) selective_scan_kernel(SelectiveScanCall c, int chunk, int phase) {
  extern __shared__ float lds[];
  constexpr int NP = 8 * R;
  float2* BC = reinterpret_cast<float2*>(lds);   // [chunk][NP] pairs (B, C): one 8-byte read for both
  float* dts = lds + (size_t)chunk * NP * 2;     // [chunk][8]
  float* xs = dts + (size_t)chunk * 8;
  float* zs = xs + (size_t)chunk * 8;
  const int lane = threadIdx.x, sub = lane & 7, cl = lane >> 3;
  const int ch = blockIdx.x * 8 + cl, seq = blockIdx.y;
  const bool live = ch < c.channels;
  const int chs = live ? ch : c.channels - 1;        // idle lanes read a valid channel and write nothing
  int first = c.seq_off[seq], last = c.seq_off[seq + 1];
  const int seq_last = last, part = blockIdx.z;
  const int64_t per_span = (int64_t)c.channels * c.state + c.channels;
  float* mine = nullptr;                             // this span's block of the carry
  if (phase) {
    first += part * c.span;
    if (first >= seq_last) return;
    last = min(first + c.span, seq_last);
    mine = c.carry + span_block(c.seq_off, seq, c.span, part) * per_span;
  }
  float* held = c.S + (int64_t)c.slots[seq] * c.state_stride + (int64_t)chs * c.state;
  const float* start = phase == 3 ? mine - per_span + (int64_t)chs * c.state : held;
  float A[R], S[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int n = sub + 8 * r;
    A[r] = n < c.state ? -expf(c.A_log[(int64_t)chs * c.state + n]) : 0.f;
    S[r] = (n < c.state && phase != 1) ? start[n] : 0.f;
  }
  float dt_sum = 0.f;
  const float Dc = c.D[chs];
  T* out = static_cast<T*>(c.out);
  for (int t0 = first; t0 < last; t0 += chunk) {
    const int count = min(chunk, last - t0);
    __syncthreads();
    // (sixteen elements of a lane at a time, all loads issued before the first is stored; with the
    // short rows of this scan, 8 to 32 pairs, the running index measured faster than `fill_pairs`)
    for (int e0 = lane; e0 < count * NP; e0 += 64 * 16) {
      float2 held_bc[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const int e = e0 + 64 * k, i = e / NP, n = e % NP;
        held_bc[k] = (e < count * NP && n < c.state)
                         ? make_float2(c.B[(int64_t)(t0 + i) * c.ld_bc + n], c.C[(int64_t)(t0 + i) * c.ld_bc + n])
                         : make_float2(0.f, 0.f);
      }
#pragma unroll
      for (int k = 0; k < 16; ++k)
        if (e0 + 64 * k < count * NP) BC[e0 + 64 * k] = held_bc[k];
    }
    {
      float held_in[8][3];
#pragma unroll
      for (int k = 0; k < 8; ++k) {          // count <= 64 tokens of 8 channels: at most eight elements a lane
        const int e = lane + 64 * k, i = min(e >> 3, count - 1);
        const int q = min((int)blockIdx.x * 8 + (e & 7), c.channels - 1);
        held_in[k][0] = c.dt[(int64_t)(t0 + i) * c.ld_dt + q];
        held_in[k][1] = c.x[(int64_t)(t0 + i) * c.ld_x + q];
        held_in[k][2] = c.z[(int64_t)(t0 + i) * c.ld_z + q];
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int e = lane + 64 * k;
        if (e < count * 8) {
          dts[e] = held_in[k][0];
          xs[e] = held_in[k][1];
          zs[e] = held_in[k][2];
        }
      }
    }
    __syncthreads();
    auto token = [&](int i) {
      const float dt = dts[i * 8 + cl], xv = xs[i * 8 + cl];
      const float dx = dt * xv;
      float acc = 0.f;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float2 bc = BC[i * NP + sub + 8 * r];
        S[r] = expf(dt * A[r]) * S[r] + dx * bc.x;
        acc = fmaf(S[r], bc.y, acc);
      }
      dt_sum += dt;
      if (phase == 1) return;                        // only the state is wanted
      acc = sum_of_8_lanes(acc);
      if (live && sub == 0)
        out[(int64_t)(t0 + i) * c.ld_out + ch] = from_float<T>((acc + Dc * xv) * silu_f(zs[i * 8 + cl]));
    };
    // four tokens at a time, written out: their reads from LDS, exponentials and sums are in flight
    // together and only the state ties them (the lane sums keep the compiler from unrolling a loop
    // whose length it does not know)
    int i = 0;
    for (; i + 4 <= count; i += 4) {
#pragma unroll
      for (int u = 0; u < 4; ++u) token(i + u);
    }
    for (; i < count; ++i) token(i);
  }
  if (phase == 1) {
    if (live) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int n = sub + 8 * r;
        if (n < c.state) mine[(int64_t)ch * c.state + n] = S[r];
      }
      if (sub == 0) mine[(int64_t)c.channels * c.state + ch] = dt_sum;
    }
    return;
  }
  if (live && phase == 0) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int n = sub + 8 * r;
      if (n < c.state) held[n] = S[r];
    }
  }
  // the columns behind the last channel, which the next product reads as zeros
  if (blockIdx.x == 0)
    for (int t = first; t < last; ++t)
      for (int col = c.channels + lane; col < c.out_cols; col += 64) out[(int64_t)t * c.ld_out + col] = from_float<T>(0.f);
}

// The same with a lane a channel, for steps of many tokens: all N state elements of a channel lie in one lane's registers, so
// nothing crosses lanes, and a token's B and C, the same for all channels, come through scalar loads (the instructions take
// them as they are).  What is left is the recurrence's own arithmetic: an exponential and seven operations a state element
// and token, 48 of the 54 cycles that a wave takes for them on its SIMD.  dt, x and z of the next SL_AHEAD tokens are on
// their way meanwhile.
//   exp(v), v = dt A <= 0, to the accuracy of expf: t = round(v / ln 2), then 2^t (1 + (v - t ln 2)); the factor makes up for
//   the rounding of t, which the hardware's exponential would otherwise carry into the decay.
#define SL_AHEAD 4
// Taken by steps whose longest sequence brings SL_MIN_TOKENS tokens, or a quarter of that where a wave for every 64 channels of
// every sequence makes SL_MIN_WAVES; smaller steps have more waves with eight lanes a channel.  Measured (us, eight lanes / one; 2,048
// channels of 16): 2 x 32 tokens 14.7 / 18.0, 4 x 48 21.0 / 23.6, 2 x 64 25.8 / 22.5, 16 x 20 25.9 / 13.9, 2 x 256 60.6 / 31.2, 8 x 300 208 / 80,
// 2 x 1,024 181 / 73 (of which 46 are the recurrence, gone through twice, and 8 the carry).  Channels of 8: 2 x 64 18.1 / 17.1, 2 x 1,024 124 / 51.
// Of 32, whose tokens' B and C are more than a wave's scalar registers: 2 x 64 26.8 / 39.7, 2 x 160 44.8 / 46.0, 2 x 256 63.6 / 58.8, 2 x 1,024
// 293 / 130, 16 x 20 40.2 / 26.8: from three times as many tokens on.
#define SL_MIN_TOKENS 64
#define SL_MIN_TOKENS_32 192
#define SL_MIN_WAVES 256

__device__ __forceinline__ float decay_of(float v) {
  const float t = v * 1.44269504088896f;
  const float e = __builtin_amdgcn_exp2f(t);
  return fmaf(e, fmaf(-t, 0.693147180559945f, v), e);
}

template <typename T, int N, int PHASE>
__global__ void __launch_bounds__(64) selective_lanes_kernel(SelectiveScanCall c) {
  typedef const __attribute__((address_space(4))) float* Uniform;
  const int lane = threadIdx.x, ch = blockIdx.x * 64 + lane;
  const bool live = ch < c.channels;
  const int chs = live ? ch : c.channels - 1;        // idle lanes read a valid channel and write nothing
  int part = 0;
  const int seq = PHASE ? piece_sequence(c.seq_off, c.n_seqs, c.tokens, c.max_count, c.span, blockIdx.y, part) : blockIdx.y;
  if (PHASE && seq < 0) return;
  int first = c.seq_off[seq], last = c.seq_off[seq + 1];
  const int64_t per_span = (int64_t)c.channels * c.state + c.channels;
  float* mine = nullptr;                             // this span's block of the carry
  if (PHASE) {
    first += part * c.span;
    if (first >= last) return;
    last = min(first + c.span, last);
    mine = c.carry + span_block(c.seq_off, seq, c.span, part) * per_span;
  }
  if (first >= last) return;
  float* held = c.S + (int64_t)c.slots[seq] * c.state_stride + (int64_t)chs * N;
  const float* start = PHASE == 3 ? mine - per_span + (int64_t)chs * N : held;
  float A[N], S[N];
  bool mild = true;
#pragma unroll
  for (int n = 0; n < N; ++n) {
    A[n] = -expf(c.A_log[(int64_t)chs * N + n]);
    S[n] = PHASE != 1 ? start[n] : 0.f;
    mild = mild && A[n] >= -1e8f;
  }
  // (a product of a step, at most 1e30, and a mild A is finite; beyond, where the exponential above would end in a difference of
  // infinities, the whole wave takes expf)
  const bool all_mild = __builtin_amdgcn_ballot_w64(!mild) == 0;
  const float Dc = c.D[chs];
  T* out = static_cast<T*>(c.out) + (int64_t)first * c.ld_out + chs;
  const float *dt_at = c.dt + (int64_t)first * c.ld_dt + chs, *x_at = c.x + (int64_t)first * c.ld_x + chs, *z_at = c.z + (int64_t)first * c.ld_z + chs;
  const float *b_at = c.B + (int64_t)first * c.ld_bc, *c_at = c.C + (int64_t)first * c.ld_bc;
  const int count = last - first;
  float dts[SL_AHEAD], xs[SL_AHEAD], zs[SL_AHEAD], dt_sum = 0.f;
  auto fetch = [&](int t, int u) {                   // (behind the end the last token again, which is not used)
    const int64_t i = min(t, count - 1);
    dts[u] = dt_at[i * c.ld_dt];
    xs[u] = x_at[i * c.ld_x];
    if (PHASE != 1) zs[u] = z_at[i * c.ld_z];
  };
  // a token's B and C are asked for while the token before is worked on (scalar registers: one wait a token, not two)
  float b[N], q[N];
  auto fetch_row = [&](int t, float* b_to, float* q_to) {
    const int64_t i = (int64_t)min(t, count - 1) * c.ld_bc;
    const Uniform from_b = (Uniform)(b_at + i), from_q = (Uniform)(c_at + i);
#pragma unroll
    for (int n = 0; n < N; ++n) {
      b_to[n] = from_b[n];
      if (PHASE != 1) q_to[n] = from_q[n];
    }
  };
  auto token = [&](int t, int u, auto steep) __attribute__((always_inline)) {
    const float dt = dts[u], xv = xs[u], z = PHASE != 1 ? zs[u] : 0.f;
    float b_next[N], q_next[N];
    fetch_row(t + 1, b_next, q_next);
    fetch(t + SL_AHEAD, u);
    __builtin_amdgcn_sched_barrier(0);
    const float step = fminf(dt, 1e30f), dx = dt * xv;               // (an infinite step: the decay is zero, not undefined)
    float acc = 0.f, acc_odd = 0.f;
#pragma unroll
    for (int n = 0; n < N; ++n) {
      S[n] = fmaf(decltype(steep)::value ? expf(dt * A[n]) : decay_of(step * A[n]), S[n], dx * b[n]);
      if (PHASE != 1) {
        if (n & 1) acc_odd = fmaf(S[n], q[n], acc_odd);
        else acc = fmaf(S[n], q[n], acc);
      }
    }
    if (PHASE == 1) dt_sum += dt;
    else if (live) out[(int64_t)t * c.ld_out] = from_float<T>((acc + acc_odd + Dc * xv) * silu_f(z));
#pragma unroll
    for (int n = 0; n < N; ++n) {
      b[n] = b_next[n];
      if (PHASE != 1) q[n] = q_next[n];
    }
  };
  fetch_row(0, b, q);
#pragma unroll
  for (int u = 0; u < SL_AHEAD; ++u) fetch(u, u);
  auto walk = [&](auto steep) __attribute__((always_inline)) {
    int t = 0;
    for (; t + SL_AHEAD <= count; t += SL_AHEAD)
#pragma unroll
      for (int u = 0; u < SL_AHEAD; ++u) token(t + u, u, steep);
#pragma unroll
    for (int u = 0; u < SL_AHEAD - 1; ++u)
      if (t + u < count) token(t + u, u, steep);
  };
  if (__builtin_expect(all_mild, 1)) walk(std::false_type());
  else walk(std::true_type());
  if (PHASE == 1) {
    if (live) {
#pragma unroll
      for (int n = 0; n < N; ++n) mine[(int64_t)ch * N + n] = S[n];
      mine[(int64_t)c.channels * c.state + ch] = dt_sum;
    }
    return;
  }
  if (PHASE == 0 && live) {
#pragma unroll
    for (int n = 0; n < N; ++n) held[n] = S[n];
  }
  // the columns behind the last channel, which the next product reads as zeros
  if (blockIdx.x == 0)
    for (int i = first; i < last; ++i)
      for (int col = c.channels + lane; col < c.out_cols; col += 64) static_cast<T*>(c.out)[(int64_t)i * c.ld_out + col] = from_float<T>(0.f);
}

// C_k = exp(A * sum of dt of span k) * C_(k-1) + E_k along every sequence, in place; C_(-1), the state the
// sequence came with, is kept in front of its spans, and the last C goes into the slot.
__global__ void __launch_bounds__(256) selective_carry_kernel(SelectiveScanCall c) {
  const int seq = blockIdx.y;
  const int64_t index = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, size = (int64_t)c.channels * c.state;
  if (index >= size) return;
  const int count = c.seq_off[seq + 1] - c.seq_off[seq];
  const int spans = (count + c.span - 1) / c.span;
  const int64_t per_span = size + c.channels;
  float* block = c.carry + span_block(c.seq_off, seq, c.span, 0) * per_span;
  float* slot = c.S + (int64_t)c.slots[seq] * c.state_stride;
  float state = slot[index];
  (block - per_span)[index] = state;
  const float A = -expf(c.A_log[index]);
  const int ch = (int)(index / c.state);
  for (int k = 0; k < spans; ++k, block += per_span) {
    state = expf(A * block[size + ch]) * state + block[index];
    block[index] = state;
  }
  slot[index] = state;
}

// Spans of the scan with eight lanes a channel may be as short as the call's room allows where a sequence brings 64 tokens, and 128
// for each wave that a SIMD has; elsewhere they have 64 at least: three launches and twice the arithmetic cost more than
// they save.  Measured (us, spans of 64 / of 16 or more): states of 24 to 32, 2 x 64 tokens on 512 waves (half a wave to a SIMD) 31.8 /
// 26.8, 2 x 128 62.1 / 38.0, 2 x 256 117 / 64, 128 tokens on 256 waves 57 / 28, on 1,024 67.6 / 61.4, but 64 tokens on 1,024 35.6 / 37.3, 3 x 56
// on 768 29.0 / 32.0, 4 x 63 on 1,024 34.9 / 37.8; states of 16, 2 x 128 48 / 29, 64 tokens on 1,024 waves 27.8 / 28.3, 3 x 56 22.5 / 23.7.
#define SS_LONG_SPAN 64

static int shortest_span(const SelectiveScanCall& c, int64_t waves) {
  const bool few = c.max_count >= SS_LONG_SPAN && (int64_t)c.max_count * simd_count() >= 2 * SS_LONG_SPAN * waves;
  return few || c.span <= 0 || c.span >= SS_LONG_SPAN ? c.span : SS_LONG_SPAN;
}

template <typename T, int R>
static void launch_selective_scan_r(hipStream_t stream, const SelectiveScanCall& c) {
  const int per_token = 2 * 8 * R + 24;
  dim3 block(64);
  const int64_t waves = (int64_t)((c.channels + 7) / 8) * c.n_seqs;
  const int span = span_tokens(shortest_span(c, waves), c.max_count, c.carry, waves, 2);
  if (span > 0) {
    SelectiveScanCall cut = c;
    cut.span = span;
    const int chunk = scan_chunk(per_token, span);
    const int spans = (c.max_count + span - 1) / span;
    dim3 grid((c.channels + 7) / 8, c.n_seqs, spans);
    const size_t lds = (size_t)chunk * per_token * sizeof(float);
    hipLaunchKernelGGL((selective_scan_kernel<T, R>), grid, block, lds, stream, cut, chunk, 1);
    hipLaunchKernelGGL(selective_carry_kernel, dim3((c.channels * c.state + 255) / 256, c.n_seqs), dim3(256), 0, stream, cut);
    hipLaunchKernelGGL((selective_scan_kernel<T, R>), grid, block, lds, stream, cut, chunk, 3);
    return;
  }
  const int chunk = scan_chunk(per_token, c.tokens);
  dim3 grid((c.channels + 7) / 8, c.n_seqs);
  hipLaunchKernelGGL((selective_scan_kernel<T, R>), grid, block, (size_t)chunk * per_token * sizeof(float), stream, c, chunk, 0);
}

// Waves of 64 channels that the step's tokens would make if all its sequences were as long as the longest: a prompt beside single
// tokens is one long walk and is cut into spans, however many tokens come with it.
static int64_t lane_waves(const SelectiveScanCall& c) {
  return (int64_t)((c.channels + 63) / 64) * (((int64_t)c.tokens + c.max_count - 1) / c.max_count);
}

// Spans have the room's shortest length at least, and so many tokens that walking one twice (0.27 us a token with 16 states, twice that
// with 32) takes no less than the carry, which goes through them in order (0.36 us each): measured (us) for one sequence of 4,000 tokens
// of 128 channels 110 in spans of 16, 78 so, of 512 channels 125 and 85.  Measured beside single tokens (eight lanes a channel / one by the sequences' number /
// so; 2,048 channels of 16): 1,000 and 32 345 / 497 / 60, 500 and 63 175 / 243 / 49, 64 and 31 25 / 34 / 23.
template <typename T, int N>
static void launch_selective_lanes(hipStream_t stream, const SelectiveScanCall& c) {
  const int groups = (c.channels + 63) / 64;
  int shortest = c.span;
  while (shortest > 0 && 3 * (int64_t)shortest * shortest * (N > 16 ? N / 16 : 1) < 2 * (int64_t)c.max_count) ++shortest;
  const int span = span_tokens(shortest, c.max_count, c.carry, lane_waves(c), 1, 2);
  if (span > 0 && c.tokens / span + c.n_seqs <= 65535) {
    SelectiveScanCall cut = c;
    cut.span = span;
    dim3 grid(groups, c.tokens / span + c.n_seqs);
    hipLaunchKernelGGL((selective_lanes_kernel<T, N, 1>), grid, dim3(64), 0, stream, cut);
    hipLaunchKernelGGL(selective_carry_kernel, dim3((c.channels * c.state + 255) / 256, c.n_seqs), dim3(256), 0, stream, cut);
    hipLaunchKernelGGL((selective_lanes_kernel<T, N, 3>), grid, dim3(64), 0, stream, cut);
    return;
  }
  hipLaunchKernelGGL((selective_lanes_kernel<T, N, 0>), dim3(groups, c.n_seqs), dim3(64), 0, stream, c);
}

template <typename T>
static int launch_selective_scan(hipStream_t stream, const SelectiveScanCall& c) {
  // (many short sequences beside the longest are waves of a few tokens: 64 tokens and 31 single ones 25 us with eight lanes, 30 with one)
  const bool others = short_sequences(c.tokens, c.n_seqs, c.max_count) * ((c.channels + 63) / 64) > 512;
  const bool many = c.max_count >= (c.state == 32 ? SL_MIN_TOKENS_32 : others ? 2 * SL_MIN_TOKENS : SL_MIN_TOKENS) ||
      (c.max_count >= SL_MIN_TOKENS / 4 && lane_waves(c) >= SL_MIN_WAVES);
  if (many && (c.state == 8 || c.state == 16 || c.state == 32)) {
    if (c.state == 8) launch_selective_lanes<T, 8>(stream, c);
    else if (c.state == 16) launch_selective_lanes<T, 16>(stream, c);
    else launch_selective_lanes<T, 32>(stream, c);
    return bt_check_launch("selective_scan");
  }
  const int per = (c.state + 7) / 8;
  if (per <= 1) launch_selective_scan_r<T, 1>(stream, c);
  else if (per <= 2) launch_selective_scan_r<T, 2>(stream, c);
  else if (per <= 4) launch_selective_scan_r<T, 4>(stream, c);
  else if (per <= 8) launch_selective_scan_r<T, 8>(stream, c);
  else if (per <= 16) launch_selective_scan_r<T, 16>(stream, c);
  else launch_selective_scan_r<T, 32>(stream, c);
  return bt_check_launch("selective_scan");
}

BT_EXPORT int bt_selective_scan_call(void* stream, const SelectiveScanCall* c) {
  if (c->tokens <= 0) return BT_OK;
  if (c->channels <= 0 || c->state <= 0 || c->state > 256 || c->n_seqs <= 0)
    BT_REFUSE("selective_scan: %d channels with %d state elements (1..256), %d sequences", c->channels, c->state, c->n_seqs);
  if (!c->x || !c->z || !c->dt || !c->B || !c->C || !c->A_log || !c->D || !c->out || !c->S || !c->seq_off || !c->slots)
    BT_REFUSE("selective_scan: missing operand");
  if (c->ld_x < c->channels || c->ld_z < c->channels || c->ld_dt < c->channels || c->ld_bc < c->state ||
      c->out_cols < c->channels || c->ld_out < c->out_cols || c->state_stride < (int64_t)c->channels * c->state)
    BT_REFUSE("selective_scan: rows or state too short for %d channels of %d", c->channels, c->state);
  return c->out_dtype == 0 ? launch_selective_scan<float>((hipStream_t)stream, *c)
                           : launch_selective_scan<bf16_t>((hipStream_t)stream, *c);
}

// ---------------------------------------------------------------------------------------------
// Scan with one decay per head.  Per head h (its group g = h / (heads / groups)), token after token:
//   dt = softplus(dt_raw_h + dt_bias_h);   a = exp(-exp(A_log_h) * dt)
//   S_h[n][p] <- a * S_h[n][p] + dt * B_g[n] * x_h[p];   y_h[p] = sum_n S_h[n][p] * C_g[n] + D_h * x_h[p]
// One wave per (4 channels p of a head, sequence): sixteen lanes share a channel, lane j of them owns
// the state elements j, j + 16, ... in registers.
struct HeadScanCall {
  int tokens, n_seqs, heads, vdim, state, groups;
  const float* x;         // [tokens][ld]: head h at columns h * vdim (after convolution and silu)
  const float* B;         // [tokens][ld]: group g at columns g * state
  const float* C;
  int64_t ld;
  const float* dt_raw;    // [tokens][ld_dt]: one per head, before bias and softplus
  int64_t ld_dt;
  const float* dt_bias;   // [heads]
  const float* A_log;     // [heads]
  const float* D;         // [heads]
  float* y;               // [tokens][ld_y] float32: head h at columns h * vdim
  int64_t ld_y;
  float* S;               // slot s: [heads][vdim / 4 rounded up][state][4] at S + s * state_stride
  int64_t state_stride;
  const int* seq_off;
  const int* slots;
  // spans, as in SelectiveScanCall: a block of the carry holds a state (in the slot's layout) and, behind
  // it, one number a head: the sum over the span of the logarithms of its decays
  int span;
  int max_count;
  float* carry;
  // null, or room for what blocks of 16 tokens leave, aligned to 16 bytes: (tokens / 16 + n_seqs + 1) blocks of 32 groups * state +
  // 288 heads floats; with it long sequences go in blocks on the matrix units
  float* blocks;
};

// The state of a slot is laid out for this kernel's lanes: [heads][tiles of 4 channels][state][4], so
// that a wave's load of one register's worth of state (16 state elements by 4 channels) is 256
// contiguous bytes.  Nobody else reads it; a new sequence's state is all zeros in any layout.
// A work-group is four waves, each with four channels of the same head: they share the run of B and C in
// LDS (every wave bringing a quarter of it in) and have one SIMD each.
#define HS_WAVES 4

template <int R, int PHASE>
__global__ void __launch_bounds__(64 * HS_WAVES) head_scan_kernel(HeadScanCall c, int chunk, int spans, int tiles) {
  extern __shared__ float lds[];
  constexpr int NP = 16 * R;
  float2* BC = reinterpret_cast<float2*>(lds);                              // [chunk][NP] pairs (B, C): one 8-byte read for both
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, sub = lane & 15, pl = lane >> 4;
  // [waves][chunk][4]: a token and channel's dt * x, D * x, decay, log decay
  float4* tok = reinterpret_cast<float4*>(lds + (size_t)chunk * NP * 2) + (size_t)wave * chunk * 4;
  const int tile = min((int)blockIdx.x * HS_WAVES + wave, tiles - 1), head = blockIdx.y;
  const bool works = (int)blockIdx.x * HS_WAVES + wave < tiles;          // (a wave without a tile only helps to bring B and C in)
  const int seq = blockIdx.z / spans, part = blockIdx.z % spans;
  const int p = tile * 4 + pl;
  const bool live = works && p < c.vdim;
  const int group = head / (c.heads / c.groups);
  int first = c.seq_off[seq], last = c.seq_off[seq + 1];
  const int seq_last = last;
  const int64_t state_size = (int64_t)c.heads * tiles * c.state * 4, per_span = state_size + c.heads;
  const int64_t in_state = ((int64_t)head * tiles + tile) * c.state * 4 + pl;
  float* mine = nullptr;                             // this span's block of the carry
  if (PHASE) {
    first += part * c.span;
    if (first >= seq_last) return;                   // (the whole work-group: it is one span's)
    last = min(first + c.span, seq_last);
    mine = c.carry + span_block(c.seq_off, seq, c.span, part) * per_span;
  }
  float* held = c.S + (int64_t)c.slots[seq] * c.state_stride + in_state;
  const float* start = PHASE == 3 ? mine - per_span + in_state : held;
  float S[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int n = sub + 16 * r;
    S[r] = (n < c.state && PHASE != 1) ? start[(int64_t)n * 4] : 0.f;
  }
  float log_decay = 0.f;
  const float rate = -expf(c.A_log[head]), bias = c.dt_bias[head], Dh = c.D[head];
  const float* Bg = c.B + group * c.state;
  const float* Cg = c.C + group * c.state;
  float* ycol = c.y + head * c.vdim + (live ? p : 0);
  for (int t0 = first; t0 < last; t0 += chunk) {
    const int count = min(chunk, last - t0);
    __syncthreads();
    fill_pairs<NP, 64 * HS_WAVES>(BC, Bg, Cg, (int)c.ld, t0, count, c.state, (int)threadIdx.x);
    for (int e = lane; e < count * 4; e += 64) {
      const int i = e >> 2, q = tile * 4 + (e & 3);
      const float xv = q < c.vdim ? c.x[(int64_t)(t0 + i) * c.ld + head * c.vdim + q] : 0.f;
      const float step = softplus_f(c.dt_raw[(int64_t)(t0 + i) * c.ld_dt + head] + bias);
      tok[e] = make_float4(step * xv, Dh * xv, expf(rate * step), rate * step);
    }
    __syncthreads();
    if (!works) continue;
    // one token: the state moves on; the channel's output (in every lane of its sixteen) is returned
    auto token = [&](int i) -> float {
      const float4 in = tok[i * 4 + pl];
      float acc = 0.f;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float2 bc = BC[i * NP + sub + 16 * r];
        S[r] = fmaf(in.z, S[r], in.x * bc.x);
        acc = fmaf(S[r], bc.y, acc);
      }
      if (PHASE == 1) {
        log_decay += in.w;
        return 0.f;                                  // only the state is wanted
      }
      return sum_of_16_lanes(acc) + in.y;
    };
    // Sixteen tokens at a time, written out: their reads from LDS and sums are in flight together and
    // only the state ties them (the lane sums keep the compiler from unrolling a loop whose length it
    // does not know); lane j of a channel's sixteen keeps the j-th of them, and one store writes all.
    int i = 0;
    for (; i + 16 <= count; i += 16) {
      float kept = 0.f;
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const float y = token(i + u);
        kept = sub == u ? y : kept;
      }
      if (PHASE != 1 && live) ycol[(int64_t)(t0 + i + sub) * c.ld_y] = kept;
    }
    for (; i < count; ++i) {
      const float y = token(i);
      if (PHASE != 1 && live && sub == 0) ycol[(int64_t)(t0 + i) * c.ld_y] = y;
    }
  }
  if (!works) return;
  if (PHASE == 1) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int n = sub + 16 * r;
      if (n < c.state) mine[in_state + (int64_t)n * 4] = S[r];
    }
    if (tile == 0 && lane == 0) mine[state_size + head] = log_decay;
    return;
  }
  if (PHASE == 0) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int n = sub + 16 * r;
      if (n < c.state) held[(int64_t)n * 4] = S[r];
    }
  }
}

// C_k = exp(sum of the span's log decays) * C_(k-1) + E_k along every sequence, in place (see selective_carry_kernel).
__global__ void __launch_bounds__(256) head_carry_kernel(HeadScanCall c, int tiles) {
  const int seq = blockIdx.y;
  const int64_t per_head = (int64_t)tiles * c.state * 4, size = per_head * c.heads;
  const int64_t index = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (index >= size) return;
  const int count = c.seq_off[seq + 1] - c.seq_off[seq];
  const int spans = (count + c.span - 1) / c.span;
  const int64_t per_span = size + c.heads;
  float* block = c.carry + span_block(c.seq_off, seq, c.span, 0) * per_span;
  float* slot = c.S + (int64_t)c.slots[seq] * c.state_stride;
  float state = slot[index];
  (block - per_span)[index] = state;
  const int head = (int)(index / per_head);
  for (int k = 0; k < spans; ++k, block += per_span) {
    state = expf(block[size + head]) * state + block[index];
    block[index] = state;
  }
  slot[index] = state;
}

// Into spans of how many tokens the step's long sequences are cut, 0 for not at all.
static int head_span(const HeadScanCall& c) {
  return span_tokens(c.span, c.max_count, c.carry, (int64_t)((c.vdim + 3) / 4) * c.heads * c.n_seqs, 1);
}

template <int R>
static void launch_head_scan_r(hipStream_t stream, const HeadScanCall& c) {
  const int per_token = 2 * 16 * R + 16 * HS_WAVES;
  const int tiles = (c.vdim + 3) / 4, groups = (tiles + HS_WAVES - 1) / HS_WAVES;
  dim3 block(64 * HS_WAVES);
  const int span = head_span(c);
  if (span > 0) {
    HeadScanCall cut = c;
    cut.span = span;
    const int chunk = scan_chunk(per_token, span);
    const int spans = (c.max_count + span - 1) / span;
    dim3 grid(groups, c.heads, c.n_seqs * spans);
    const size_t lds = (size_t)chunk * per_token * sizeof(float);
    hipLaunchKernelGGL((head_scan_kernel<R, 1>), grid, block, lds, stream, cut, chunk, spans, tiles);
    const int64_t size = (int64_t)c.heads * tiles * c.state * 4;
    hipLaunchKernelGGL(head_carry_kernel, dim3((unsigned)((size + 255) / 256), c.n_seqs), dim3(256), 0, stream, cut, tiles);
    hipLaunchKernelGGL((head_scan_kernel<R, 3>), grid, block, lds, stream, cut, chunk, spans, tiles);
    return;
  }
  const int chunk = scan_chunk(per_token, c.tokens);
  dim3 grid(groups, c.heads, c.n_seqs);
  hipLaunchKernelGGL((head_scan_kernel<R, 0>), grid, block, (size_t)chunk * per_token * sizeof(float), stream, c, chunk, 1, tiles);
}

// --- the same in blocks of sixteen tokens on the matrix units -----------------------------------
//
// With one decay a head a block of 16 tokens does to the state what a few products do.  With a_t the product of the
// block's decays up to and with token t, b_s that of the decays behind token s and
//     G = C B^T,   M[t][s] = G[t][s] g_(s+1) .. g_t dt_s   (s <= t):
//     y = diag(a) C S0 + M x + D x,   S = a_16 S0 + B^T diag(b dt) x
// B and C are the group's, so one kernel lays them out for the lanes once for all heads, with G behind every head's M, a and
// b dt, and a second one walks the blocks in order with the state in registers (v_mfma_f32_16x16x4_f32: 32 bits throughout;
// decays are only multiplied with each other).  Operand layouts and the K values' order as in linear_attention.hip: a
// lane's four values of a 16 x 16 tile lie side by side, step i of a product takes K number 4 g + i in lane group g, and
// results land where the next product reads them.
#define HB_TOKENS 16
#define HB_HEADS 8              // heads a work-group of the first kernel prepares
// Steps whose longest sequence brings at least this many tokens may go in blocks (blocks_pay).  Measured (us, as whole sequences or spans / in
// blocks; 32 heads of 64 x 128): 2 x 40 tokens 16.1 / 13.2, 16 x 40 48.7 / 36.1, 2 x 128 39 / 17, 2 x 1,024 225 / 58, 8 x 300 141 / 60.
// Of the longest, 11 us go to the operands; a block then takes 0.7 us, 0.25 of them on the matrix units: a wave is alone on
// its SIMD and pays every instruction around them, and the trip through LDS, itself.
#define HB_MIN_TOKENS 40

// Floats of a block: a group's C and B [tiles of 16 state elements][64 lanes][4] each, then every head's M [64][4], a [16], b dt [16].
__host__ __device__ __forceinline__ int64_t hb_floats(const HeadScanCall& c) {
  return (int64_t)c.groups * 2 * HB_TOKENS * c.state + (int64_t)c.heads * (HB_TOKENS * HB_TOKENS + 2 * HB_TOKENS);
}
__device__ __forceinline__ float* hb_place(const HeadScanCall& c, int seq, int block) {
  return c.blocks + (int64_t)(c.seq_off[seq] / HB_TOKENS + seq + block) * hb_floats(c);
}

template <int DT>
__global__ void __launch_bounds__(256) head_blocks_kernel(HeadScanCall c) {
  constexpr int DIM = 16 * DT, PITCH = DIM + 4;
  __shared__ __attribute__((aligned(16))) float B[HB_TOKENS][PITCH], C[HB_TOKENS][PITCH];
  __shared__ __attribute__((aligned(16))) floatx4 parts[4][64];
  __shared__ float steps[HB_HEADS][HB_TOKENS], decays[HB_HEADS][HB_TOKENS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, n = lane & 15;
  int part;
  const int seq = piece_sequence(c.seq_off, c.n_seqs, c.tokens, c.max_count, HB_TOKENS, blockIdx.y, part);
  if (seq < 0) return;                                                   // (the whole work-group)
  const int first = c.seq_off[seq] + part * HB_TOKENS, count = min(HB_TOKENS, c.seq_off[seq + 1] - first);
  const int per_group = c.heads / c.groups, sets = (per_group + HB_HEADS - 1) / HB_HEADS;
  const int group = blockIdx.x / sets, head0 = group * per_group + blockIdx.x % sets * HB_HEADS;
  const int heads = min(HB_HEADS, (group + 1) * per_group - head0);
  float* place = hb_place(c, seq, part);
  // rows behind the sequence's end hold zeros and decay by one: they change nothing
#pragma unroll
  for (int j = 0; j < DT; ++j) {
    const int i = (tid + 256 * j) / DIM, d = (tid + 256 * j) % DIM;
    const int64_t at = (int64_t)(first + min(i, count - 1)) * c.ld + group * DIM + d;
    const float b = c.B[at], q = c.C[at];
    B[i][d] = i < count ? b : 0.f;
    C[i][d] = i < count ? q : 0.f;
  }
  if (tid < HB_HEADS * HB_TOKENS) {
    const int h = tid / HB_TOKENS, i = tid % HB_TOKENS, head = head0 + min(h, heads - 1);
    const float step = softplus_f(c.dt_raw[(int64_t)(first + min(i, count - 1)) * c.ld_dt + head] + c.dt_bias[head]);
    steps[h][i] = i < count ? step : 0.f;
    decays[h][i] = i < count ? expf(-expf(c.A_log[head]) * step) : 1.f;
  }
  __syncthreads();
  // (four sums side by side, added in pairs: one chain of a wave's 32 products rounds a third more than the walk's sums do)
  floatx4 sums[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) sums[i] = floatx4{0.f, 0.f, 0.f, 0.f};
  floatx4* frag = reinterpret_cast<floatx4*>(place + (int64_t)group * 2 * HB_TOKENS * DIM);
  for (int tile = wave; tile < DT; tile += 4) {
    const floatx4 q = *reinterpret_cast<const floatx4*>(&C[n][16 * tile + 4 * g]), k = *reinterpret_cast<const floatx4*>(&B[n][16 * tile + 4 * g]);
#pragma unroll
    for (int i = 0; i < 4; ++i) sums[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(q[i], k[i], sums[i], 0, 0, 0);
    if (blockIdx.x % sets == 0) {
      floatx4 u;
#pragma unroll
      for (int i = 0; i < 4; ++i) u[i] = B[4 * g + i][16 * tile + n];
      frag[64 * tile + lane] = q;
      frag[64 * (DT + tile) + lane] = u;
    }
  }
  parts[wave][lane] = (sums[0] + sums[1]) + (sums[2] + sums[3]);         // lane holds G[4 g + i][n]
  __syncthreads();
  const int t = tid >> 4, s = tid & 15;
  auto part_of = [&](int w) { return reinterpret_cast<const float*>(&parts[w][16 * (t >> 2) + s])[t & 3]; };
  const float product = (part_of(0) + part_of(1)) + (part_of(2) + part_of(3));
  for (int h = 0; h < heads; ++h) {
    float decay = 1.f;                                                   // of the tokens behind s up to t
#pragma unroll
    for (int r = 1; r < HB_TOKENS; ++r) decay *= r > s && r <= t ? decays[h][r] : 1.f;
    float* mine = place + (int64_t)c.groups * 2 * HB_TOKENS * DIM + (int64_t)(head0 + h) * (HB_TOKENS * HB_TOKENS + 2 * HB_TOKENS);
    mine[(t + 16 * (s >> 2)) * 4 + (s & 3)] = s <= t ? product * decay * steps[h][s] : 0.f;
    if (s == 0) mine[HB_TOKENS * HB_TOKENS + t] = decays[h][0] * decay;
    if (t == HB_TOKENS - 1) mine[HB_TOKENS * HB_TOKENS + HB_TOKENS + s] = decay * steps[h][s];
  }
}

// One work-group per 16 channels of a head and sequence; four waves share the state elements, every wave's part of
// C S0 (and one step of M x) meets in LDS.  The operands of the next HB_AHEAD - 1 blocks are on their way.
// What bounds a block is one wave's chain on each SIMD, 17 matrix instructions of 32 cycles, and the address unit that four waves' loads
// share: a load stands behind each matrix instruction, a token's factors come a lane each of a quad, sums meet behind the next
// block's first products, and the loop takes whole turns of HB_AHEAD (with a way out between two blocks all loads were waited for in
// front of a turn).  Measured (us, 32 heads of 64 x 128, 2 x 1,024 tokens, the walk alone): 50.1 -> 40.7.
#define HB_AHEAD 4

template <int TW>
struct HbStage {
  floatx4 c[TW], b[TW];
  float a, strength, m, all, x[4];                         // (of a quad's four lanes each has one of the tokens' a and strength)
};

// M's zeros for the tokens behind a row's own are multiplied too, so an x there that is not finite makes the row not a number.  A
// work-group that has met one (`seen` is not a number then) goes through its sequence again behind the walk, token by token from the state
// that still lies in its slot.  (us for 2 x 1,024 tokens of 32 heads of 64 x 128 / 4,000 of 24 of 64 x 64: without 57.5 / 123.5, so 58.2 / 129;
// summing again in the block that holds it, a test for every block, 60 to 62 / 130 to 138; a second walk over blocks in this
// kernel 59 / 131, in a function of its own, for its scratch memory, 72 / 136.)
template <int DT>
__global__ void __launch_bounds__(256, 2) head_blocks_walk_kernel(HeadScanCall c) {
  constexpr int TW = (DT + 3) / 4, DIM = 16 * DT;
  __shared__ __attribute__((aligned(16))) floatx4 parts[2][4][64];
  __shared__ int spoiled[4];
  // the columns of a head and sequence, and the heads of a group, read the same operands: they are numbered onto one XCD
  const int columns = c.vdim / 16, pair = blockIdx.x / (8 * columns) * 8 + blockIdx.x % 8;
  if (pair >= c.heads * c.n_seqs) return;
  const int column = blockIdx.x / 8 % columns, head = pair % c.heads, seq = pair / c.heads;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, n = lane & 15;
  const int first = c.seq_off[seq], count = c.seq_off[seq + 1] - first;
  if (count <= 0) return;
  const int blocks = (count + HB_TOKENS - 1) / HB_TOKENS, group = head / (c.heads / c.groups);
  const int64_t stride = hb_floats(c) * 4;
  const int vtiles = (c.vdim + 3) / 4, p = 16 * column + n;
  float* slot = c.S + (int64_t)c.slots[seq] * c.state_stride + ((int64_t)head * vtiles + p / 4) * DIM * 4 + p % 4;
  auto mine = [&](int j) { return DT % 4 == 0 || wave * TW + j < DT; };
  floatx4 S[TW];
#pragma unroll
  for (int j = 0; j < TW; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) S[j][i] = mine(j) ? slot[(int64_t)(16 * (wave * TW + j) + 4 * g + i) * 4] : 0.f;
  const float Dh = c.D[head];
  float seen = 0.f;
  // a block's operands: one address that all lanes share, and every lane's distances from it
  uint32_t from_tile[TW], from_x[4], from_last[4];
#pragma unroll
  for (int j = 0; j < TW; ++j) from_tile[j] = (group * 2 * HB_TOKENS * DIM + 256 * min(wave * TW + j, DT - 1) + 4 * lane) * 4;
  const uint32_t from_head = (c.groups * 2 * HB_TOKENS * DIM + head * (HB_TOKENS * HB_TOKENS + 2 * HB_TOKENS)) * 4;
  const uint32_t from_m = from_head + (4 * lane + wave) * 4, from_a = from_head + (HB_TOKENS * HB_TOKENS + 4 * g + (n & 3)) * 4;
  const int left = count - (blocks - 1) * HB_TOKENS;                      // tokens of the last block
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    from_x[i] = (uint32_t)((4 * g + i) * c.ld + p) * 4;
    from_last[i] = (uint32_t)(min(4 * g + i, left - 1) * c.ld + p) * 4;
  }
  const char* at = reinterpret_cast<const char*>(hb_place(c, seq, 0));
  const char* x_at = reinterpret_cast<const char*>(c.x + (int64_t)first * c.ld + head * c.vdim);
  int row = 4 * g + wave, fetched = 0;                                   // a wave finishes every fourth token
  float* out = c.y + (first + (int64_t)min(row, count - 1)) * c.ld_y + head * c.vdim + p;
  const int64_t out_step = HB_TOKENS * c.ld_y;
  HbStage<TW> stages[HB_AHEAD];
  constexpr int LOADS = 2 * TW + 8;
  auto fetch = [&](HbStage<TW>& st, auto number) {         // one of a block's LOADS, in order
    constexpr int load = decltype(number)::value, j = load % TW, other = load - 2 * TW;
    auto value = [&](const char* base, uint32_t from) { return *reinterpret_cast<const float*>(base + from); };
    if constexpr (load < 2 * TW) {
      const floatx4 four = *reinterpret_cast<const floatx4*>(at + (from_tile[j] + (load < TW ? 0 : HB_TOKENS * DIM * 4)));
      if constexpr (load < TW) st.c[j] = four;
      else st.b[j] = four;
    } else if constexpr (other == 0) {
      st.a = value(at, from_a);
    } else if constexpr (other == 1) {
      st.strength = value(at, from_a + HB_TOKENS * 4);
    } else if constexpr (other == 2) {
      st.m = value(at, from_m);
    } else if constexpr (other == 3) {
      st.all = value(at, from_head + (HB_TOKENS * HB_TOKENS + HB_TOKENS - 1) * 4);
    } else if constexpr (other < 8) {
      st.x[other - 4] = value(x_at, fetched >= blocks - 1 ? from_last[other - 4] : from_x[other - 4]);
      if constexpr (other == 7) {
        // on to the next block; at the end the last one's operands are asked for again and not used
        const bool more = ++fetched < blocks;
        at += more ? stride : 0;
        x_at += more ? HB_TOKENS * c.ld * 4 : 0;
      }
    }
  };
  // A block's outputs are added up from LDS behind the next block's barrier.
  float pending = 0.f;
  auto read_parts = [&](int turn, float (&r)[4]) {
    const float* at = reinterpret_cast<const float*>(&parts[turn][0][lane]) + wave;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = at[256 * i];
  };
  auto finish = [&](const float (&r)[4]) {
    const float y = ((r[0] + r[1]) + (r[2] + r[3])) + pending;
    if (row < count) *out = y;
    row += HB_TOKENS;
    out += out_step;
  };
  auto walk = [&](HbStage<TW>& st, int turn, int block, auto asks, HbStage<TW>& next) {
    auto ask = [&](auto number) {                          // a load of the next block's operands behind each matrix instruction
      if constexpr (decltype(asks)::value) fetch(next, number);
      __builtin_amdgcn_sched_barrier(0);
    };
    // (a sum a tile, taken in turn: an instruction that adds to the one before it waits for it)
    floatx4 sums[TW];
#pragma unroll
    for (int j = 0; j < TW; ++j) sums[j] = floatx4{0.f, 0.f, 0.f, 0.f};
    each<4 * TW>([&](auto number) {
      constexpr int j = decltype(number)::value % TW, i = decltype(number)::value / TW;
      if (mine(j)) sums[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(st.c[j][i], S[j][i], sums[j], 0, 0, 0);
      ask(number);
    });
    float x[4], u[4], r[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = block * HB_TOKENS + 4 * g + i < count ? st.x[i] : 0.f;
    u[0] = dpp_move<0x00>(st.strength) * x[0];
    u[1] = dpp_move<0x55>(st.strength) * x[1];
    u[2] = dpp_move<0xAA>(st.strength) * x[2];
    u[3] = dpp_move<0xFF>(st.strength) * x[3];
    const float own = (wave & 2) ? ((wave & 1) ? x[3] : x[2]) : ((wave & 1) ? x[1] : x[0]);
    lds_barrier();
    read_parts(turn ^ 1, r);
    const floatx4 within = __builtin_amdgcn_mfma_f32_16x16x4f32(st.m, own, floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    ask(Number<4 * TW>());
    seen = fmaf(own, 0.f, seen);
#pragma unroll
    for (int j = 0; j < TW; ++j) S[j] *= st.all;
    each<4 * TW>([&](auto number) {
      constexpr int j = decltype(number)::value % TW, i = decltype(number)::value / TW;
      if (mine(j)) S[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(st.b[j][i], u[i], S[j], 0, 0, 0);
      ask(Number<4 * TW + 1 + decltype(number)::value>());
    });
    ask(Number<8 * TW + 1>());
    static_assert(8 * TW + 2 >= LOADS, "every load has its place");
    if (TW > 1) sums[0] += sums[TW - 1];
    floatx4 sum;
    sum[0] = sums[0][0] * dpp_move<0x00>(st.a);
    sum[1] = sums[0][1] * dpp_move<0x55>(st.a);
    sum[2] = sums[0][2] * dpp_move<0xAA>(st.a);
    sum[3] = sums[0][3] * dpp_move<0xFF>(st.a);
    parts[turn][wave][lane] = sum + within;
    if (block > 0) finish(r);
    pending = Dh * own;
  };
#pragma unroll
  for (int i = 0; i < HB_AHEAD - 1; ++i) {
    each<LOADS>([&](auto number) { fetch(stages[i], number); });
    __builtin_amdgcn_sched_barrier(0);                     // (in order: a stage is waited for by the loads behind it)
  }
  landed(S);
  int block = 0;
  for (; block + HB_AHEAD <= blocks; block += HB_AHEAD) {  // (whole turns: see HB_AHEAD)
#pragma unroll
    for (int i = 0; i < HB_AHEAD; ++i) walk(stages[i], i & 1, block + i, Number<1>(), stages[(i + HB_AHEAD - 1) % HB_AHEAD]);
  }
#pragma unroll
  for (int i = 0; i < HB_AHEAD - 1; ++i)
    if (block + i < blocks) walk(stages[i], i & 1, block + i, Number<0>(), stages[i]);     // (the same for all four waves)
  lds_barrier();
  {
    float r[4];
    read_parts((blocks - 1) & 1, r);
    finish(r);
  }
  const int found = __builtin_amdgcn_ballot_w64(!(seen == 0.f)) != 0;
  if (lane == 0) spoiled[wave] = found;
  __syncthreads();
  if (__builtin_expect(spoiled[0] | spoiled[1] | spoiled[2] | spoiled[3], 0)) {
    // sixteen lanes a channel, every sixteenth state element in each of them
    const int channel = 16 * column + (tid >> 4), part = tid & 15;
    float* held = c.S + (int64_t)c.slots[seq] * c.state_stride + ((int64_t)head * vtiles + channel / 4) * DIM * 4 + channel % 4;
    float state[DT];
#pragma unroll
    for (int j = 0; j < DT; ++j) state[j] = held[(part + 16 * j) * 4];
    const float rate = expf(c.A_log[head]);
#pragma unroll 1
    for (int t = first; t < first + count; ++t) {
      const float step = softplus_f(c.dt_raw[(int64_t)t * c.ld_dt + head] + c.dt_bias[head]), decay = expf(-rate * step);
      const float value = c.x[(int64_t)t * c.ld + head * c.vdim + channel];
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < DT; ++j) {
        const int64_t at = (int64_t)t * c.ld + group * DIM + part + 16 * j;
        state[j] = fmaf(decay, state[j], c.B[at] * (step * value));
        sum = fmaf(state[j], c.C[at], sum);
      }
      sum = sum_of_16_lanes(sum);
      if (part == 0) c.y[(int64_t)t * c.ld_y + head * c.vdim + channel] = fmaf(Dh, value, sum);
    }
#pragma unroll
    for (int j = 0; j < DT; ++j) held[(part + 16 * j) * 4] = state[j];
    return;
  }
#pragma unroll
  for (int j = 0; j < TW; ++j)
    if (mine(j))
#pragma unroll
      for (int i = 0; i < 4; ++i) slot[(int64_t)(16 * (wave * TW + j) + 4 * g + i) * 4] = S[j][i];
}

template <int DT>
static void launch_head_blocks(hipStream_t stream, const HeadScanCall& c) {
  const int sets = (c.heads / c.groups + HB_HEADS - 1) / HB_HEADS;
  dim3 side(c.groups * sets, c.tokens / HB_TOKENS + c.n_seqs), block(256);
  dim3 walk((unsigned)((c.heads * c.n_seqs + 7) / 8 * 8 * (c.vdim / 16)));
  hipLaunchKernelGGL((head_blocks_kernel<DT>), side, block, 0, stream, c);
  hipLaunchKernelGGL((head_blocks_walk_kernel<DT>), walk, block, 0, stream, c);
}

// Whether blocks are the cheaper way, by what was measured of both as for the keyed scan (linear_attention.hip; R tiles of 16
// state elements).  Measured (us, token by token or in spans / in blocks): 8 heads of 64 x 16, 4,000 tokens 55 / 138, 1,000 25 / 42, 64 tokens 9 / 12;
// 24 of 64 x 64, 4,000 tokens 174 / 125; 32 of 64 x 128, 64 tokens and 31 single ones 29 / 41, 300 and 20 95 / 36, 1,000 and 200 306 / 193.
static bool blocks_pay(const HeadScanCall& c) {
  const float r = c.state / 16, longest = c.max_count;
  const int span = head_span(c);
  const float token = 0.06f + 0.03f * r;
  const float walk = span == 0 ? 3.5f + token * longest
                               : 2.f + 2.f * token * span * span_crowding((int64_t)c.heads * (c.vdim / 4), c.tokens, span) +
                                     (0.45f + 1.6e-5f * c.heads * c.state * c.vdim) * (longest / span);
  const float others = short_sequences(c.tokens, c.n_seqs, c.max_count) * (c.heads * (c.vdim / 16)) * (0.003f + 4e-5f * c.state);
  return 9.f + 0.2f * r + (0.0335f + 0.001f * r) * longest + others < walk;
}

// True if the call went in blocks: it brings the room, tiles of 16 and enough tokens.
static bool head_blocks(hipStream_t stream, const HeadScanCall& c) {
  if (!c.blocks || c.max_count < HB_MIN_TOKENS || c.state % 16 != 0 || c.state > 128 || c.vdim % 16 != 0 || c.tokens / HB_TOKENS + c.n_seqs > 65535 ||
      (int64_t)c.heads * c.n_seqs * (c.vdim / 16) > 1 << 30 || c.groups > 4096 || hb_floats(c) > 1 << 28 || 64 * c.ld > 1 << 30 || !blocks_pay(c))
    return false;
  switch (c.state / 16) {
    case 1: launch_head_blocks<1>(stream, c); break;
    case 2: launch_head_blocks<2>(stream, c); break;
    case 3: launch_head_blocks<3>(stream, c); break;
    case 4: launch_head_blocks<4>(stream, c); break;
    case 5: launch_head_blocks<5>(stream, c); break;
    case 6: launch_head_blocks<6>(stream, c); break;
    case 7: launch_head_blocks<7>(stream, c); break;
    default: launch_head_blocks<8>(stream, c); break;
  }
  return true;
}

BT_EXPORT int bt_head_scan_call(void* stream, const HeadScanCall* c) {
  if (c->tokens <= 0) return BT_OK;
  if (c->heads <= 0 || c->vdim <= 0 || c->state <= 0 || c->state > 256 || c->groups <= 0 || c->heads % c->groups != 0 || c->n_seqs <= 0)
    BT_REFUSE("head_scan: %d heads of %d in %d groups with %d state elements (1..256)", c->heads, c->vdim, c->groups, c->state);
  if (!c->x || !c->B || !c->C || !c->dt_raw || !c->dt_bias || !c->A_log || !c->D || !c->y || !c->S || !c->seq_off || !c->slots)
    BT_REFUSE("head_scan: missing operand");
  if (c->ld_dt < c->heads || c->ld_y < (int64_t)c->heads * c->vdim ||
      c->state_stride < (int64_t)c->heads * c->state * ((c->vdim + 3) / 4 * 4))
    BT_REFUSE("head_scan: rows or state too short for %d heads of %d", c->heads, c->vdim);
  if ((int64_t)c->tokens * c->ld >= (int64_t)1 << 31) BT_REFUSE("head_scan: the rows of B and C are addressed with 32 bits");
  if ((uintptr_t)c->blocks % 16 != 0) BT_REFUSE("head_scan: the room for blocks is not aligned to 16 bytes");
  hipStream_t s = (hipStream_t)stream;
  if (head_blocks(s, *c)) return bt_check_launch("head_scan");
  const int per = (c->state + 15) / 16;
  if (per <= 1) launch_head_scan_r<1>(s, *c);
  else if (per <= 2) launch_head_scan_r<2>(s, *c);
  else if (per <= 4) launch_head_scan_r<4>(s, *c);
  else if (per <= 8) launch_head_scan_r<8>(s, *c);
  else launch_head_scan_r<16>(s, *c);
  return bt_check_launch("head_scan");
}

// ---------------------------------------------------------------------------------------------
// v = y * silu(z); out = v / sqrt(mean(v^2) + eps) * weight, the mean over each of `parts` equal
// parts of the row on its own.
struct GatedNormCall {
  int out_dtype;
  int tokens, channels, parts;
  int out_cols;           // columns of out written: the channels, then zeros
  float eps;
  const float* y;         // [tokens][ld_y]
  int64_t ld_y;
  const float* z;         // [tokens][ld_z] gate, pre-activation
  int64_t ld_z;
  const float* weight;    // [channels]
  void* out;              // [tokens][ld_out]
  int64_t ld_out;
};

template <typename T>
__global__ void __launch_bounds__(256) gated_norm_kernel(GatedNormCall c) {
  extern __shared__ float row_buf[];
  __shared__ __attribute__((aligned(16))) float scratch[32];
  const int t = blockIdx.x, part = blockIdx.y;
  const int n = c.channels / c.parts, base = part * n;
  float partial = 0.f;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const float v = c.y[(int64_t)t * c.ld_y + base + i] * silu_f(c.z[(int64_t)t * c.ld_z + base + i]);
    row_buf[i] = v;
    partial += v * v;
  }
  const float rstd = 1.0f / sqrtf(block_sum<256>(partial, scratch) / (float)n + c.eps);
  T* out = static_cast<T*>(c.out) + (int64_t)t * c.ld_out;
  for (int i = threadIdx.x; i < n; i += blockDim.x) out[base + i] = from_float<T>(row_buf[i] * rstd * c.weight[base + i]);
  if (part == 0)
    for (int col = c.channels + threadIdx.x; col < c.out_cols; col += blockDim.x) out[col] = from_float<T>(0.f);
}

BT_EXPORT int bt_gated_norm_call(void* stream, const GatedNormCall* c) {
  if (c->tokens <= 0) return BT_OK;
  if (c->channels <= 0 || c->parts <= 0 || c->channels % c->parts != 0 || c->channels / c->parts > 15360)
    BT_REFUSE("gated_norm: %d channels in %d equal parts (each up to 15360)", c->channels, c->parts);
  if (!c->y || !c->z || !c->weight || !c->out || c->ld_y < c->channels || c->ld_z < c->channels ||
      c->out_cols < c->channels || c->ld_out < c->out_cols)
    BT_REFUSE("gated_norm: missing operand or rows too short");
  dim3 grid(c->tokens, c->parts), block(256);
  size_t lds = (size_t)(c->channels / c->parts) * sizeof(float);
  if (c->out_dtype == 0)
    hipLaunchKernelGGL(gated_norm_kernel<float>, grid, block, lds, (hipStream_t)stream, *c);
  else
    hipLaunchKernelGGL(gated_norm_kernel<bf16_t>, grid, block, lds, (hipStream_t)stream, *c);
  return bt_check_launch("gated_norm");
}
