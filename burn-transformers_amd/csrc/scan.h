// Helpers shared by the kernels that walk a sequence's tokens in order with a state in registers.
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"

// Sums over groups of 8 or 16 neighbouring lanes with data-parallel moves between lanes of a row
// (no trip through the LDS crossbar as a shuffle takes; a recurrence pays this once per token): first
// within quads (swap neighbours, swap pairs: then every lane of a quad holds the quad's sum), then
// the mirror image within half a row pairs the two quads of eight lanes, then the mirror image within
// the row pairs its halves.  Every lane of the group ends with the group's sum.
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ float sum_of_8_lanes(float v) {
  v += dpp_move<0xB1>(v);     // quad_perm [1, 0, 3, 2]
  v += dpp_move<0x4E>(v);     // quad_perm [2, 3, 0, 1]
  v += dpp_move<0x141>(v);    // row_half_mirror
  return v;
}
__device__ __forceinline__ float sum_of_16_lanes(float v) {
  v = sum_of_8_lanes(v);
  v += dpp_move<0x140>(v);    // row_mirror
  return v;
}

// A barrier that waits for this wave's LDS traffic only: operands asked for blocks ahead stay on their way.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);                      // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Waits for values that a loop with loads on their way starts from: asked for behind those, they would be waited for, and the loads
// with them, in every turn (the compiler's wait is the same for all).
template <int N>
__device__ __forceinline__ void landed(floatx4 (&values)[N]) {
#pragma unroll
  for (int j = 0; j < N; ++j) asm volatile("" : "+v"(values[j]));
}

template <int N>
struct Number {
  static constexpr int value = N;
};

// f(Number<0>()) .. f(Number<N - 1>()): steps whose numbers choose code.
template <int N, int FROM = 0, typename F>
__device__ __forceinline__ void each(F&& f) {
  if constexpr (FROM < N) {
    f(Number<FROM>());
    each<N, FROM + 1>(f);
  }
}

__device__ __forceinline__ float silu_f(float v) { return v / (1.0f + expf(-v)); }
__device__ __forceinline__ float softplus_f(float v) { return v > 20.0f ? v : log1pf(expf(v)); }

// Tokens of a run: as many as keep a work-group's LDS at about 24 KiB, at most 64, no more than the step has.
static int scan_chunk(int floats_per_token, int tokens) {
  int chunk = 6144 / floats_per_token;
  chunk = chunk < 1 ? 1 : chunk > 64 ? 64 : chunk;
  return chunk < tokens ? chunk : tokens;
}


// Spans.  A recurrence S_t = a_t S_(t-1) + u_t is linear in S, so a long sequence need not be walked
// by one wave: cut into spans of `span` tokens, (1) every span is scanned from a zero state, side by
// side, and leaves its end state E_k and the sum of its step sizes (its decays multiply up to
// P_k = exp(A * that sum)); (2) a short kernel carries the state across the spans in order,
// C_k = P_k C_(k-1) + E_k, from the slot's state; (3) every span is scanned again, side by side, from
// the state C_(k-1) it really starts with, and writes the outputs.  The carrying kernel also keeps the
// state the sequence came with (as "span -1": the third pass reads only the carry, never the slot, which
// by then holds the state after the sequence's last token, written by the carrying kernel).  Twice the
// arithmetic, on (sequence length / span) times the waves.  Span k of sequence s keeps its block at
// index seq_off[s] / span + 2 s + 1 + k: ranges of different sequences do not meet.
__device__ __forceinline__ int64_t span_block(const int* seq_off, int seq, int span, int part) {
  return (int64_t)(seq_off[seq] / span + 2 * seq + 1 + part);
}

// Pieces of `size` tokens that are worked on side by side are numbered through the step, a sequence's behind those of the ones
// before it: there are at most tokens / size + n_seqs of them, whatever its sequences bring (a grid of the longest
// sequence's pieces for every sequence is mostly empty where a prompt comes beside single tokens: of 500 and 63 x 1 tokens with
// 8 heads 16,384 work-groups for 784, and the keyed scan took 256 us for 62).  Where all sequences are alike the sequence of a
// number is a quotient, elsewhere a wave finds it, 64 sequences at a time; `part` is the piece.  Numbers behind the last piece have no
// sequence (-1): they come last, so that the others are dealt evenly to the compute units (empty ones among them cost the
// selective scan a fifth).
__device__ __forceinline__ int piece_sequence(const int* seq_off, int n_seqs, int tokens, int longest, int size, int number, int& part) {
  if ((int64_t)n_seqs * longest == tokens) {
    const int pieces = (longest + size - 1) / size, seq = number / pieces;
    part = number - seq * pieces;
    return seq < n_seqs ? seq : -1;
  }
  const int lane = threadIdx.x & 63;
  for (int s0 = 0; s0 < n_seqs; s0 += 64) {
    const int s = s0 + lane, pieces = s < n_seqs ? (seq_off[s + 1] - seq_off[s] + size - 1) / size : 0;
    int upto = pieces;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int before = __shfl_up(upto, o, 64);
      upto += lane >= o ? before : 0;
    }
    const unsigned long long reached = __builtin_amdgcn_ballot_w64(upto > number);
    if (reached != 0) {
      const int first = __builtin_ctzll(reached);
      part = number - (__builtin_amdgcn_readlane(upto, first) - __builtin_amdgcn_readlane(pieces, first));
      return s0 + first;
    }
    number -= __builtin_amdgcn_readlane(upto, 63);
  }
  return -1;
}

// Sequences of at least this many spans are cut (fewer gain nothing over walking them).
#define MIN_SPANS 3

static int simd_count() {
  static int count = 0;
  if (count == 0) {
    int device = 0, units = 0;
    if (hipGetDevice(&device) != hipSuccess ||
        hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || units <= 0)
      units = 256;
    count = 4 * units;
  }
  return count;
}

// Into spans of how many tokens a step's long sequences are cut, 0 for not at all.  Spans double the
// arithmetic, so they pay only while whole sequences leave the chip short of waves: `waves` (those that
// walk whole sequences) must be at most `fill` to a SIMD, and there are as many spans as bring `times`
// that, none shorter than the call's `span`, which its room for the spans' states was sized
// for.  Measured for 2 x 1,024 tokens (us, whole / cut): the head scan with one wave to a SIMD 309 / 205,
// with two 327 / 380; the selective scan with half a wave to a SIMD 334 / 176, with one 369 / 311.
static int span_tokens(int span, int max_count, const float* carry, int64_t waves, int fill, int times = 4) {
  if (span <= 0 || !carry || waves > (int64_t)fill * simd_count()) return 0;
  const int64_t wanted = times * (int64_t)fill * simd_count() / waves;
  int tokens = (int)((max_count + wanted - 1) / wanted);
  if (tokens < span) tokens = span;
  return max_count >= MIN_SPANS * tokens ? tokens : 0;
}

// What a token of a span costs beside one of a wave alone on its SIMD, with `waves` walking a sequence: spans bring up to four
// times `fill` to a SIMD, which then share it (measured: four take 1.6 to 2 times as long as one).
static float span_crowding(int64_t waves, int tokens, int span) {
  const float on_a_simd = (float)waves * tokens / span / simd_count();
  return on_a_simd > 1.f ? 1.f + 0.2f * (on_a_simd - 1.f) : 1.f;
}

// How many sequences of a step it holds beyond those that would bring its tokens at the longest one's length: none where all are
// alike, all but one where a prompt comes beside single tokens.
static int64_t short_sequences(int tokens, int n_seqs, int max_count) {
  const int64_t alike = ((int64_t)tokens + max_count - 1) / max_count;
  return n_seqs > alike ? n_seqs - alike : 0;
}

