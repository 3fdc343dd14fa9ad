// What a matrix product does with its accumulators: it adds the bias and then either stores, applies the
// activation, writes 32-bit partial sums, or scatters a fused query/key/value projection into the query
// buffer and the paged cache.  The skinny kernel hands 1, 2 or 4 neighbouring columns of a row to `epilogue_values`,
// the plain and small tile kernels four to `epilogue4`, those whose tiles leave through LDS a whole tile to `epilogue_tile`.
#pragma once

#include "common.h"

enum EpilogueMode {
  EPI_STORE = 0,  // out[m][n] = acc + bias                      (element type T)
  EPI_ACT = 1,    // out[m][n] = act(acc + bias)                 (element type T)
  EPI_F32 = 2,    // out[split][m][n] = acc (+ bias in split 0)  (float; the consumer sums the splits)
  EPI_QKV = 3,    // columns [0,n_q) -> out, [n_q,n_q+n_kv) -> keys, the next n_kv -> values
  EPI_RESIDUAL = 4,  // out[m][n] += acc + bias                  (float: the residual stream itself)
  EPI_F32_ACT = 5,   // columns [0,n_q) -> out as in EPI_F32, those behind -> act(acc + bias) in out2 (element type T), columns
                     //   from 0: two products of the same rows as one (the skinny kernel only)
  EPI_TURN = 6,      // out[m][n] = acc, of every turn.pitch columns the turn.dim from turn.at on rotated in neighbouring pairs
                     //   by the row's position (element type T; the skinny kernel only)
};
// What the skinny kernel is built for: the common modes, or one of the three that are forms of the kernel of their own.
enum EpilogueKind { EPILOGUE_COMMON = 0, EPILOGUE_TWO = 1, EPILOGUE_TURN = 2, EPILOGUE_QKV = 3 };

enum Activation {
  ACT_GELU_TANH = 0,
  ACT_GELU_ERF = 1,
  ACT_SQUARED_RELU = 2,
};

// EPI_TURN: columns at + 2 i and at + 2 i + 1 of a head of `pitch` columns (a multiple of four; at and dim even) turn by the
// angle tok_pos[m] * inv_freq[i], sine and cosine times `amplitude`.
struct TurnedColumns {
  const float* inv_freq;
  int pitch, at, dim;
  float amplitude;
};

// Mirrored field by field by a ctypes.Structure on the Python side.
struct Epilogue {
  int mode;
  int act;
  const float* bias;     // [N] or null
  void* out;
  int64_t ldo;           // row pitch of out, in elements
  int64_t split_stride;  // elements between the partial sums of two splits (EPI_F32)
  int n_q;
  int n_kv;
  const int* tok_seq;    // [M] index of the token's sequence in the step
  const int* tok_pos;    // [M] position of the token in its sequence
  union {                // (together: every kernel's arguments are as short as they were without the second)
    KvView kv;           // EPI_QKV
    TurnedColumns turn;  // EPI_TURN
  };
  int out_rows;          // EPI_STORE, EPI_ACT (EPI_F32_ACT: `out2`): 0, or `out` is chunk-major with that many rows (activation_offset)
  void* out2;            // EPI_F32_ACT only
  int64_t ldo2;
};

// 32-bit activations.  The float32 path (T = float) uses the library's tanhf / erff; the
// bfloat16 path writes the tanh form as x / (1 + exp(-2u)), which is the same function
// (0.5 (1 + tanh u) = 1 / (1 + exp(-2u))) evaluated with the hardware exponential: its error
// (a few ulp of float32) is far below the rounding of the bfloat16 result, and it is a handful of
// instructions instead of some forty for each of the millions of elements a prefill produces.
template <typename T, int ACT>
__device__ __forceinline__ float activate_as(float x) {
  if constexpr (ACT == ACT_GELU_TANH) {
    // 0.5 x (1 + tanh(sqrt(2/pi) (x + 0.044715 x^3)))
    float inner = 0.7978845608028654f * (x + 0.044715f * x * x * x);
    if (sizeof(T) == 2) return x / (1.0f + __expf(-2.0f * inner));
    return 0.5f * x * (1.0f + tanhf(inner));
  } else if constexpr (ACT == ACT_SQUARED_RELU) {
    return x > 0.f ? x * x : 0.f;
  } else {
    // x (1 + erf(x / sqrt 2)) / 2
    return 0.5f * x * (1.0f + erff(x * 0.7071067811865476f));
  }
}
template <typename T>
__device__ __forceinline__ float activate(float x, int act) {
  return act == ACT_GELU_TANH ? activate_as<T, ACT_GELU_TANH>(x) : act == ACT_SQUARED_RELU ? activate_as<T, ACT_SQUARED_RELU>(x)
                                                                                            : activate_as<T, ACT_GELU_ERF>(x);
}

template <typename T>
__device__ __forceinline__ void store4(T* dst, const float* v, int count, bool aligned);

template <>
__device__ __forceinline__ void store4<float>(float* dst, const float* v, int count, bool aligned) {
  if (count == 4 && aligned) {
    *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < count) dst[i] = v[i];
  }
}
template <>
__device__ __forceinline__ void store4<bf16_t>(bf16_t* dst, const float* v, int count, bool aligned) {
  if (count == 4 && aligned) {
    bf16x4 packed = {(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
    *reinterpret_cast<bf16x4*>(dst) = packed;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < count) dst[i] = (bf16_t)v[i];
  }
}

// What the skinny kernel's epilogue adds to the sums of neighbouring columns: the bias, and in EPI_RESIDUAL the old values of the
// residual stream.
template <int KIND, int VALUES>
__device__ __forceinline__ void epilogue_addends(const Epilogue& e, int M, int n_end, int m, int n0, int split, float (&add)[VALUES]) {
#pragma unroll
  for (int i = 0; i < VALUES; ++i) add[i] = 0.f;
  if (KIND == EPILOGUE_TURN) return;
  int n[VALUES];                            // (values beyond the rows or columns are dropped)
#pragma unroll
  for (int i = 0; i < VALUES; ++i) n[i] = n0 + i < n_end ? n0 + i : n_end - 1;
  if (e.bias != nullptr && split == 0) {
#pragma unroll
    for (int i = 0; i < VALUES; ++i) add[i] = e.bias[n[i]];
  }
  if (KIND == EPILOGUE_COMMON && e.mode == EPI_RESIDUAL) {
    const float* x = static_cast<const float*>(e.out) + (int64_t)(m < M ? m : M - 1) * e.ldo;
#pragma unroll
    for (int i = 0; i < VALUES; ++i) add[i] += x[n[i]];
  }
}

// What the skinny kernel's epilogue looks up in the step's tables, of up to 16 * MT rows (and 16 * NT columns).  As vector loads of
// the waves that stream, the lookups, which depend on each other, would wait for all the weights before them (loads return in order): a second
// round trip to memory behind every product.  For forms of one column block a ninth wave, which multiplies nothing, does it meanwhile (`fill`; of
// turned columns up to sixteen rows, more sines than that take one wave too long).  Nine waves put three on one SIMD, which leaves them 168
// registers each, and room for two work-groups a compute unit only up to 96.  The forms of two column blocks have neither, nor that of two row blocks and
// eight chunks the latter, so there every streaming wave takes a share: places of tokens through the scalar cache (TokenPlaces), sines of its own values (TurnedPairs).  Measured (us, a ninth wave in all
// forms / so): 4800 x 1600 into the cache, one row with a norm 7.9 / 6.3, 24 rows 12.5 / 8.1; 9216 x 3072, eight rows 16.0 / 14.5, 24 rows in 16 columns 29.3 / 26.9; turned 10240 x 1536, 24 rows 20.9 /
// 13.3, 2560 x 768, 64 rows 7.5 / 6.3.  The streaming waves' share in all forms: 2304 x 768 with a norm 3.8 -> 4.0, 1280 x 384 turned 2.7 -> 3.4.
// A share of the rows' places:
template <int ROWS, int WAVES>
struct TokenPlaces {
  static constexpr int SHARE = ROWS / WAVES;
  int pos[SHARE], seq[SHARE], block[SHARE];
  __device__ __forceinline__ void ask(const Epilogue& e, int M, int wave) {
    const int first = wave * SHARE;
    if (first + SHARE <= M) {               // (neighbours, in one load: a load a row, 64 rows of 4800 x 1600 10.3 us, so 10.2)
#pragma unroll
      for (int i = 0; i < SHARE; ++i) {
        pos[i] = e.tok_pos[first + i];
        seq[i] = e.tok_seq[first + i];
      }
    } else {
#pragma unroll
      for (int i = 0; i < SHARE; ++i) {     // (rows beyond M repeat the last)
        const int m = first + i < M ? first + i : M - 1;
        pos[i] = e.tok_pos[m];
        seq[i] = e.tok_seq[m];
      }
    }
  }
  __device__ __forceinline__ void look(const Epilogue& e) {
#pragma unroll
    for (int i = 0; i < SHARE; ++i) block[i] = e.kv.blocks[(int64_t)seq[i] * e.kv.max_blocks + pos[i] / BT_KV_BLOCK];
  }
  // (a lane a row; eight rows one after the other, with the planes worked out here, took 0.2 us longer at 64 rows of 4800 x 1600)
  template <typename Tables>
  __device__ __forceinline__ void put(int wave, Tables& tables) const {
    const int lane = threadIdx.x & 63;
    int2 mine = {0, 0};
#pragma unroll
    for (int i = 0; i < SHARE; ++i) mine = lane == i ? make_int2(block[i], pos[i]) : mine;
    if (lane < SHARE) tables.place[wave * SHARE + lane] = mine;
  }
};
template <int KIND, int MT, int NT>
struct EpilogueTables {};     // (the other kinds need none)
template <int MT, int NT>
struct EpilogueTables<EPILOGUE_QKV, MT, NT> {
  int2 place[16 * MT];        // the block of the row's token and its position
  __device__ __forceinline__ void fill(const Epilogue& e, int M, int) {
    const int m = threadIdx.x & 63;
    if (m < M) {
      const int pos = e.tok_pos[m], seq = e.tok_seq[m];
      place[m] = make_int2(e.kv.blocks[(int64_t)seq * e.kv.max_blocks + pos / BT_KV_BLOCK], pos);
    }
  }
};
template <int MT, int NT>
struct EpilogueTables<EPILOGUE_TURN, MT, NT> {
  float2 turn[16 * MT][8 * NT];      // cosine and sine of a row's pair of columns
  __device__ __forceinline__ void fill(const Epilogue& e, int M, int n_base) {
    for (int at = threadIdx.x & 63; at < M * 8 * NT; at += 64) {
      const int m = at / (8 * NT), pair = at % (8 * NT);
      const int j = (n_base + 2 * pair) % e.turn.pitch - e.turn.at;
      const bool turned = j >= 0 && j < e.turn.dim;
      float sn = 0.f, cs = 1.f;
      const float f = turned ? e.turn.inv_freq[j >> 1] : 0.f;
      if (f != 0.f) sincosf((float)e.tok_pos[m] * f, &sn, &cs);
      turn[m][pair] = make_float2(cs, sn);
    }
  }
};
// The sines of a thread's own values: asked for behind the first batch of weights, worked out behind the products.
template <int VALUES>
struct TurnedPairs {
  static constexpr int PAIRS = (VALUES + 1) / 2;
  int pos;
  float f[PAIRS];
  float2 turn[PAIRS];
  __device__ __forceinline__ void ask(const Epilogue& e, int M, int m, int n0) {
    pos = e.tok_pos[m < M ? m : M - 1];
    const int j = n0 % e.turn.pitch - e.turn.at;       // (of an odd column the pair is the even one's)
#pragma unroll
    for (int p = 0; p < PAIRS; ++p) {
      const bool turned = j + 2 * p >= 0 && j + 2 * p < e.turn.dim;
      const float there = e.turn.inv_freq[turned ? (j + 2 * p) >> 1 : 0];
      f[p] = turned ? there : 0.f;
    }
  }
  __device__ __forceinline__ void work() {
#pragma unroll
    for (int p = 0; p < PAIRS; ++p) {
      float sn = 0.f, cs = 1.f;
      if (f[p] != 0.f) sincosf((float)pos * f[p], &sn, &cs);
      turn[p] = make_float2(cs, sn);
    }
  }
};

// Stores of neighbours: together where all are inside and the place is aligned.
template <typename T, int VALUES>
__device__ __forceinline__ void store_values(T* dst, const float (&v)[VALUES], int count) {
  typedef __attribute__((__vector_size__(VALUES * sizeof(T)))) T Ts;
  if (VALUES > 1 && count >= VALUES && ((uintptr_t)dst & (VALUES * sizeof(T) - 1)) == 0) {
    Ts all;
#pragma unroll
    for (int i = 0; i < VALUES; ++i) all[i] = from_float<T>(v[i]);
    *reinterpret_cast<Ts*>(dst) = all;
  } else {
#pragma unroll
    for (int i = 0; i < VALUES; ++i)
      if (i < count) dst[i] = from_float<T>(v[i]);
  }
}

// The skinny kernel's epilogue for VALUES neighbouring columns of a row, inside four: v are the sums with what is added to them,
// column is n0 inside the work-group.  One value a lane with up to sixteen rows: a wave that takes four of each lane has most of
// its lanes idle then, and the longer chain behind the last barrier showed in every product (0.3 us, with a GELU 0.7, of 2.7 and 3.7).
// tables: EpilogueTables; turn: what the values' pairs turn by.
template <typename T, int KIND, int VALUES, typename Tables>
__device__ __forceinline__ void epilogue_values(const Epilogue& e, int N, int m, int n0, int column, float (&v)[VALUES], int split,
                                                const Tables& tables, const float2* turn) {
  const int count = N - n0;
  if constexpr (KIND == EPILOGUE_TURN) {    // (pairs of columns are one lane's or two neighbours'; N is whole pairs)
    float y[VALUES];
#pragma unroll
    for (int i = 0; i < VALUES; ++i) {
      const float other = VALUES == 1 ? lane_moved<0xb1>(v[i]) : v[VALUES == 1 ? i : i ^ 1];
      const int j = (n0 + i) % e.turn.pitch - e.turn.at;
      const float2 t = turn[i >> 1];
      const float amplitude = j >= 0 && j < e.turn.dim ? e.turn.amplitude : 1.f;
      const bool odd = (column + i) & 1;
      y[i] = amplitude * fmaf(odd ? other : v[i], odd ? t.y : t.x, odd ? v[i] * t.x : -(other * t.y));
    }
    if (count > 0) store_values<T, VALUES>(static_cast<T*>(e.out) + (int64_t)m * e.ldo + n0, y, count);
    return;
  }
  if (count <= 0) return;
  if constexpr (KIND == EPILOGUE_TWO) {
    if (n0 < e.n_q) {                       // (n_q is a multiple of four)
      store_values<float, VALUES>(static_cast<float*>(e.out) + (int64_t)m * e.ldo + n0, v, count);
    } else {
#pragma unroll
      for (int i = 0; i < VALUES; ++i) v[i] = activate<T>(v[i], e.act);
      store_values<T, VALUES>(static_cast<T*>(e.out2) + activation_offset<T>(e.out_rows, e.ldo2, m, n0 - e.n_q), v, count);
    }
  } else if constexpr (KIND == EPILOGUE_QKV) {
    if (n0 < e.n_q) {
      store_values<T, VALUES>(static_cast<T*>(e.out) + (int64_t)m * e.ldo + n0, v, count);
    } else {                                // (queries, keys, values and heads are multiples of sixteen columns)
      int c = n0 - e.n_q;
      const bool is_value = c >= e.n_kv;
      if (is_value) c -= e.n_kv;
      const int head = c / e.kv.head_dim, channel = c % e.kv.head_dim;
      const int2 place = tables.place[m];
      const int64_t base = kv_plane(e.kv, place.x, head);
      const int pos = place.y;
      if (!is_value) {
        store_values<T, VALUES>(static_cast<T*>(e.kv.keys) + base + key_offset(e.kv.head_dim, pos, channel), v, count);
      } else {
        T* dst = static_cast<T*>(e.kv.values) + base + value_offset(e.kv.head_dim, pos, channel);
#pragma unroll
        for (int i = 0; i < VALUES; ++i)    // consecutive channels of one position lie four elements apart
          if (i < count) dst[4 * i] = from_float<T>(v[i]);
      }
    }
  } else if (e.mode == EPI_STORE || e.mode == EPI_ACT) {
    if (e.mode == EPI_ACT) {
#pragma unroll
      for (int i = 0; i < VALUES; ++i) v[i] = activate<T>(v[i], e.act);
    }
    store_values<T, VALUES>(static_cast<T*>(e.out) + activation_offset<T>(e.out_rows, e.ldo, m, n0), v, count);
  } else {                                  // EPI_F32, EPI_RESIDUAL (whose products are not split)
    store_values<float, VALUES>(static_cast<float*>(e.out) + (e.mode == EPI_F32 ? (int64_t)split * e.split_stride : 0) + (int64_t)m * e.ldo + n0, v,
                                count);
  }
}

// Row m, columns n0 .. n0+3 (n0 a multiple of four), of an [M, N] product; `split` is the
// index of the K slice that produced `acc`.
template <typename T>
__device__ __forceinline__ void epilogue4(const Epilogue& e, int N, int m, int n0, const float* acc,
                                          int split) {
  int count = N - n0 < 4 ? N - n0 : 4;
  if (count <= 0) return;
  float v[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float b = (e.bias != nullptr && split == 0 && i < count) ? e.bias[n0 + i] : 0.f;
    v[i] = acc[i] + b;
  }
  bool aligned = (e.ldo & 3) == 0;
  if (e.mode == EPI_STORE) {
    if (e.out_rows == 0) store4<T>(static_cast<T*>(e.out) + (int64_t)m * e.ldo + n0, v, count, aligned);     // (one branch for all threads)
    else store4<T>(static_cast<T*>(e.out) + activation_offset<T>(e.out_rows, e.ldo, m, n0), v, count, true);
  } else if (e.mode == EPI_ACT) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = activate<T>(v[i], e.act);
    if (e.out_rows == 0) store4<T>(static_cast<T*>(e.out) + (int64_t)m * e.ldo + n0, v, count, aligned);     // (one branch for all threads)
    else store4<T>(static_cast<T*>(e.out) + activation_offset<T>(e.out_rows, e.ldo, m, n0), v, count, true);
  } else if (e.mode == EPI_F32) {
    store4<float>(static_cast<float*>(e.out) + (int64_t)split * e.split_stride + (int64_t)m * e.ldo + n0,
                  v, count, aligned);
  } else if (e.mode == EPI_RESIDUAL) {
    float* x = static_cast<float*>(e.out) + (int64_t)m * e.ldo + n0;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < count) v[i] += x[i];
    store4<float>(x, v, count, aligned);
#ifdef BT_EPILOGUE_ANY_HEAD_SIZE
  } else if ((e.kv.head_dim & 3) != 0) {
    // EPI_QKV with a head size that four columns do not divide: every column finds its own place
    // among the queries, keys and values.  Compiled into the plain product only (it defines
    // BT_EPILOGUE_ANY_HEAD_SIZE): the MFMA kernels refuse such head sizes, and in them this path
    // would only cost registers (their tiles of 128 x 128 spilled with it, at a third of the speed).
    int seq = e.tok_seq[m], pos = e.tok_pos[m];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (i >= count) break;
      int n = n0 + i;
      if (n < e.n_q) {
        static_cast<T*>(e.out)[(int64_t)m * e.ldo + n] = from_float<T>(v[i]);
        continue;
      }
      int c = n - e.n_q;
      bool is_value = c >= e.n_kv;
      if (is_value) c -= e.n_kv;
      int head = c / e.kv.head_dim, channel = c % e.kv.head_dim;
      int64_t base = kv_block_base(e.kv, seq, pos, head);
      if (!is_value) static_cast<T*>(e.kv.keys)[base + key_offset(e.kv.head_dim, pos, channel)] = from_float<T>(v[i]);
      else static_cast<T*>(e.kv.values)[base + value_offset(e.kv.head_dim, pos, channel)] = from_float<T>(v[i]);
    }
#endif
  } else {  // EPI_QKV: head_dim (and with it n_q and n_kv) is a multiple of four, so the four columns share a head
    if (n0 < e.n_q) {
      store4<T>(static_cast<T*>(e.out) + (int64_t)m * e.ldo + n0, v, count, aligned);
    } else {
      int c = n0 - e.n_q;
      bool is_value = c >= e.n_kv;
      if (is_value) c -= e.n_kv;
      int head = c / e.kv.head_dim, channel = c % e.kv.head_dim;
      int seq = e.tok_seq[m], pos = e.tok_pos[m];
      int64_t base = kv_block_base(e.kv, seq, pos, head);
      if (!is_value) {
        store4<T>(static_cast<T*>(e.kv.keys) + base + key_offset(e.kv.head_dim, pos, channel), v, count,
                  true);
      } else {
        T* dst = static_cast<T*>(e.kv.values) + base + value_offset(e.kv.head_dim, pos, channel);
#pragma unroll
        for (int i = 0; i < 4; ++i)     // consecutive channels of one position lie four elements apart
          if (i < count) dst[4 * i] = from_float<T>(v[i]);
      }
    }
  }
}

// The epilogue of a whole wave's TM x TN blocks of 32 x 32 (lane holds D[i][j]: i = 8 (r / 4) + 4 g + r % 4 the column, j = lane
// % 32 the row): through LDS, so that memory sees whole rows' 16-byte pieces instead of 32 rows' 8 bytes with every
// instruction, and with all that a step needs from memory asked for together.  One call of epilogue4 after the other took 5 us
// (stored rows) to 12 us (the residual stream, whose old values every call waited for) of a product of 128 x 128 tiles.
// `scratch`: tile_scratch_bytes<TM, TN>() of this wave's own; every wave has passed a barrier behind its last read of it.
template <int TM, int TN>
constexpr int tile_scratch_bytes() { return TM * 32 * (TN * 32 * 4 + 16); }

template <typename T, int TM, int TN>
__device__ __forceinline__ void epilogue_tile(const Epilogue& e, int M, int N, int m0, int n0, floatx16 (&acc)[TN][TM], int split,
                                              unsigned char* scratch) {
  const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
  constexpr int COLUMNS = TN * 32, ROWS = TM * 32;
  const bool f32 = sizeof(T) == 4 || e.mode == EPI_F32 || e.mode == EPI_RESIDUAL;
  const int piece = f32 ? 4 : 8;                       // values in 16 bytes
  // key/value columns: the wave's columns are all queries, or all keys or all values of one head
  const int kv_column = n0 - e.n_q, kv_last = kv_column + COLUMNS - 1;
  const bool scatter = e.mode == EPI_QKV && kv_column >= 0 && kv_last < 2 * e.n_kv && kv_column / e.kv.head_dim == kv_last / e.kv.head_dim &&
                       kv_column / e.n_kv == kv_last / e.n_kv && (e.kv.head_dim & 7) == 0 && (((uintptr_t)e.kv.keys | (uintptr_t)e.kv.values) & 15) == 0;
  const bool values = scatter && kv_column >= e.n_kv, keys = scatter && !values;
  const bool whole = (e.mode != EPI_QKV || n0 + COLUMNS <= e.n_q || scatter) && e.out_rows == 0 && N % piece == 0 && e.ldo % piece == 0 &&
                     e.split_stride % piece == 0 && (((uintptr_t)e.out | (uintptr_t)e.bias) & 15) == 0;
  auto spread = [&](auto element) {                    // the wave's rows into LDS
    typedef decltype(element) E;
    constexpr int PITCH = COLUMNS * (int)sizeof(E) + 16;
#pragma unroll
    for (int bm = 0; bm < TM; ++bm)
#pragma unroll
      for (int bn = 0; bn < TN; ++bn)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float v[4] = {acc[bn][bm][4 * q], acc[bn][bm][4 * q + 1], acc[bn][bm][4 * q + 2], acc[bn][bm][4 * q + 3]};
          store4<E>(reinterpret_cast<E*>(scratch + (bm * 32 + l32) * PITCH) + bn * 32 + q * 8 + g * 4, v, 4, true);
        }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");       // (a wave's accesses of LDS are served in order)
  };
  if (!whole) {                                        // (the same for the whole wave)
    spread(0.f);
#pragma nounroll
    for (int i = lane; i < ROWS * COLUMNS / 4; i += 64) {
      const int r = i / (COLUMNS / 4), c = i % (COLUMNS / 4) * 4;
      const floatx4 row = *reinterpret_cast<const floatx4*>(scratch + r * (COLUMNS * 4 + 16) + c * 4);
      const float v[4] = {row[0], row[1], row[2], row[3]};
      if (m0 + r < M) epilogue4<T>(e, N, m0 + r, n0 + c, v, split);
    }
    return;
  }
  if (e.bias != nullptr && split == 0) {
    floatx4 b[TN][4];
#pragma unroll
    for (int bn = 0; bn < TN; ++bn)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = n0 + bn * 32 + q * 8 + g * 4;
        b[bn][q] = *reinterpret_cast<const floatx4*>(e.bias + (n < N ? n : 0));
      }
#pragma unroll
    for (int bn = 0; bn < TN; ++bn)
#pragma unroll
      for (int bm = 0; bm < TM; ++bm)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[bn][bm][r] += b[bn][r >> 2][r & 3];
  }
  if (e.mode == EPI_ACT) {
    // (one choice for all values: with the choice at every value the code of every activation lay between each two of them, 64 KiB
    // for 128 x 256, and fetching it took 2.6 to 5 us of a work-group's epilogue)
    auto all = [&](auto act) {
#pragma unroll
      for (int bn = 0; bn < TN; ++bn)
#pragma unroll
        for (int bm = 0; bm < TM; ++bm)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[bn][bm][r] = activate_as<T, decltype(act)::value>(acc[bn][bm][r]);
    };
    if (e.act == ACT_GELU_TANH) all(Constant<ACT_GELU_TANH>());
    else if (e.act == ACT_SQUARED_RELU) all(Constant<ACT_SQUARED_RELU>());
    else all(Constant<ACT_GELU_ERF>());
  }
  if (values) {          // four positions lie interleaved: every lane stores its own row's channels, 8 bytes of a line for four rows
    const int c = kv_column - e.n_kv, head = c / e.kv.head_dim;
    int seq[TM], pos[TM];
    T* plane[TM];
#pragma unroll
    for (int bm = 0; bm < TM; ++bm) {
      const int m = m0 + bm * 32 + l32 < M ? m0 + bm * 32 + l32 : M - 1;
      seq[bm] = e.tok_seq[m];
      pos[bm] = e.tok_pos[m];
    }
#pragma unroll
    for (int bm = 0; bm < TM; ++bm)
      plane[bm] = static_cast<T*>(e.kv.values) + kv_block_base(e.kv, seq[bm], pos[bm], head) + value_offset(e.kv.head_dim, pos[bm], c % e.kv.head_dim + 4 * g);
#pragma unroll
    for (int bm = 0; bm < TM; ++bm) {
      if (m0 + bm * 32 + l32 >= M) continue;
#pragma unroll
      for (int bn = 0; bn < TN; ++bn)
#pragma unroll
        for (int r = 0; r < 16; ++r) plane[bm][4 * (bn * 32 + 8 * (r >> 2) + (r & 3))] = from_float<T>(acc[bn][bm][r]);
    }
    return;
  }
  auto exchange = [&](auto element) {
    typedef decltype(element) E;
    constexpr int PIECE = 16 / (int)sizeof(E), LANES = COLUMNS / PIECE, TURNS = ROWS * LANES / 64;   // lanes a row, pieces a lane
    constexpr int PITCH = COLUMNS * (int)sizeof(E) + 16;
    const int n = n0 + lane % LANES * PIECE;
    E* row[TURNS];
    floatx4 old[TURNS];
    int seq[TURNS], pos[TURNS];
    if (keys) {
#pragma unroll
      for (int t = 0; t < TURNS; ++t) {
        int m = m0 + (64 / LANES) * t + lane / LANES;
        m = m < M ? m : M - 1;
        seq[t] = e.tok_seq[m];
        pos[t] = e.tok_pos[m];
      }
    }
#pragma unroll
    for (int t = 0; t < TURNS; ++t) {
      int m = m0 + (64 / LANES) * t + lane / LANES;
      m = m < M ? m : M - 1;
      if (keys) {
        const int c = n - e.n_q;
        row[t] = static_cast<E*>(e.kv.keys) + kv_block_base(e.kv, seq[t], pos[t], c / e.kv.head_dim) + key_offset(e.kv.head_dim, pos[t], c % e.kv.head_dim);
      } else {
        row[t] = static_cast<E*>(e.out) + (e.mode == EPI_F32 ? (int64_t)split * e.split_stride : 0) + (int64_t)m * e.ldo + (n < N ? n : 0);
      }
      if constexpr (sizeof(E) == 4)
        if (e.mode == EPI_RESIDUAL) old[t] = *reinterpret_cast<const floatx4*>(row[t]);
    }
    spread(element);
#pragma unroll
    for (int t = 0; t < TURNS; ++t) {
      const int r = (64 / LANES) * t + lane / LANES;
      int4v v = *reinterpret_cast<const int4v*>(scratch + r * PITCH + lane % LANES * 16);
      if constexpr (sizeof(E) == 4)
        if (e.mode == EPI_RESIDUAL) v = __builtin_bit_cast(int4v, __builtin_bit_cast(floatx4, v) + old[t]);
      if (m0 + r < M && n < N) *reinterpret_cast<int4v*>(row[t]) = v;
    }
  };
  if constexpr (sizeof(T) == 4) {
    exchange(0.f);
  } else {
    if (f32) exchange(0.f);
    else exchange((bf16_t)0.f);
  }
}

// The epilogue of a wave's TM x TN blocks of 16 x 16 (lane holds D[i][j]: i = 4 g + r the column, j = lane % 16 the row), straight out
// of registers.  Of 16-bit results the rows of sixteen lanes swap halves of two neighbouring blocks, so that a lane stores 16 bytes and a
// row 64; of 32-bit ones a lane has 16 bytes and a row 64 already (the residual stream's, which is read as well, goes through LDS).  Every block of sixteen columns is queries, keys or values of one
// head.  Values, of which four positions lie interleaved, go through LDS, where a lane takes four such positions of a channel, whatever row
// they start at; where the wave's rows do not have all four behind one another (tokens may come in any order) each is stored by itself.  (One
// by one for all whose quad does not start at a multiple of four rows: 1295 x 3072 x 1024 in two sequences 23.6 us, aligned 15.6.)
// `scratch`: block_scratch_bytes<TM, TN>() of this wave's own.
template <int TM, int TN>
constexpr int block_scratch_bytes() { return 16 * (TN * 64 + 16) > TM * 16 * (8 + 32) ? 16 * (TN * 64 + 16) : TM * 16 * (8 + 32); }

// Four values each of two blocks beside each other -> eight of one: the rows of sixteen lanes 0 and 2 get the first block's columns 0 to 7 and 8 to
// 15, the rows 1 and 3 the second's.
__device__ __forceinline__ int4v neighbours_joined(__attribute__((__vector_size__(8))) int a, __attribute__((__vector_size__(8))) int b) {
  const auto low = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false), high = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  return int4v{(int)low[0], (int)high[0], (int)low[1], (int)high[1]};
}

template <typename T, int TM, int TN>
__device__ __forceinline__ void epilogue_blocks(const Epilogue& e, int M, int N, int m0, int n0, floatx4 (&acc)[TN][TM], int split,
                                                unsigned char* scratch) {
  const int lane = threadIdx.x & 63, i16 = lane & 15, g = lane >> 4;
  constexpr int COLUMNS = TN * 16;
  static_assert(sizeof(T) == 2, "float products have no forms on these blocks");
  const bool f32 = e.mode == EPI_F32 || e.mode == EPI_RESIDUAL;
  const int piece = f32 ? 4 : 8;                       // values in 16 bytes
  const bool scatters = e.mode == EPI_QKV && n0 + COLUMNS > e.n_q;
  const bool whole = e.out_rows == 0 && N % piece == 0 && e.ldo % piece == 0 && e.split_stride % piece == 0 &&
                     (((uintptr_t)e.out | (uintptr_t)e.bias) & 15) == 0 &&
                     (!scatters || (e.kv.head_dim % 16 == 0 && e.n_q % 16 == 0 && (((uintptr_t)e.kv.keys | (uintptr_t)e.kv.values) & 15) == 0));
  if (!whole) {                                        // (the same for the whole wave)
    constexpr int PITCH = COLUMNS * 4 + 16;
#pragma unroll
    for (int bm = 0; bm < TM; ++bm) {
#pragma unroll
      for (int bn = 0; bn < TN; ++bn) *reinterpret_cast<floatx4*>(scratch + i16 * PITCH + (bn * 16 + g * 4) * 4) = acc[bn][bm];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");       // (a wave's accesses of LDS are served in order)
#pragma nounroll
      for (int i = lane; i < 4 * COLUMNS; i += 64) {
        const int r = i / (COLUMNS / 4), c = i % (COLUMNS / 4) * 4, m = m0 + bm * 16 + r;
        const floatx4 row = *reinterpret_cast<const floatx4*>(scratch + r * PITCH + c * 4);
        const float v[4] = {row[0], row[1], row[2], row[3]};
        if (m < M) epilogue4<T>(e, N, m, n0 + c, v, split);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    return;
  }
  // what has to come from memory is asked for first: places of the rows' tokens, the bias, the first rows of the residual stream
  int pos[TM], seq[TM];
  if (scatters) {
#pragma unroll
    for (int bm = 0; bm < TM; ++bm) {
      const int m = m0 + bm * 16 + i16 < M ? m0 + bm * 16 + i16 : M - 1;
      pos[bm] = e.tok_pos[m];
      seq[bm] = e.tok_seq[m];
    }
  }
  if (e.bias != nullptr && split == 0) {
    floatx4 b[TN];
#pragma unroll
    for (int bn = 0; bn < TN; ++bn) {
      const int n = n0 + bn * 16 + g * 4;
      b[bn] = *reinterpret_cast<const floatx4*>(e.bias + (n < N ? n : 0));
    }
#pragma unroll
    for (int bn = 0; bn < TN; ++bn)
#pragma unroll
      for (int bm = 0; bm < TM; ++bm) acc[bn][bm] += b[bn];
  }
  if (f32) {
    float* const first = static_cast<float*>(e.out) + (e.mode == EPI_F32 ? (int64_t)split * e.split_stride : 0) + (n0 < N ? n0 : 0);
    if (e.mode == EPI_RESIDUAL) {
      // Through LDS, sixteen rows at a time, so that neighbouring lanes ask for neighbouring pieces of the stream's rows.  Asked for by the
      // lanes that hold the sums, the pieces of neighbouring lanes are of sixteen rows, and the address unit, which takes sixteen lanes at a time,
      // had 64 requests of every load (us, so / through LDS: 2048 x 1600 x 1600 in tiles of 128 x 128 24.4 / 22.7, 1959 x 1600 x 6400 55.5 / 54.2, 3072 x 1600 x
      // 1600 in 128 x 160 27.2 / 25.7, 2048 x 1024 x 1024 in 128 x 64 12.9 / 12.1).  Stores, which nothing waits for, gain nothing by it, nor did 128 bytes of a
      // row with every instruction (two neighbouring blocks' halves swapped) or the stream asked for before the bias.
      constexpr int PITCH = COLUMNS * 4 + 16;
      floatx4 old[2][TN];
      auto at = [&](int t, int& r) {                 // the column of a lane's t-th piece of sixteen rows; its row in r
        const int i = lane + 64 * t;
        r = i / (4 * TN);
        return 4 * (i - r * (4 * TN));
      };
      auto ask = [&](int bm) {
#pragma unroll
        for (int t = 0; t < TN; ++t) {
          int r;
          const int c = at(t, r), m = m0 + bm * 16 + r;
          old[bm & 1][t] = *reinterpret_cast<const floatx4*>(first + (int64_t)(m < M ? m : M - 1) * e.ldo + (n0 + c < N ? c : 0));
        }
      };
      ask(0);
#pragma unroll
      for (int bm = 0; bm < TM; ++bm) {
        if (bm + 1 < TM) ask(bm + 1);
#pragma unroll
        for (int bn = 0; bn < TN; ++bn) *reinterpret_cast<floatx4*>(scratch + i16 * PITCH + (bn * 16 + g * 4) * 4) = acc[bn][bm];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // (a wave's accesses of LDS are served in order)
#pragma unroll
        for (int t = 0; t < TN; ++t) {
          int r;
          const int c = at(t, r), m = m0 + bm * 16 + r;
          const floatx4 sum = *reinterpret_cast<const floatx4*>(scratch + r * PITCH + c * 4) + old[bm & 1][t];
          if (m < M && n0 + c < N) *reinterpret_cast<floatx4*>(first + (int64_t)m * e.ldo + c) = sum;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      }
      return;
    }
#pragma unroll
    for (int bm = 0; bm < TM; ++bm) {
      const int m = m0 + bm * 16 + i16;
      if (m >= M) continue;
#pragma unroll
      for (int bn = 0; bn < TN; ++bn) {
        const int c = bn * 16 + g * 4;
        if (n0 + c < N) *reinterpret_cast<floatx4*>(first + (int64_t)m * e.ldo + c) = acc[bn][bm];
      }
    }
    return;
  }
  if (e.mode == EPI_ACT) {                           // (one choice for all values)
    auto all = [&](auto act) {
#pragma unroll
      for (int bn = 0; bn < TN; ++bn)
#pragma unroll
        for (int bm = 0; bm < TM; ++bm)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[bn][bm][r] = activate_as<T, decltype(act)::value>(acc[bn][bm][r]);
    };
    if (e.act == ACT_GELU_TANH) all(Constant<ACT_GELU_TANH>());
    else if (e.act == ACT_SQUARED_RELU) all(Constant<ACT_SQUARED_RELU>());
    else all(Constant<ACT_GELU_ERF>());
  }
  typedef __attribute__((__vector_size__(8))) int int2v;
  auto packed = [&](floatx4 v) {
    const bf16x4 p = {(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
    return __builtin_bit_cast(int2v, p);
  };
  if (!scatters) {
    T* const out = static_cast<T*>(e.out) + n0;
#pragma unroll
    for (int bm = 0; bm < TM; ++bm) {
      const int m = m0 + bm * 16 + i16;
      T* const row = out + (int64_t)m * e.ldo;
#pragma unroll
      for (int bn = 0; bn < TN; bn += 2) {
        if (bn + 1 < TN) {
          const int c = (bn + (g & 1)) * 16 + 8 * (g >> 1);
          const int4v v = neighbours_joined(packed(acc[bn][bm]), packed(acc[bn + 1 < TN ? bn + 1 : bn][bm]));
          if (m < M && n0 + c < N) *reinterpret_cast<int4v*>(row + c) = v;
        } else {
          const int c = bn * 16 + 4 * g;
          if (m < M && n0 + c < N) *reinterpret_cast<int2v*>(row + c) = packed(acc[bn][bm]);
        }
      }
    }
    return;
  }
  // An element's place is what its row gives (of queries, keys and values) and what its block of columns gives, which is the same for
  // the whole wave: both worked out here, once.  (A head's number and channel divided out at every store: 2048 x 4800 x 1600 38.4 us,
  // so 32.7.)
  const int hd = e.kv.head_dim;
  int64_t key_row[TM], value_row[TM];
  uint64_t leads = 0, follows = 0;                   // rows whose position and the three behind it lie interleaved, all of them this wave's
  auto before = [&](const int (&of)[TM], int bm) {   // of the row before (of the wave's first row: not used)
    const int here = lane_moved<0x121>(of[bm]), last = lane_moved<0x121>(of[bm > 0 ? bm - 1 : 0]);     // (row_ror:1)
    return i16 == 0 ? last : here;
  };
#pragma unroll
  for (int bm = 0; bm < TM; ++bm) {
    const bool here = m0 + bm * 16 + i16 < M;
    const int seq_before = before(seq, bm), pos_before = before(pos, bm);      // (by all lanes: one that is switched off passes nothing on)
    leads |= (__ballot(here && pos[bm] % 4 == 0) & 0xffff) << (16 * bm);
    follows |= (__ballot(here && seq[bm] == seq_before && pos[bm] == pos_before + 1) & 0xffff) << (16 * bm);
  }
  leads &= follows >> 1 & follows >> 2 & follows >> 3;
#pragma unroll
  for (int bm = 0; bm < TM; ++bm) {
    const int64_t plane = (int64_t)e.kv.blocks[(int64_t)seq[bm] * e.kv.max_blocks + pos[bm] / BT_KV_BLOCK] * e.kv.block_stride;
    key_row[bm] = plane + key_offset(hd, pos[bm], 0);
    value_row[bm] = plane + value_offset(hd, pos[bm], 0);
  }
  const uint64_t together = leads | leads << 1 | leads << 2 | leads << 3;
  int64_t* const value_rows = reinterpret_cast<int64_t*>(scratch);
  bf16_t* const turned = reinterpret_cast<bf16_t*>(scratch + TM * 16 * 8);
  if (n0 + COLUMNS > e.n_q + e.n_kv && g == 0) {
#pragma unroll
    for (int bm = 0; bm < TM; ++bm) value_rows[bm * 16 + i16] = value_row[bm];
  }
  int64_t column[TN];                                // of queries: the column; of keys and values: the head's plane and the channel (of values times 4)
  int kind[TN];                                      // 0 queries, 1 keys, 2 values, 3 beyond the columns
  {
    const int first = n0 - e.n_q;                    // (below zero: so many columns of queries come first)
    int k = first < 0 ? 0 : first >= e.n_kv ? first - e.n_kv : first;
    int head = k / hd, channel = k - head * hd;
#pragma unroll
    for (int bn = 0; bn < TN; ++bn) {
      const int n = n0 + bn * 16;
      kind[bn] = n < e.n_q ? 0 : n < e.n_q + e.n_kv ? 1 : n < N ? 2 : 3;
      if (n == e.n_q || n == e.n_q + e.n_kv) head = channel = 0;
      column[bn] = kind[bn] == 0 ? n : head * e.kv.head_stride + (kind[bn] == 1 ? channel : 4 * channel);
      if (n >= e.n_q) {
        channel += 16;
        if (channel == hd) { channel = 0; ++head; }
      }
    }
  }
  T *const out = static_cast<T*>(e.out), *const keys = static_cast<T*>(e.kv.keys), *const values = static_cast<T*>(e.kv.values);
#pragma unroll
  for (int bm = 0; bm < TM; ++bm) {
    const int m = m0 + bm * 16 + i16;
    T *const out_row = out + (int64_t)m * e.ldo, *const keys_row = keys + key_row[bm];
#pragma unroll
    for (int bn = 0; bn < TN; bn += 2) {
      const int next = bn + 1 < TN ? bn + 1 : bn;
      if (next > bn && kind[next] < 2) {             // (the kinds come in order)
        const int4v v = neighbours_joined(packed(acc[bn][bm]), packed(acc[next][bm]));
        const bool second = g & 1, is_key = second ? kind[next] == 1 : kind[bn] == 1;
        if (m < M) *reinterpret_cast<int4v*>((is_key ? keys_row : out_row) + (second ? column[next] : column[bn]) + 8 * (g >> 1)) = v;
        continue;
      }
#pragma unroll
      for (int b = bn; b <= next; ++b)
        if (kind[b] < 2 && m < M) *reinterpret_cast<int2v*>((kind[b] == 1 ? keys_row : out_row) + column[b] + 4 * g) = packed(acc[b][bm]);
    }
  }
#pragma unroll
  for (int b = 0; b < TN; ++b) {
    if (kind[b] != 2) continue;
#pragma unroll
    for (int bm = 0; bm < TM; ++bm) *reinterpret_cast<int2v*>(turned + (bm * 16 + i16) * 16 + 4 * g) = packed(acc[b][bm]);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");       // (a wave's accesses of LDS are served in order)
#pragma unroll
    for (int t = 0; t < TM; ++t) {                   // of every four rows one leads at most; a lane takes a channel
      const int window = 4 * t + g, lead = (int)(leads >> (4 * window)) & 15;
      if (lead) {
        const int r = 4 * window + __builtin_ctz(lead);
        const bf16_t* const from = turned + r * 16 + i16;
        const bf16x4 four = {from[0], from[16], from[32], from[48]};
        *reinterpret_cast<bf16x4*>(values + value_rows[r] + column[b] + 4 * i16) = four;
      }
    }
#pragma unroll
    for (int bm = 0; bm < TM; ++bm)
      if (m0 + bm * 16 + i16 < M && !(together >> (16 * bm + i16) & 1)) {
        T* const dst = values + value_row[bm] + column[b] + 16 * g;
#pragma unroll
        for (int r = 0; r < 4; ++r) dst[4 * r] = from_float<T>(acc[b][bm][r]);
      }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
}
