// Shared device helpers for the gfx950 kernels: element types, vector types,
// the paged key/value addressing and wave/block reductions.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#define BT_EXPORT extern "C" __attribute__((visibility("default")))

// Error codes returned by every entry point (0 = launched).
#define BT_OK 0
#define BT_REFUSED 1  // the sizes are outside what the kernel takes; see bt_last_error()
#define BT_HIP_ERROR 2

// Tokens per block of the paged key/value storage.  A key tile of 32 never straddles a block.
#define BT_KV_BLOCK 64

typedef __bf16 bf16_t;
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;
typedef __attribute__((__vector_size__(4 * sizeof(int)))) int int4v;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;

void bt_set_error(const char* fmt, ...);
int bt_check_launch(const char* what);

#define BT_REFUSE(...)            \
  do {                            \
    bt_set_error(__VA_ARGS__);    \
    return BT_REFUSED;            \
  } while (0)

// A number as a type: what a choice made once hands to the code that is compiled for it.
template <int N>
struct Constant {
  static constexpr int value = N;
};

__device__ __forceinline__ float to_float(float v) { return v; }
__device__ __forceinline__ float to_float(bf16_t v) { return (float)v; }

template <typename T>
__device__ __forceinline__ T from_float(float v);
template <>
__device__ __forceinline__ float from_float<float>(float v) { return v; }
template <>
__device__ __forceinline__ bf16_t from_float<bf16_t>(float v) { return (bf16_t)v; }  // round to nearest even

// Geometry of one group of layers in the paged key/value storage.  A (block, head) *plane* holds
// the keys (or values) of one head for the 64 positions of one block:
//   keys:   plane = [BT_KV_BLOCK][head_dim]
//   values: plane = [BT_KV_BLOCK / 4][head_dim][4]   (four positions interleaved per channel, so
//           that a lane reads four consecutive positions of one channel at once)
// The plane of (block, head) starts block * block_stride + head * head_stride elements into the
// layer: the storage decides which of the two lies closer together (with the heads outermost, the
// blocks a sequence took one after the other are one contiguous run for each head).
// `blocks` is the table of the step's sequences: blocks[seq * max_blocks + position / BT_KV_BLOCK].
struct KvView {
  void* keys;            // base of the layer
  void* values;          // base of the layer
  const int* blocks;     // [n_seqs][max_blocks]
  int max_blocks;
  int kv_heads;
  int head_dim;
  int64_t block_stride;  // elements from a block's plane to the next block's, same head
  int64_t head_stride;   // elements from a head's plane to the next head's, same block
};

__device__ __forceinline__ int64_t kv_plane(const KvView& kv, int block, int kv_head) {
  return (int64_t)block * kv.block_stride + (int64_t)kv_head * kv.head_stride;
}
__device__ __forceinline__ int64_t kv_block_base(const KvView& kv, int seq, int pos, int kv_head) {
  return kv_plane(kv, kv.blocks[(int64_t)seq * kv.max_blocks + pos / BT_KV_BLOCK], kv_head);
}
// Element offset of key (pos, channel) inside its (block, head) plane.
__device__ __forceinline__ int key_offset(int head_dim, int pos, int channel) {
  return (pos % BT_KV_BLOCK) * head_dim + channel;
}
// Element offset of value (pos, channel) inside its (block, head) plane.
__device__ __forceinline__ int value_offset(int head_dim, int pos, int channel) {
  int p = pos % BT_KV_BLOCK;
  return ((p >> 2) * head_dim + channel) * 4 + (p & 3);
}

// Activations of a step of few rows may be kept "chunk-major": the chunks of 64 bytes of K (32
// bfloat16, 16 float32 columns) one after the other, each holding that chunk of every row,
// [columns / chunk][rows][chunk].  The lanes of an MFMA operand load (16 rows by 64 bytes) then read
// one contiguous KiB, where row-major rows lie a whole row apart: reading 64 rows of 1,600
// columns that way takes a work-group 1 us instead of 5.8.  Element offset of (row, column);
// `rows` = 0 means row-major with the given pitch.
template <typename T>
__host__ __device__ __forceinline__ int64_t activation_offset(int rows, int64_t pitch, int row, int column) {
  constexpr int CHUNK = 64 / (int)sizeof(T);
  return rows > 0 ? ((int64_t)(column / CHUNK) * rows + row) * CHUNK + column % CHUNK : (int64_t)row * pitch + column;
}

// Reductions over a wave without LDS: v_permlane32_swap and v_permlane16_swap bring the lanes 32 and 16 apart together, rotations
// inside rows of sixteen those 8 and 4 apart, quad permutations the last two.  Six steps of one or two vector instructions, where a
// shuffle through LDS (__shfl_xor) has every step wait some 50 ns for its lane: a decode step's kernels have one to four reductions
// in a row on their critical path.  (Decode steps, us: GPT-2 small, one sequence, 337 -> 319, xl, eight sequences, 2,068 -> 2,019.)  The pairs and their order are those of a butterfly from 32 down to 1, so the sums are the same
// bit for bit.  (The rotations by 8 and 4 meet lane ^ 8 and lane ^ 4 only because the values are alike by then in the lanes
// further apart.)
template <int APART>      // 32 or 16: in every lane the values of its pair, the one of the lower lanes first
__device__ __forceinline__ void lane_pair(int v, int& low, int& high) {
  static_assert(APART == 32 || APART == 16, "lanes of the two halves, or of neighbouring rows of sixteen");
  if constexpr (APART == 32) {
    const auto both = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    low = both[0];
    high = both[1];
  } else {
    const auto both = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    low = both[0];
    high = both[1];
  }
}
template <int CONTROL>
__device__ __forceinline__ int lane_moved(int v) { return __builtin_amdgcn_update_dpp(0, v, CONTROL, 0xf, 0xf, true); }
template <int CONTROL>
__device__ __forceinline__ float lane_moved(float v) {
  return __builtin_bit_cast(float, lane_moved<CONTROL>(__builtin_bit_cast(int, v)));
}
struct LaneSum {
  __device__ __forceinline__ float operator()(float a, float b) const { return a + b; }
};
struct LaneMax {
  __device__ __forceinline__ float operator()(float a, float b) const { return fmaxf(a, b); }
};
template <int APART, typename F>
__device__ __forceinline__ float across(float v, F f) {       // with the lane 32 or 16 away
  int low, high;
  lane_pair<APART>(__builtin_bit_cast(int, v), low, high);
  return f(__builtin_bit_cast(float, low), __builtin_bit_cast(float, high));
}
template <typename F>
__device__ __forceinline__ float row_reduce(float v, F f) {   // over the sixteen lanes of a row
  v = f(v, lane_moved<0x128>(v));                             // row_ror:8
  v = f(v, lane_moved<0x124>(v));                             // row_ror:4
  v = f(v, lane_moved<0x4e>(v));                              // quad_perm:[2,3,0,1]
  return f(v, lane_moved<0xb1>(v));                           // quad_perm:[1,0,3,2]
}
// The value of lane ^ 2^STEP, steps taken from the highest down (see above for steps 3 and 2).
template <int STEP>
__device__ __forceinline__ int lane_other(int v) {
  if constexpr (STEP >= 4) {
    int low, high;
    lane_pair<1 << STEP>(v, low, high);
    return threadIdx.x & (1 << STEP) ? low : high;
  } else {
    return lane_moved<STEP == 3 ? 0x128 : STEP == 2 ? 0x124 : STEP == 1 ? 0x4e : 0xb1>(v);
  }
}
// The best (value, index) of a wave; among equal values the lowest index.  Every lane gets it.
template <int STEP = 5>
__device__ __forceinline__ void wave_best(float& value, int& index) {
  const float other = __builtin_bit_cast(float, lane_other<STEP>(__builtin_bit_cast(int, value)));
  const int other_index = lane_other<STEP>(index);
  if (other > value || (other == value && other_index < index)) { value = other; index = other_index; }
  if constexpr (STEP > 0) wave_best<STEP - 1>(value, index);
}
__device__ __forceinline__ float wave_sum(float v) { return row_reduce(across<16>(across<32>(v, LaneSum()), LaneSum()), LaneSum()); }
__device__ __forceinline__ float wave_max(float v) { return row_reduce(across<16>(across<32>(v, LaneMax()), LaneMax()), LaneMax()); }

// Block-wide reductions for blocks of up to 1024 threads; `scratch` holds 32 floats of LDS, on 16 bytes.
// Every thread gets the result.  Safe to call repeatedly with the same scratch.  THREADS: the block's size where it is a
// constant (the waves' shares are then read together and not in a loop that waits for each); 0 otherwise.
template <int THREADS, typename F>
__device__ __forceinline__ float block_join(float v, float* scratch, float start, F f) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = start;
  if constexpr (THREADS > 0) {
    constexpr int WAVES = THREADS / 64;
    static_assert(THREADS % 256 == 0, "whole quads of waves");
    floatx4 part[WAVES / 4];
#pragma unroll
    for (int q = 0; q < WAVES / 4; ++q) part[q] = reinterpret_cast<const floatx4*>(scratch)[q];
#pragma unroll
    for (int w = 0; w < WAVES; ++w) total = f(total, part[w >> 2][w & 3]);
  } else {
    const int waves = (blockDim.x + 63) >> 6;
    for (int w = 0; w < waves; ++w) total = f(total, scratch[w]);
  }
  return total;
}
template <int THREADS = 0>
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  return block_join<THREADS>(wave_sum(v), scratch, 0.f, LaneSum());
}
template <int THREADS = 0>
__device__ __forceinline__ float block_max(float v, float* scratch) {
  return block_join<THREADS>(wave_max(v), scratch, NAN, LaneMax());
}
