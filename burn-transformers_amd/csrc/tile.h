// What the kernels that multiply tiles from LDS on the matrix units share: the element types' instructions, the layout
// of a tile's rows in LDS, the order of tiles and the waits for loads that write LDS directly.
#pragma once

#include "common.h"

#define TILE_ROW_BYTES 128

typedef __attribute__((__vector_size__(4 * sizeof(int)))) int int4v;

// What a lane's 16-byte operand read is to the matrix cores.  bfloat16: eight K values, one
// instruction of depth 32 (16-wide blocks; the lane's K group is lane / 16) or 16 (32-wide
// blocks; lane / 32).  float: four K values, taken by four instructions of depth 4 (or 2), the
// i-th multiplying element i of both operands: a lane's K group is the same for both operands,
// so the four instructions cover 16 (or 8) distinct K values exactly once.  The result lies in
// the lanes the same way for both types.
template <typename T>
struct Mma;
template <>
struct Mma<bf16_t> {
  static constexpr int ELEMS = 8;
  static __device__ __forceinline__ void block16(floatx4& acc, int4v w, int4v a) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, a), acc, 0, 0, 0);
  }
  static __device__ __forceinline__ void block32(floatx16& acc, int4v w, int4v a) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, a), acc, 0, 0, 0);
  }
};
template <>
struct Mma<float> {
  static constexpr int ELEMS = 4;
  static __device__ __forceinline__ void block16(floatx4& acc, int4v w, int4v a) {
    floatx4 wf = __builtin_bit_cast(floatx4, w), af = __builtin_bit_cast(floatx4, a);
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[i], af[i], acc, 0, 0, 0);
  }
  static __device__ __forceinline__ void block32(floatx16& acc, int4v w, int4v a) {
    floatx4 wf = __builtin_bit_cast(floatx4, w), af = __builtin_bit_cast(floatx4, a);
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(wf[i], af[i], acc, 0, 0, 0);
  }
};

// 16-byte chunk `chunk` of row `row` of an LDS tile with 128-byte rows.  LDS has 64 banks of four
// bytes and serves 16 lanes of a 16-byte access at a time, so two rows span the banks once and
// the 16 consecutive rows that read the same chunk for an MFMA operand must land in 16 different
// 16-byte slots: the chunk is XORed with bits 1..3 of the row (rows 2j and 2j + 1 share a value
// and differ in the half of the banks they occupy).  Measured with SQ_LDS_BANK_CONFLICT: a third
// of the LDS cycles were conflicts with the XOR taken from bits 0..2.
__device__ __forceinline__ int swizzled(int row, int chunk) {
  return row * TILE_ROW_BYTES + ((chunk ^ ((row >> 1) & 7)) << 4);
}

// Work-groups are handed to the eight XCDs in turn and each XCD has an L2 of its own, so the
// tiles are renumbered to give every XCD one contiguous range of them; inside a range, tiles
// that share a block of W's rows come first.
__device__ __forceinline__ int xcd_contiguous(int bid, int blocks) {
  int xcd = bid & 7, local = bid >> 3;
  int q = blocks >> 3, r = blocks & 7;
  return xcd * q + (xcd < r ? xcd : r) + local;
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <int NEWER, int LOADS>
__device__ __forceinline__ void wait_for_all_but(int newer) {
  // waits until at most `newer` tiles' loads (LOADS instructions each) of this wave are in flight
  if constexpr (NEWER == 0) {
    wait_vmcnt<0>();
  } else {
    if (newer >= NEWER) wait_vmcnt<NEWER * LOADS>();
    else wait_for_all_but<NEWER - 1, LOADS>(newer);
  }
}
