// What the kernels that multiply tiles from LDS on the matrix units share: the element types' instructions, the layout
// of a tile's rows in LDS, the order of tiles and the waits for loads that write LDS directly.
#pragma once

#include "common.h"

#define TILE_ROW_BYTES 128

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

// A tile's product over K: operands go from memory straight into LDS (128-byte rows, BM of A, then BN of W, swizzled on the
// memory side) and from there into the matrix units, on WM x WN waves, each with TM x TN blocks of 32 x 32.
//   stages   STAGES tiles of 128 bytes of K lie in LDS or are on their way; one barrier a tile
//   operands a quarter's are read while the quarter two before it is multiplied; those of the next tile's first half behind
//            the barrier, beside the second half of this one, so that the barrier and the reads' latency show nowhere
//   the loop is one straight line: behind the last tile the last one is asked for again, so that the waits are constants.  (A
//            test inside made the compiler copy all accumulators once or twice a tile, 64 to 128 moves beside 16 matrix
//            instructions, and the time of a tile was taken for what a compute unit can pull; a unit pulls 150 GB/s.)
template <typename T, int BM, int BN, int WM, int WN, int STAGES>
struct TilePipe {
  static constexpr int WAVES = WM * WN, ROWS = BM + BN, STAGE_BYTES = ROWS * TILE_ROW_BYTES;
  static constexpr int STEP = 8 * WAVES, LOADS = ROWS / STEP;      // a wave's load instruction: eight rows
  static constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
  static_assert(BM % STEP == 0 && BN % STEP == 0 && TM >= 1 && TN >= 1 && STAGES >= 2 && (STAGES - 1) * LOADS < 64,
                "whole loads, whole blocks, and no more loads in flight than the wave's counter holds");

  // acc += the product of `count` tiles; row_bytes(stage_row, from_w): what that row's first byte lies behind `a` or `w`.
  // On return every wave's loads have landed and nobody reads the stages any more once all have passed the next barrier.
  template <typename Offset, typename RowBytes>
  static __device__ __forceinline__ void multiply(unsigned char* lds, const unsigned char* a, const unsigned char* w, int count,
                                                  RowBytes row_bytes, floatx16 (&acc)[TN][TM]) {
    if (count <= 0) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave % WM, wn = wave / WM, l32 = lane & 31, g = lane >> 5;
    Offset off[LOADS];
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      const int stage_row = STEP * j + 8 * wave + (lane >> 3);
      off[j] = (Offset)(row_bytes(stage_row, STEP * j >= BM) + (((lane & 7) ^ ((stage_row >> 1) & 7)) << 4));
    }
    int issued = 0;
    auto issue = [&](int stage) {
#pragma unroll
      for (int j = 0; j < LOADS; ++j)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)((STEP * j >= BM ? w : a) + off[j]),
                                         (__attribute__((address_space(3))) void*)(lds + stage * STAGE_BYTES + (STEP * j + 8 * wave) * TILE_ROW_BYTES),
                                         16, 0, 0);
      const int step = ++issued < count ? TILE_ROW_BYTES : 0;
      a += step;
      w += step;
    };
    int w_rd[4], a_rd[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      w_rd[kk] = BM * TILE_ROW_BYTES + swizzled(wn * (BN / WN) + l32, 2 * kk + g);
      a_rd[kk] = swizzled(wm * (BM / WM) + l32, 2 * kk + g);
    }
    int4v op[4][TM + TN];
    auto read = [&](int stage, int kk) {
      const unsigned char* base = lds + stage * STAGE_BYTES;
#pragma unroll
      for (int b = 0; b < TM; ++b) op[kk][b] = *reinterpret_cast<const int4v*>(base + a_rd[kk] + b * 4096);
#pragma unroll
      for (int b = 0; b < TN; ++b) op[kk][TM + b] = *reinterpret_cast<const int4v*>(base + w_rd[kk] + b * 4096);
    };
    auto quarter = [&](int kk) {
#pragma unroll
      for (int bn = 0; bn < TN; ++bn)
#pragma unroll
        for (int bm = 0; bm < TM; ++bm) Mma<T>::block32(acc[bn][bm], op[kk][TM + bn], op[kk][bm]);
      __builtin_amdgcn_sched_barrier(0);
    };
    auto turn = [&](int stage, int next, bool more) {
      read(stage, 2);
      quarter(0);
      read(stage, 3);
      quarter(1);
      if (more) {       // this wave's loads of the next tile have landed and its reads of this one are done: so have everyone's
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((STAGES - 2) * LOADS) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        issue(stage);
        __builtin_amdgcn_sched_barrier(0);
        read(next, 0);
      }
      quarter(2);
      if (more) read(next, 1);
      quarter(3);
    };
#pragma unroll
    for (int t = 0; t < STAGES; ++t) issue(t);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STAGES - 1) * LOADS) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read(0, 0);
    read(0, 1);
    __builtin_amdgcn_sched_barrier(0);
    int stage = 0, next = 1;
    for (int i = 1; i < count; ++i) {
      turn(stage, next, true);
      stage = next;
      next = next + 1 == STAGES ? 0 : next + 1;
    }
    turn(stage, next, false);
    wait_vmcnt<0>();
  }
};

// The same product on blocks of 16 x 16, for tiles that take a compute unit's LDS and registers whole: WM x WN waves, each TM x TN blocks,
// SA tiles of A's rows and SW tiles of W's in LDS or on their way (W, which comes from memory, may be asked for further ahead than A,
// which the kernel before left in the caches).  Differences from TilePipe, each measured at 2048 x 4800 x 1600 on 256 x 160 and 2048 x 6400 x
// 1600 on 256 x 256 (weights from memory):
//   reads     of the next half tile stand one before each of the first matrix instructions of this half, behind a wait that the
//             compiler knows: with reads in front of them it waited for those as well (lgkmcnt(0)), a trip to LDS every half
//   loads     of the tile after the last one in LDS stand between the matrix instructions of the half behind the barrier: eight
//             waves that ask for all theirs at once wait for the address unit (33.7 -> 32.3 us)
//   stages    A's and W's counted by themselves (256 x 256, two of A and three of W where three of both do not fit, 46.9 -> 42.2 us; the forms that
//             are used have three to five of A and three to eight of W, eight of A for 64 rows)
// What a compute unit has asked for and not got is 32 KiB at most, however many stages there are: 150 GB/s out of L2, 95 from the
// memory-side cache and 65 from memory, so a tile wants 2 * BM * BN / (BM + BN) operations a byte and one round of tiles over the
// chip (figures of the forms with the kernels).
template <typename T, int BM, int BN, int WM, int WN, int SA, int SW>
struct BlockPipe {
  static constexpr int WAVES = WM * WN, TM = BM / WM / 16, TN = BN / WN / 16;
  static constexpr int A_GROUPS = BM / 8, W_GROUPS = BN / 8;               // a wave's load instruction: eight rows
  static constexpr int A_LOADS = A_GROUPS / WAVES, W_LEAST = W_GROUPS / WAVES, W_LOADS = (W_GROUPS + WAVES - 1) / WAVES;
  static constexpr int LOADS = A_LOADS + W_LOADS;
  static constexpr int A_STAGE = BM * TILE_ROW_BYTES, W_STAGE = BN * TILE_ROW_BYTES, BYTES = SA * A_STAGE + SW * W_STAGE;
  static_assert(BM % (16 * WM) == 0 && BN % (16 * WN) == 0 && A_GROUPS % WAVES == 0 && SA >= 2 && SW >= 2 && BYTES <= 160 * 1024,
                "whole blocks, whole loads of A, and what LDS holds");
  // Loads that may still be on their way when the tile behind the barrier has landed: those behind its A (issued with W of the
  // same turn, then whole turns) and behind its W.  (Waves with one load of W less than others wait for as many fewer.)
  static constexpr int A_BEHIND = (SA - 2) * (A_LOADS + W_LEAST) + W_LEAST, W_BEHIND = (SW - 2) * (A_LOADS + W_LEAST);
  static constexpr int BEHIND = A_BEHIND < W_BEHIND ? A_BEHIND : W_BEHIND;
  static_assert((SA > SW ? SA : SW) * LOADS < 64, "no more loads in flight than the wave's counter holds");

  // acc += the product of `count` tiles; row_bytes(row of the tile, of W): what that row's first byte lies behind `a` or `w`.
  // On return every wave's loads have landed and nobody reads the stages any more once all have passed the next barrier.
  template <typename Offset, typename RowBytes>
  static __device__ __forceinline__ void multiply(unsigned char* lds, const unsigned char* a, const unsigned char* w, int count,
                                                  RowBytes row_bytes, floatx4 (&acc)[TN][TM]) {
    if (count <= 0) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave % WM, wn = wave / WM, i16 = lane & 15, g = lane >> 4;
    Offset off[LOADS];
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      const bool from_w = j >= A_LOADS;
      const int row = 8 * ((from_w ? j - A_LOADS : j) * WAVES + wave) + (lane >> 3);
      off[j] = (Offset)(row_bytes(row, from_w) + (((lane & 7) ^ ((row >> 1) & 7)) << 4));
    }
    auto load = [&](int j, int a_stage, int w_stage) {
      const bool from_w = j >= A_LOADS;
      const int group = (from_w ? j - A_LOADS : j) * WAVES + wave;
      if (!from_w || (j - A_LOADS + 1) * WAVES <= W_GROUPS || group < W_GROUPS)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)((from_w ? w : a) + off[j]),
                                         (__attribute__((address_space(3))) void*)(lds + (from_w ? SA * A_STAGE + w_stage * W_STAGE : a_stage * A_STAGE) +
                                                                                   group * (8 * TILE_ROW_BYTES)),
                                         16, 0, 0);
    };
    int a_issued = 0, w_issued = 0;        // (behind the last tile the last one is asked for again)
    auto a_next = [&]() { a += ++a_issued < count ? TILE_ROW_BYTES : 0; };
    auto w_next = [&]() { w += ++w_issued < count ? TILE_ROW_BYTES : 0; };
    int a_rd[2], w_rd[2];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      a_rd[half] = swizzled(wm * (BM / WM) + i16, 4 * half + g);
      w_rd[half] = SA * A_STAGE + swizzled(wn * (BN / WN) + i16, 4 * half + g);
    }
    int4v op[2][TM + TN];
    auto read = [&](int r, int half, int a_stage, int w_stage) {
      op[half][r] = *reinterpret_cast<const int4v*>(lds + (r < TM ? a_stage * A_STAGE + a_rd[half] + r * (16 * TILE_ROW_BYTES)
                                                                 : w_stage * W_STAGE + w_rd[half] + (r - TM) * (16 * TILE_ROW_BYTES)));
    };
    // Multiplies half a tile, reads the other half of the tile in the stages, or of the next tile, and asks for a tile.
    auto multiply_half = [&](int half, bool reads, bool loads, int a_read, int w_read, int a_free, int w_free) {
      constexpr int BLOCKS = TM * TN;
      __builtin_amdgcn_s_waitcnt(0xc07f);                    // lgkmcnt(0): this half's operands, asked for half a tile ago
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 0; x < BLOCKS; ++x) {
#pragma unroll
        for (int r = 0; r < TM + TN; ++r)
          if (reads && r * BLOCKS / (2 * (TM + TN)) == x) read(r, half ^ 1, a_read, w_read);
#pragma unroll
        for (int j = 0; j < LOADS; ++j)
          if (loads && (2 * j + 1) * BLOCKS / (2 * LOADS) == x) load(j, a_free, w_free);
        __builtin_amdgcn_sched_barrier(0);
        Mma<T>::block16(acc[x / TM][x % TM], op[half][TM + x / TM], op[half][x % TM]);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
#pragma unroll
    for (int t = 0; t < (SA > SW ? SA : SW); ++t) {
#pragma unroll
      for (int j = 0; j < LOADS; ++j)
        if (j < A_LOADS ? t < SA : t < SW) load(j, t, t);
      if (t < SA) a_next();
      if (t < SW) w_next();
    }
    wait_vmcnt<(SA - 1) * A_LOADS + (SW - 1) * W_LEAST>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int r = 0; r < TM + TN; ++r) read(r, 0, 0, 0);
    multiply_half(0, true, false, 0, 0, 0, 0);
    int a_stage = 0, a_then = 1, w_stage = 0, w_then = 1;
    for (int i = 1; i < count; ++i) {
      // this wave's loads of the next tile have landed and its reads of this one are done: behind the barrier so have everyone's
      __builtin_amdgcn_s_waitcnt((BEHIND & 15) | (BEHIND >> 4) << 14 | 0x70);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      multiply_half(1, true, true, a_then, w_then, a_stage, w_stage);
      a_next();
      w_next();
      a_stage = a_then;
      a_then = a_then + 1 == SA ? 0 : a_then + 1;
      w_stage = w_then;
      w_then = w_then + 1 == SW ? 0 : w_then + 1;
      multiply_half(0, true, false, a_stage, w_stage, 0, 0);
    }
    multiply_half(1, false, false, 0, 0, 0, 0);
    wait_vmcnt<0>();
  }
};
