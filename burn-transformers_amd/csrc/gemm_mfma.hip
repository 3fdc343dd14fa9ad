// Matrix products on the MFMA units of gfx950, C[M,N] = A[M,K] . W[N,K]^T with 32-bit
// accumulation, in bfloat16 and in float (the float instructions multiply and add in full
// 32-bit: no reduced-precision mode exists in them; products made of parts: see gemm_tile_parts_kernel).  Both operands are K-contiguous, which is
// what an MFMA lane wants: consecutive K values in one 16-byte load.
//
//   gemm_tile    tiles for many rows (prefill): of 64 x 96 to 256 x 160 (gemm_tile_blocks_kernel) and of 64 x 64
//                (gemm_tile_pipe_kernel), whose operands go straight into LDS and whose loops are tile.h's;
//                gemm_tile_kernel for any K and operands of 4 GiB and more, through registers.  Tiles are
//                numbered so that each XCD's L2 sees neighbours.  Float products of many tiles are made of
//                the products of three bfloat16 parts of each operand (gemm_tile_parts_kernel).
//   gemm_skinny  up to 64 rows (decode).  The product is bound by streaming W once from HBM:
//                a work-group owns 16 columns, its eight waves split K, every lane keeps several
//                16-byte loads of W in flight, v_mfma_f32_16x16x32_bf16 does the arithmetic and
//                the waves' partial sums meet in LDS.  K can also be split across work-groups
//                into 32-bit partial sums that the consumer adds up.
//
// The weights are the MFMA "A" operand (rows = output columns n), the activations the "B"
// operand (columns = rows m), so a lane ends up with four consecutive n of one m.
//
// All are templates over the element type but the one on parts.

#include "host.h"
#include "tile.h"
#include "epilogue.h"
#include "calls.h"

#define TILE_K 64            // bfloat16 values in a 128-byte row of an LDS tile

// BM x BN tiles of 128-byte rows (64 bfloat16 or 32 float K values), WM x WN waves, each wave
// (BM / WM) x (BN / WN) as 32-wide MFMA blocks; LDS holds two stages, registers the tile
// on its way from memory to LDS: the loads of tile i + 1 fly while tile i is multiplied.
template <typename T, int BM, int BN, int WM, int WN>
__global__ void __launch_bounds__(WM * WN * 64)
gemm_tile_kernel(const T* __restrict__ A, int64_t lda, const T* __restrict__ W, int M, int N,
                 int K, Epilogue epi, int tiles_m, int tiles_n) {
  constexpr int ELEMS = Mma<T>::ELEMS;          // K values in a 16-byte chunk
  constexpr int ROW_K = 8 * ELEMS;              // K values in a 128-byte row of a tile
  constexpr int THREADS = WM * WN * 64;
  constexpr int ROWS = BM + BN;                 // rows of a stage: A's, then W's
  constexpr int PER_THREAD = ROWS * 8 / THREADS;  // 16-byte chunks a thread moves per tile
  constexpr int ROW_STEP = THREADS / 8;
  constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
  static_assert(ROWS * 8 % THREADS == 0 && BM % ROW_STEP == 0, "tile does not divide among the threads");
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];   // [2][ROWS * 128]
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int wm = wave % WM, wn = wave / WM;
  const int l32 = lane & 31, g = lane >> 5;
  const int tile = xcd_contiguous(blockIdx.x, tiles_m * tiles_n);
  const int m_base = (tile % tiles_m) * BM, n_base = (tile / tiles_m) * BN;
  const int split = blockIdx.z, splits = gridDim.z;
  const int k_tiles = (K + ROW_K - 1) / ROW_K;
  const int kt_begin = (int)((int64_t)k_tiles * split / splits);
  const int kt_end = (int)((int64_t)k_tiles * (split + 1) / splits);

  // chunk c of rows r0, r0 + ROW_STEP, ... of the stage: A's rows first, then W's.  Addresses
  // are rebuilt from the two bases for every load; keeping one pointer per row would not fit
  // the registers of the larger tiles.
  const int c = tid & 7, r0 = tid >> 3;
  constexpr int A_CHUNKS = BM / ROW_STEP;
  int4v regs[PER_THREAD];
  auto load_tile = [&](int kt) {
    // a chunk beyond K (a multiple of the chunk) reads the row's last chunk and is cleared when stored
    int k = kt * ROW_K + c * ELEMS;
    int kc = k < K ? k : K - ELEMS;
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) {
      int row = r0 + ROW_STEP * i;
      const T* src;
      if (i < A_CHUNKS) {
        int m = m_base + row;
        src = A + (int64_t)(m < M ? m : M - 1) * lda;
      } else {
        int n = n_base + row - BM;
        src = W + (int64_t)(n < N ? n : N - 1) * K;
      }
      regs[i] = *reinterpret_cast<const int4v*>(src + kc);
    }
  };
  auto store_tile = [&](int kt, int stage) {
    int keep = kt * ROW_K + c * ELEMS < K ? -1 : 0;
    unsigned char* base = lds + stage * (ROWS * TILE_ROW_BYTES);
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i)
      *reinterpret_cast<int4v*>(base + swizzled(r0 + ROW_STEP * i, c)) = regs[i] & keep;
  };

  floatx16 acc[TN][TM];
#pragma unroll
  for (int bn = 0; bn < TN; ++bn)
#pragma unroll
    for (int bm = 0; bm < TM; ++bm)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[bn][bm][r] = 0.f;

  auto multiply = [&](int stage) {
    // all operands of the tile are read before the first multiplication: LDS latency is paid once
    // per tile, and the reads of later steps return while earlier steps multiply
    const unsigned char* a_lds = lds + stage * (ROWS * TILE_ROW_BYTES);
    const unsigned char* w_lds = a_lds + BM * TILE_ROW_BYTES;
    constexpr int STEPS = TILE_ROW_BYTES / 32;      // a step: the two K groups' chunks
    int4v wop[STEPS][TN], aop[STEPS][TM];
#pragma unroll
    for (int kk = 0; kk < STEPS; ++kk) {
#pragma unroll
      for (int b = 0; b < TN; ++b)
        wop[kk][b] = *reinterpret_cast<const int4v*>(w_lds + swizzled(wn * (BN / WN) + b * 32 + l32, 2 * kk + g));
#pragma unroll
      for (int b = 0; b < TM; ++b)
        aop[kk][b] = *reinterpret_cast<const int4v*>(a_lds + swizzled(wm * (BM / WM) + b * 32 + l32, 2 * kk + g));
    }
#pragma unroll
    for (int kk = 0; kk < STEPS; ++kk)
#pragma unroll
      for (int bn = 0; bn < TN; ++bn)
#pragma unroll
        for (int bm = 0; bm < TM; ++bm)
          Mma<T>::block32(acc[bn][bm], wop[kk][bn], aop[kk][bm]);
  };

  const int count = kt_end - kt_begin;
  // tile i is multiplied from stage i % 2 while the loads of tile i + 1 fly into the registers
  if (count > 0) {
    load_tile(kt_begin);
    store_tile(kt_begin, 0);
  }
  __syncthreads();
  for (int i = 0; i < count; ++i) {
    if (i + 1 < count) load_tile(kt_begin + i + 1);
    multiply(i & 1);
    if (i + 1 < count) store_tile(kt_begin + i + 1, (i + 1) & 1);
    __syncthreads();
  }

  // lane holds D[i][j]: i = 8 * (r / 4) + 4 * g + r % 4 (column n), j = lane % 32 (row m)
#pragma unroll
  for (int bm = 0; bm < TM; ++bm) {
    const int m = m_base + wm * (BM / WM) + bm * 32 + l32;
#pragma unroll
    for (int bn = 0; bn < TN; ++bn) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float v[4] = {acc[bn][bm][4 * q], acc[bn][bm][4 * q + 1], acc[bn][bm][4 * q + 2], acc[bn][bm][4 * q + 3]};
        int n0 = n_base + wn * (BN / WN) + bn * 32 + q * 8 + g * 4;
        if (m < M) epilogue4<T>(epi, N, m, n0, v, split);
      }
    }
  }
}

// Tiles of 64 x 64 on TilePipe (tile.h).  K a multiple of 64 (float: 32), operands below 4 GiB.  Few rows, where a tile's start and end are
// most of it: on four waves half a microsecond less than on the eight of BlockPipe (bias included, us: 300 x 3072 x 1024 7.1, the vendor's
// library 9.4; 566 x 1024 x 1024 into the residual stream 7.7 / 9.3; 566 x 1024 x 4096 17.4 / 18.2).  Larger tiles were 128 x 128 and 128 x 256 of
// blocks of 32 x 32 on this loop, whose waves wait for the reads that they have just asked for: 2048 x 4800 x 1600 50 us, BlockPipe 34; 1295 x 4096 x 1024
// 23 / 20; 1600 x 1600 x 6400 53 / 46.
template <typename T, int BM, int BN, int WM, int WN, int STAGES>
__global__ void __launch_bounds__(WM * WN * 64, 2)
gemm_tile_pipe_kernel(const T* __restrict__ A, int64_t lda, const T* __restrict__ W, int M, int N,
                      int K, Epilogue epi, int tiles_m, int tiles_n, int group_m) {
  typedef TilePipe<T, BM, BN, WM, WN, STAGES> Pipe;
  constexpr int ROW_K = 8 * Mma<T>::ELEMS;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];   // [STAGES][BM + BN][128 bytes]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tile = xcd_contiguous(blockIdx.x, tiles_m * tiles_n);
  // (an XCD's run of tiles is a block of group_m by as many columns, about square: it pulls the fewest rows of A and W)
  const int per_group = group_m * tiles_n, first = tile / per_group * group_m, rest = tile % per_group;
  const int rows_m = group_m < tiles_m - first ? group_m : tiles_m - first;
  const int m_base = (first + rest % rows_m) * BM, n_base = rest / rows_m * BN;
  const int split = blockIdx.z, splits = gridDim.z;
  const int k_tiles = K / ROW_K;
  const int kt_begin = (int)((int64_t)k_tiles * split / splits);
  const int count = (int)((int64_t)k_tiles * (split + 1) / splits) - kt_begin;
  floatx16 acc[Pipe::TN][Pipe::TM];
#pragma unroll
  for (int bn = 0; bn < Pipe::TN; ++bn)
#pragma unroll
    for (int bm = 0; bm < Pipe::TM; ++bm)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[bn][bm][r] = 0.f;
  Pipe::template multiply<unsigned>(
      lds, reinterpret_cast<const unsigned char*>(A) + (int64_t)kt_begin * TILE_ROW_BYTES,
      reinterpret_cast<const unsigned char*>(W) + (int64_t)kt_begin * TILE_ROW_BYTES, count,
      [&](int stage_row, bool from_w) {
        const int row = from_w ? n_base + stage_row - BM : m_base + stage_row, limit = from_w ? N : M;
        return (int64_t)(row < limit ? row : limit - 1) * (from_w ? (int64_t)K : lda) * (int64_t)sizeof(T);
      },
      acc);
  __syncthreads();
  epilogue_tile<T, Pipe::TM, Pipe::TN>(epi, M, N, m_base + wave % WM * (BM / WM), n_base + wave / WM * (BN / WN), acc, split,
                                       lds + wave * tile_scratch_bytes<Pipe::TM, Pipe::TN>());
}

// Tiles of BM x BN on BlockPipe (tile.h), which take a compute unit whole.  A tile is as large as leaves most units one: what bounds
// it is what a unit can pull, 32 KiB under way at a time, so 256 x 160 x 64 takes 0.8 us where the matrix instructions alone need 0.72 and 128 x 128
// x 64 0.45 where they need 0.31 (busy for 0.51 and 0.36 of a unit's time in 2048 x 4800 x 1600 and 2048 x 1600 x 1600); around that 5 to 11 us of
// first loads (2), last stores (1 to 4) and launch.  Measured with operands from memory (us, in brackets TilePipe's best form and the vendor's library):
// 2048 x 4800 x 1600 with keys and values into the cache 35 (50, 47 with their copy); 1295 x 3072 x 1024 likewise 17.6 (20, 24.7); into the residual stream
// 1959 x 1024 x 4096 27 (28, 31), 1959 x 1600 x 6400 54 (56, 61), 2048 x 1600 x 1600 22.7 (22.6, 24.3); 1295 x 4096 x 1024 with a GELU 22 (23, 25); 4096 x 1600 x
// 6400 87 (99, 95).
// Tried: tiles of 256 x 208 and 256 x 256 (2048 x 6400 x 1600 42 us without an epilogue, the library 37, with one 164 registers spilled); a ninth wave that
// asks for lines some turns ahead (55.8 -> 55.7 at 2048 x 1600 x 6400: requests bound it); W packed by tiles (2 to 8 % faster, a third copy of the weights).
template <typename T, int BM, int BN, int WM, int WN, int SA, int SW>
__global__ void __launch_bounds__(WM * WN * 64, 2)
gemm_tile_blocks_kernel(const T* __restrict__ A, int64_t lda, const T* __restrict__ W, int M, int N,
                        int K, Epilogue epi, int tiles_m, int tiles_n, int group_m) {
  typedef BlockPipe<T, BM, BN, WM, WN, SA, SW> Pipe;
  constexpr int ROW_K = 8 * Mma<T>::ELEMS;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];   // SA stages of A's rows, SW of W's
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tile = xcd_contiguous(blockIdx.x, tiles_m * tiles_n);
  const int per_group = group_m * tiles_n, first = tile / per_group * group_m, rest = tile % per_group;
  const int rows_m = group_m < tiles_m - first ? group_m : tiles_m - first;
  const int m_base = (first + rest % rows_m) * BM, n_base = rest / rows_m * BN;
  const int split = blockIdx.z, splits = gridDim.z;
  const int k_tiles = K / ROW_K;
  const int kt_begin = (int)((int64_t)k_tiles * split / splits);
  const int count = (int)((int64_t)k_tiles * (split + 1) / splits) - kt_begin;
  floatx4 acc[Pipe::TN][Pipe::TM];
#pragma unroll
  for (int bn = 0; bn < Pipe::TN; ++bn)
#pragma unroll
    for (int bm = 0; bm < Pipe::TM; ++bm) acc[bn][bm] = floatx4{0.f, 0.f, 0.f, 0.f};
  Pipe::template multiply<unsigned>(
      lds, reinterpret_cast<const unsigned char*>(A) + (int64_t)kt_begin * TILE_ROW_BYTES,
      reinterpret_cast<const unsigned char*>(W) + (int64_t)kt_begin * TILE_ROW_BYTES, count,
      [&](int tile_row, bool from_w) {
        const int row = (from_w ? n_base : m_base) + tile_row, limit = from_w ? N : M;
        return (int64_t)(row < limit ? row : limit - 1) * (from_w ? (int64_t)K : lda) * (int64_t)sizeof(T);
      },
      acc);
  __syncthreads();
  epilogue_blocks<T, Pipe::TM, Pipe::TN>(epi, M, N, m_base + wave % WM * (BM / WM), n_base + wave / WM * (BN / WN), acc, split,
                                         lds + wave * block_scratch_bytes<Pipe::TM, Pipe::TN>());
}

// Float products of many rows on the bfloat16 matrix instructions, sixteen times the rate of the float ones.
// A float is the sum of three bfloat16 values (the nearest to it, the nearest to what that leaves, the rest, which has at most
// seven bits) and a product of two floats the sum of nine products of such parts, each exact in 32 bits.  The six
// largest are added up in 32 bits, the smallest first.  The three left out come to less than 2^-24 of the product, as much as rounding
// it to 32 bits may cost: over all mantissas the second part is at most 2^-8.005 of a float and the third 2^-17.002 (with the
// second part cut off instead of rounded 2^-16.01, and twice as much left out), 2^-27.5 (root of the mean square) over drawn ones, of either sign.
// Beside that a sum is rounded 6 K / 16 times where the float instructions, which do not round products, round it K / 2 times and more:
// against 64 bits the error of normal values is 0.67 of theirs at K = 32, 0.85 at K = 768, 0.88 at K = 3072.
// A tile goes from memory to registers (two tiles of K = 32 on their way), is cut there into its parts, every value once for
// the whole work-group, and lies in LDS as three planes of bfloat16 in three stages: the tile that is multiplied, the
// next one, whose first operands are read behind the multiplications of the second half of this one, and the one being cut.
// One barrier a tile; eight waves, two to a SIMD, so that one's cutting fills the other's matrix instructions.
// A value beyond the largest bfloat16, an infinity or a NaN makes parts whose products are not the floats' (infinity times
// a part that is zero): they all leave a sum that is not finite, and a tile with such a sum is made again on the float
// instructions, all waves together, operands straight from memory (2298 x 3072 x 768 called alone, us: finite 86, one NaN 151, every value
// NaN 209, where the float instructions alone take 118; with a lane making its own sums again one after the other 1,092 and 11,336).
// Values below 2^-110 lose what falls below the smallest bfloat16, 2^-134 each at most.  (To look for such values while they are cut and
// make their tiles again costs every product 5 to 8 %: 66 -> 72 us for 2298 x 2304 x 768.)
// What bounds it: 1.05 us for a tile of 128 x 128 x 32 where the matrix instructions take 0.64; 0.73 without the loads from memory and
// the cutting, the same with four tiles on their way in place of two: a compute unit's requests (256 lines a tile), not their
// latency.  Measured (us, float instructions / 128 x 64 / 128 x 128): 400 x 3072 x 768 33 / 23 / 30; 2298 x 768 x 768
// 35 / 24 / 31; 2298 x 2304 x 768 85 / 68 / 66; 2298 x 3072 x 768 105 / 90 / 71; 2298 x 768 x 3072 in two slices 108 / 84 / 66;
// 4096 x 1600 x 6400 800 / 653 / 493 (170 TFLOP/s).  Not taken: four waves (every wave's cutting shows: 554 for the last), 64 x 64
// tiles (19.0 where the float instructions take 18.8: a unit alone waits for its lines either way), matrix instructions
// and cutting interleaved one by one by hand (the same).
struct FloatParts {
  int part[3];
};
__device__ __forceinline__ FloatParts float_parts(float x0, float x1) {      // of two floats, a pair to a word
  typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
  FloatParts p;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const bf16x2 near = {(bf16_t)x0, (bf16_t)x1};
    p.part[i] = __builtin_bit_cast(int, near);
    x0 -= __builtin_bit_cast(float, p.part[i] << 16);
    x1 -= __builtin_bit_cast(float, p.part[i] & (int)0xffff0000);
  }
  return p;
}

template <int BM, int BN, int WM, int WN>
__global__ void __launch_bounds__(WM * WN * 64)
gemm_tile_parts_kernel(const float* __restrict__ A, int64_t lda, const float* __restrict__ W, int M, int N,
                       int K, Epilogue epi, int tiles_m, int tiles_n, int group_m) {
  constexpr int ROWS = BM + BN, THREADS = WM * WN * 64;
  constexpr int PLANE_BYTES = ROWS * 64, STAGE_BYTES = 3 * PLANE_BYTES;       // a row: 32 values of K in bfloat16
  constexpr int STEP = THREADS / 8, LOADS = ROWS / STEP;                      // eight lanes a row's 128 bytes
  constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
  constexpr int SETS = 2;                         // tiles on their way from memory
  static_assert(ROWS % STEP == 0 && BM % STEP == 0 && TM >= 1 && TN >= 1, "whole loads and whole blocks for every wave");
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];         // [3][3 planes][ROWS][64 bytes]
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int wm = wave % WM, wn = wave / WM;
  const int l32 = lane & 31, g = lane >> 5;
  const int tile = xcd_contiguous(blockIdx.x, tiles_m * tiles_n);
  // (an XCD's run of tiles is a block of group_m by as many columns, about square: it pulls the fewest rows of A and W)
  const int per_group = group_m * tiles_n, first = tile / per_group * group_m, rest = tile % per_group;
  const int rows_m = group_m < tiles_m - first ? group_m : tiles_m - first;
  const int m_base = (first + rest % rows_m) * BM, n_base = rest / rows_m * BN;
  const int split = blockIdx.z, splits = gridDim.z;
  const int k_tiles = K / 32;
  const int kt_begin = (int)((int64_t)k_tiles * split / splits);
  const int count = (int)((int64_t)k_tiles * (split + 1) / splits) - kt_begin;

  const int row = tid >> 3, quad = tid & 7;
  unsigned off[LOADS];
  int put[LOADS];
#pragma unroll
  for (int j = 0; j < LOADS; ++j) {
    const int stage_row = row + STEP * j;
    const bool from_w = STEP * j >= BM;
    int at = from_w ? n_base + stage_row - BM : m_base + stage_row;
    const int limit = from_w ? N : M;
    at = at < limit ? at : limit - 1;
    off[j] = (unsigned)(((int64_t)at * (from_w ? (int64_t)K : lda) + quad * 4) * 4);
    put[j] = stage_row * 64 + (((quad >> 1) ^ ((stage_row >> 2) & 3)) << 4) + (quad & 1) * 8;
  }
  const unsigned char* a_bytes = reinterpret_cast<const unsigned char*>(A) + (int64_t)kt_begin * TILE_ROW_BYTES;
  const unsigned char* w_bytes = reinterpret_cast<const unsigned char*>(W) + (int64_t)kt_begin * TILE_ROW_BYTES;
  floatx4 held[SETS][LOADS];
  int fetched = 0;
  auto fetch = [&](floatx4* set, int j) {
    set[j] = *reinterpret_cast<const floatx4*>((STEP * j >= BM ? w_bytes : a_bytes) + off[j]);
  };
  auto advance = [&] {         // (no branch: behind the last tile comes the last again)
    const int64_t step = ++fetched < count ? TILE_ROW_BYTES : 0;
    a_bytes += step;
    w_bytes += step;
  };
  auto cut = [&](const floatx4* set, int j, int stage) {
    unsigned char* base = lds + stage * STAGE_BYTES + put[j];
    const FloatParts lo = float_parts(set[j][0], set[j][1]), hi = float_parts(set[j][2], set[j][3]);
#pragma unroll
    for (int p = 0; p < 3; ++p) *reinterpret_cast<int2*>(base + p * PLANE_BYTES) = make_int2(lo.part[p], hi.part[p]);
  };
  int w_rd[2], a_rd[2];        // (blocks of 32 rows lie 2,048 bytes apart, the swizzle repeats every sixteen rows)
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    const int chunk = ((2 * kk + g) ^ ((l32 >> 2) & 3)) << 4;
    a_rd[kk] = (wm * (BM / WM) + l32) * 64 + chunk;
    w_rd[kk] = (BM + wn * (BN / WN) + l32) * 64 + chunk;
  }
  int4v op[2][3][TM + TN];     // of a half of a tile (sixteen values of K): the planes of the wave's blocks of A, then of W
  constexpr int READS = 3 * (TM + TN);
  auto read = [&](int stage, int kk, int r) {
    const int p = r / (TM + TN), b = r % (TM + TN);
    const unsigned char* base = lds + stage * STAGE_BYTES + p * PLANE_BYTES;
    op[kk][p][b] = *reinterpret_cast<const int4v*>(base + (b < TM ? a_rd[kk] + b * 2048 : w_rd[kk] + (b - TM) * 2048));
  };
  floatx16 acc[TN][TM];
#pragma unroll
  for (int bn = 0; bn < TN; ++bn)
#pragma unroll
    for (int bm = 0; bm < TM; ++bm)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[bn][bm][r] = 0.f;
  auto meet = [&] {            // this wave's planes are written; its loads from memory stay on their way
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // one tile: twelve products of parts (six to a half), beside each a share of the reads of the half after it, of the
  // cutting of the tile after the next and of the loads of the one SETS behind that
  int now = 0, next = 1, free = 2;              // stages
  auto turn = [&](floatx4* set) {
    constexpr int OF_W[6] = {0, 2, 1, 0, 1, 0}, OF_A[6] = {2, 0, 1, 1, 0, 0};      // the smallest products first
#pragma unroll
    for (int c = 0; c < 12; ++c) {
      const int kk = c / 6, p = c % 6;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int bn = 0; bn < TN; ++bn)
#pragma unroll
        for (int bm = 0; bm < TM; ++bm)
          Mma<bf16_t>::block32(acc[bn][bm], op[kk][OF_W[p]][TM + bn], op[kk][OF_A[p]][bm]);
#pragma unroll
      for (int r = 0; r < READS; ++r)
        if (r * 6 / READS == p) read(kk == 0 ? now : next, kk ^ 1, r);
#pragma unroll
      for (int j = 0; j < LOADS; ++j)
        if (j * 12 / LOADS == c) {
          cut(set, j, free);
          fetch(set, j);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    advance();
    meet();
    const int was = now;
    now = next, next = free, free = was;
  };
  if (count > 0) {
#pragma unroll
    for (int t = 0; t < SETS + 2; ++t) {
#pragma unroll
      for (int j = 0; j < LOADS; ++j) {
        if (t >= SETS) cut(held[t - SETS], j, t - SETS);
        fetch(held[t % SETS], j);
      }
      advance();
    }
    meet();
#pragma unroll
    for (int r = 0; r < READS; ++r) read(0, 0, r);
    int left = count;
    for (; left >= SETS; left -= SETS)
#pragma unroll
      for (int t = 0; t < SETS; ++t) turn(held[(t + 2) % SETS]);
#pragma unroll
    for (int t = 0; t < SETS - 1; ++t)
      if (t < left) turn(held[(t + 2) % SETS]);
  }

  bool finite = true;
#pragma unroll
  for (int bn = 0; bn < TN; ++bn)
#pragma unroll
    for (int bm = 0; bm < TM; ++bm)
#pragma unroll
      for (int r = 0; r < 16; ++r) finite = finite && fabsf(acc[bn][bm][r]) < INFINITY;
  if (__syncthreads_or(!finite)) {      // the whole tile again, on the float instructions
    const float* rows[TM + TN];
#pragma unroll
    for (int b = 0; b < TM + TN; ++b) {
      const int at = b < TM ? m_base + wm * (BM / WM) + b * 32 + l32 : n_base + wn * (BN / WN) + (b - TM) * 32 + l32;
      const int limit = b < TM ? M : N;
      rows[b] = (b < TM ? A : W) + (int64_t)(at < limit ? at : limit - 1) * (b < TM ? lda : (int64_t)K) + (int64_t)kt_begin * 32 + 4 * g;
    }
#pragma unroll
    for (int bn = 0; bn < TN; ++bn)
#pragma unroll
      for (int bm = 0; bm < TM; ++bm)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[bn][bm][r] = 0.f;
#pragma nounroll
    for (int i = 0; i < count; ++i) {
      int4v of[4][TM + TN];
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int b = 0; b < TM + TN; ++b) of[kk][b] = *reinterpret_cast<const int4v*>(rows[b] + (int64_t)i * 32 + kk * 8);
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int bn = 0; bn < TN; ++bn)
#pragma unroll
          for (int bm = 0; bm < TM; ++bm) Mma<float>::block32(acc[bn][bm], of[kk][TM + bn], of[kk][bm]);
    }
  }
  __syncthreads();
  epilogue_tile<float, TM, TN>(epi, M, N, m_base + wm * (BM / WM), n_base + wn * (BN / WN), acc, split,
                               lds + wave * tile_scratch_bytes<TM, TN>());
}

// What bounds it at a decode step's sizes, from clocks inside the kernel (768 x 768, one row, us): from one kernel's last wave to the
// next one's first 1.45, its waves' start 0.2, addresses and loads 0.35, memory 0.35, the waves' meeting and the epilogue 0.4 (with
// a GELU 0.8).  So beside enough work-groups (splitting K is for products of few columns) what counts is the chain of
// instructions of one work-group, and the loads that its compute unit takes, 16 cycles each whatever they bring:
//   addresses are a scalar base and a 32-bit offset a lane, from numbers that the host has worked out (SkinnyOperands); a batch's loads
//   have scalar branches between them and nothing else; K's partial chunk is outside the batches;
//   up to eight rows (four) two (four) chunks of the activations come with one load, and two of the weights where a work-group has
//   eight columns (AP, WP below: 768 x 3072, one row 4.8 -> 4.3; 1600 x 1600, eight rows 4.3 -> 4.1);
//   what depends on a table of the step is looked up by a wave that streams nothing or through the scalar cache (EpilogueTables): as a
//   streaming wave's vector loads it stood behind all the weights, a second trip to memory in every product;
//   the epilogue takes one value a lane (VALUES below: 3072 x 768 with a GELU 3.7 -> 3.4).
// In all, against a kernel with none of these (weights from memory, in a HIP graph, us): one row 768 x 768 3.1 -> 2.7, 768 x 3072 5.2 ->
// 4.3, 3072 x 768 with a norm and a GELU 5.1 -> 4.2; eight rows 4800 x 1600 6.0 -> 5.4, 6400 x 1600 with a GELU 6.9 -> 6.1, 1600 x 6400
// in five slices 6.4 -> 6.1, 18432 x 2048 16.5 -> 15.5; 64 rows 1600 x 6400 in five 11.4 -> 10.1.  Tried: loads without branches
// (chunks that do not exist read again: 5.2 -> 5.5 for 768 x 3072), lanes without a row or column masked out of the loads (no
// gain: a load costs its 16 cycles), the bias ahead of the weights (2.7 -> 2.9).
// MT row blocks of 16 (activations) by NT column blocks of 16 (weights) per work-group.  With
// more than 16 rows the activations a work-group reads (all rows, its whole K range) outweigh its
// weights, and they are read once per work-group: two column blocks halve that traffic.
//
// QPL > 0 (bfloat16, up to 16 rows): the activations are not read from memory but made here, as
// the normalised rows of the float32 residual stream (NormOperand): the norm that would
// otherwise be a kernel of its own in front of this one.  Every work-group normalises all rows
// (a wave takes rows w and w + 8: the row in its registers, QPL quads of four floats per lane,
// statistics as wave reductions) and leaves them in LDS as bfloat16, where the multiplication
// reads its operand.  The rows' loads are issued before the first batch of weights, so the
// statistics are computed while the weights are on their way.
__device__ float bt_norm_zeros[4] = {0.f, 0.f, 0.f, 0.f};

// Eight waves that stream, and in some forms a ninth beside them (EpilogueTables).
constexpr bool skinny_ninth(int kind, int mt, int nt, int u) {
  return nt == 1 && ((kind == EPILOGUE_QKV && mt * u < 16) || (kind == EPILOGUE_TURN && mt == 1));
}
constexpr int skinny_threads(int waves, int kind, int mt, int nt, int u) { return (waves + skinny_ninth(kind, mt, nt, u)) * 64; }
// Waves a SIMD must have room for: two work-groups of eight waves a compute unit for forms of one block.  (Those of two blocks take 97 to 119
// registers and so have room too.)
constexpr int skinny_occupancy(int mt, int nt, int qpl) { return mt == 1 && nt == 1 && qpl == 0 ? 4 : 2; }

// Of a load that holds `16 / ROWS` chunks of ROWS rows in every sixteen lanes, the operand of chunk `sub`: its rows in the first ROWS lanes.
template <int ROWS>
__device__ __forceinline__ int4v lanes_down(int4v v, int sub) {      // (sub: a constant where this is used)
  if (ROWS == 16 || sub == 0) return v;
  int4v r;
#pragma unroll
  for (int i = 0; i < 4; ++i)        // row_ror:16 - sub * ROWS: lane j takes what lane j + sub * ROWS holds
    r[i] = ROWS == 8 ? lane_moved<0x128>(v[i]) : sub == 1 ? lane_moved<0x12c>(v[i]) : sub == 2 ? lane_moved<0x128>(v[i]) : lane_moved<0x124>(v[i]);
  return r;
}

// The skinny kernel's operands as its addresses need them, in one line of the arguments (64 bytes).
// tile_columns: how many of its 16 * NT output columns a work-group really owns (a multiple of
// four).  Fewer than all of them is for balance: 300 work-groups of 16 columns leave 44 of 256
// compute units with twice the bytes of the others, 400 of 12 columns leave every unit at most
// 24 columns.  The lanes of the columns left out repeat the last real one and store nothing.
// W is [N][K], or packed: for each work-group's `tile_columns` columns the chunks of K one
// after the other, [group][chunk][tile_columns][64 bytes], K and the last group padded with zeros:
// a wave's load of a chunk is then one contiguous run of bytes and a work-group reads one
// contiguous block front to back.  A is row-major or chunk-major (activation_offset in common.h): the
// 64 lanes of an operand load then read one contiguous KiB.
struct SkinnyOperands {
  const void* W;
  const void* A;
  int64_t w_group;                 // bytes from a work-group's first column to the next one's
  int w_step, a_step;              // bytes from a chunk of 64 bytes of K to the next
  unsigned w_pitch, a_pitch;       // bytes from a column to the next, from a row to the next (of the form for far operands: sixteens of bytes)
  int whole, rest;                 // whole chunks of K, values behind them
  int M, N, tile_columns, splits;
};
template <typename T>
static SkinnyOperands skinny_operands(const void* A, int64_t lda, const void* W, int M, int N, int K, int splits, int columns, int packed,
                                      int a_rows, bool far = false) {
  constexpr int CHUNK = 64 / (int)sizeof(T);
  SkinnyOperands o;
  o.W = W;
  o.A = A;
  o.whole = K / CHUNK;
  o.rest = K % CHUNK;
  o.w_step = packed ? columns * 64 : 64;
  o.w_pitch = (unsigned)((packed ? 64 : K * sizeof(T)) / (far ? 16 : 1));
  o.w_group = packed ? (int64_t)((K + CHUNK - 1) / CHUNK) * o.w_step : (int64_t)columns * K * (int64_t)sizeof(T);
  o.a_step = a_rows > 0 ? a_rows * 64 : 64;
  o.a_pitch = (unsigned)((a_rows > 0 ? 64 : lda * (int64_t)sizeof(T)) / (far ? 16 : 1));
  o.M = M;
  o.N = N;
  o.tile_columns = columns;
  o.splits = splits;
  return o;
}

// FAR: with offsets of 64 bits, for rows or columns that lie or reach 2 GiB apart (launch_skinny_far).
template <typename T, int MT, int NT, int U, int WAVES, int QPL, int KIND, int AP, int WP, int FAR = 0>
__global__ void __launch_bounds__(skinny_threads(WAVES, KIND, MT, NT, U), skinny_occupancy(MT, NT, QPL))
gemm_skinny_kernel(SkinnyOperands o, Epilogue epi, NormOperand norm) {
  constexpr int ELEMS = Mma<T>::ELEMS;      // K values in a lane's 16-byte load
  constexpr bool NORM = QPL > 0, NINTH = skinny_ninth(KIND, MT, NT, U), OWN_SINES = KIND == EPILOGUE_TURN && !NINTH,
                 OWN_PLACES = KIND == EPILOGUE_QKV && !NINTH;
  static_assert(!NORM || (MT == 1 && sizeof(T) == 2), "the fused norm is for bfloat16 and up to 16 rows");
  extern __shared__ __attribute__((aligned(16))) unsigned char normed[];   // NORM: [16][K * 2 + 16] bytes
  const int M = o.M, whole = o.whole, rest = o.rest, splits = o.splits;
  const int K = whole * (4 * ELEMS) + rest, normed_pitch = K * 2 + 16;      // the 16 bytes spread the rows over the LDS banks
  // (72 floats for eight blocks with tables: 80 KiB and the tables would keep a second work-group out.  Into the cache, us at 80 / 72:
  // 33 rows of 9216 x 3072 30.2 / 28.2, 64 rows 40.5 / 38.0, 64 rows of 18432 x 2048 43.4 / 39.3.  Without tables 80 KiB are half of a unit's
  // LDS and 80 floats the faster way: 64 rows of 6400 x 1600 with a GELU 11.2 / 11.3, 1600 x 6400 in five slices 10.4 / 10.5)
  constexpr int GROUP_PITCH = MT * NT > 4 && OWN_PLACES ? 72 : 80;
  __shared__ __attribute__((aligned(16))) float red[WAVES][MT * NT][4][GROUP_PITCH];
  __shared__ EpilogueTables<OWN_SINES ? (int)EPILOGUE_COMMON : KIND, MT, NT> tables;
  // the wave's number is the same in all its lanes: saying so keeps every test on it a scalar
  // branch, which costs no wait for loads in flight (a divergent one does)
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int n_base = blockIdx.x * o.tile_columns;
  const int n_end = n_base + o.tile_columns < o.N ? n_base + o.tile_columns : o.N;   // one past this work-group's last column
  if constexpr (NINTH) {
    if (wave == WAVES) {                    // nothing here waits for weights
      tables.fill(epi, M, n_base);
      if constexpr (NORM) __syncthreads();
      __syncthreads();
      return;
    }
  }
  const int i16 = lane & 15, g = lane >> 4;
  const int split = blockIdx.y;
  // Addresses are a uniform base and a lane's offset of 32 bits, which one addition moves from chunk to chunk.
  typedef typename std::conditional<FAR != 0, uint64_t, unsigned>::type Offset;
  constexpr Offset PITCHES = FAR ? 16 : 1;
  const char* w_base = static_cast<const char*>(o.W) + (int64_t)blockIdx.x * o.w_group;
  const char* a_base = static_cast<const char*>(o.A);
  const int c_first = split * WAVES + wave, stride = splits * WAVES;
  const Offset w_jump = (Offset)stride * o.w_step, a_jump = (Offset)stride * o.a_step;
  // AP chunks of the activations to a load where the rows are few enough, WP of the weights: sixteen lanes hold 16 / AP rows of
  // the wave's chunk u, then of u + 1, ..., and a rotation in the row of lanes brings the later ones down.  (Lanes whose chunk
  // does not exist read the last whole one; what they hold is not multiplied.)
  constexpr int A_ROWS = 16 / AP, W_COLS = 16 / WP;
  static_assert(U % AP == 0 && U % WP == 0 && (MT == 1 || AP == 1) && (NT == 1 || WP == 1), "whole loads of one block");
  Offset w_off[NT], a_off[MT], w_most = 0, a_most = 0;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int n = WP > 1 ? i16 % W_COLS : nt * 16 + i16, last = n_end - n_base - 1;
    const Offset column = (Offset)(n < last ? n : last) * o.w_pitch * PITCHES + g * 16;
    w_off[nt] = column + (Offset)(c_first + i16 / W_COLS * (WP > 1 ? stride : 0)) * o.w_step;
    if (WP > 1) w_most = column + (Offset)(whole - 1) * o.w_step;
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {         // (rows beyond M repeat the last; the epilogue drops them)
    const int m = AP > 1 ? i16 % A_ROWS : mt * 16 + i16;
    const Offset row = (Offset)(m < M ? m : M - 1) * o.a_pitch * PITCHES + g * 16;
    a_off[mt] = row + (Offset)(c_first + i16 / A_ROWS * (AP > 1 ? stride : 0)) * o.a_step;
    if (AP > 1) a_most = row + (Offset)(whole - 1) * o.a_step;
  }
  auto from = [](const char* base, Offset off) { return *reinterpret_cast<const int4v*>(base + off); };
  floatx4 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = floatx4{0.f, 0.f, 0.f, 0.f};
  // A batch: all its loads, then what waits for them.  (A place whose chunk does not exist is neither loaded nor multiplied.)
  int4v wv[U / WP][NT], av[U / AP][MT];
  auto issue = [&](int c0) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if ((u % WP == 0 || (!NORM && u % AP == 0)) && c0 + u * stride < whole) {
        // (a place's lanes add their offsets here and not before the batch's first load, which kept them all in registers at once: the forms of
        // eight chunks and two blocks took 138, so that one work-group of theirs shared a compute unit with no other.  18432 x 2048, nine rows
        // 18.7 us, so 16.5.  Batches of two chunks have the registers, and the additions between their loads only cost: 64 rows of 50257 x 1600
        // 61.8 us, so 60.4; nor do the plain epilogues' forms with several chunks a load need it: eight rows of 18432 x 2048 19.5, so 19.0, while into the
        // cache one row of 9216 x 3072 takes 13.5 with it and 15.7 without.  Not volatile: behind an assembly statement that may do anything loads no longer go through the scalar cache.)
        Offset w_to = u * w_jump, a_to = u * a_jump;
        if constexpr (U > 2 && (AP == 1 || KIND != EPILOGUE_COMMON)) asm("" : "+s"(w_to), "+s"(a_to));
        if (u % WP == 0) {
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) {
            const Offset off = w_off[nt] + w_to;
            wv[u / WP][nt] = from(w_base, WP > 1 && off > w_most ? w_most : off);
          }
        }
        if (!NORM && u % AP == 0) {
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            const Offset off = a_off[mt] + a_to;
            av[u / AP][mt] = from(a_base, AP > 1 && off > a_most ? a_most : off);
          }
        }
      }
  };
  auto multiply = [&](int c0) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (c0 + u * stride < whole) {
        int4v a[MT];
        if constexpr (NORM) {               // the operand from LDS
          a[0] = *reinterpret_cast<const int4v*>(normed + (i16 < M ? i16 : M - 1) * normed_pitch + (c0 + u * stride) * 64 + g * 16);
        } else {
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) a[mt] = lanes_down<A_ROWS>(av[u / AP][mt], u % AP);
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const int4v w = lanes_down<W_COLS>(wv[u / WP][nt], u % WP);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) Mma<T>::block16(acc[mt][nt], w, a[mt]);
        }
      }
  };
  int c0 = c_first;
  // (With batches of two chunks the lookups' two trips are spread over the kernel: right behind the first batch, which is soon there,
  // 33 rows of 4800 x 1600 took 9.7 us, so 9.5.  With more chunks they are over before the weights come; one row with a norm 6.5 spread, so 6.3.)
  TokenPlaces<16 * MT, WAVES> places;       // OWN_PLACES only
  constexpr bool SPREAD = MT == 4;
  auto look_up = [&]() {
    if constexpr (OWN_PLACES) {
      places.ask(epi, M, wave);
      if constexpr (!SPREAD) {
        places.look(epi);
        places.put(wave, tables);
      }
    }
  };
  if constexpr (NORM) {
    const int quads = K >> 2;
    const float4* g4 = reinterpret_cast<const float4*>(norm.gamma);
    const float4* b4 = reinterpret_cast<const float4*>(norm.beta ? norm.beta : bt_norm_zeros);
    float4 xv[QPL], gv[QPL], bv[QPL];
    auto load_row = [&](int r) {
      const float4* xr = reinterpret_cast<const float4*>(norm.x + (int64_t)r * norm.ldx);
#pragma unroll
      for (int q = 0; q < QPL; ++q) {
        int c = lane + 64 * q;
        int cc = c < quads ? c : 0;          // lanes beyond the row read its start; the result is never used
        xv[q] = xr[cc];
        gv[q] = g4[cc];
        bv[q] = b4[norm.beta ? cc : 0];
      }
    };
    auto normalise_row = [&](int r) {
      float part = 0.f;
#pragma unroll
      for (int q = 0; q < QPL; ++q)
        if (lane + 64 * q < quads)
          part += norm.kind == 0 ? (xv[q].x + xv[q].y + xv[q].z + xv[q].w)
                                 : (xv[q].x * xv[q].x + xv[q].y * xv[q].y + xv[q].z * xv[q].z + xv[q].w * xv[q].w);
      float total = wave_sum(part);
      float mean = 0.f, rstd;
      if (norm.kind == 0) {
        mean = total / (float)K;
        float sq = 0.f;
#pragma unroll
        for (int q = 0; q < QPL; ++q)
          if (lane + 64 * q < quads) {
            float a0 = xv[q].x - mean, a1 = xv[q].y - mean, a2 = xv[q].z - mean, a3 = xv[q].w - mean;
            sq += a0 * a0 + a1 * a1 + a2 * a2 + a3 * a3;
          }
        rstd = 1.0f / sqrtf(wave_sum(sq) / (float)K + norm.eps);
      } else {
        rstd = 1.0f / sqrtf(total / (float)K + norm.eps);
      }
#pragma unroll
      for (int q = 0; q < QPL; ++q) {
        int c = lane + 64 * q;
        if (c < quads) {
          bf16x4 y = {(bf16_t)((xv[q].x - mean) * rstd * gv[q].x + bv[q].x), (bf16_t)((xv[q].y - mean) * rstd * gv[q].y + bv[q].y),
                      (bf16_t)((xv[q].z - mean) * rstd * gv[q].z + bv[q].z), (bf16_t)((xv[q].w - mean) * rstd * gv[q].w + bv[q].w)};
          *reinterpret_cast<bf16x4*>(normed + r * normed_pitch + c * 8) = y;
        }
      }
    };
    if (wave < M) load_row(wave);            // (the wave's number is scalar: no lane-dependent branch)
    issue(c0);                               // the weights of the first batch, behind the row
    look_up();
    if (wave < M) normalise_row(wave);
    if (wave + WAVES < M) {
      load_row(wave + WAVES);
      normalise_row(wave + WAVES);
    }
    __syncthreads();
  } else {
    issue(c0);
    look_up();
  }
  // A thread finishes one output value, or VALUES neighbours of a row: what is added to them is fetched now, behind the first batch,
  // so that no load is left on the critical path after the last multiply.
  constexpr int COLUMNS = 16 * NT, THREADS = 64 * WAVES, VALUES = (16 * MT * COLUMNS + THREADS - 1) / THREADS;
  static_assert(VALUES == 1 || VALUES == 2 || VALUES == 4, "neighbours inside four columns");
  const int out_m = tid * VALUES / COLUMNS, column = tid * VALUES % COLUMNS;
  float add[VALUES];
  epilogue_addends<KIND>(epi, M, n_end, out_m, n_base + column, split, add);
  TurnedPairs<VALUES> pairs;                // EPILOGUE_TURN only
  if constexpr (OWN_SINES) pairs.ask(epi, M, out_m, n_base + column);
  if constexpr (OWN_PLACES && SPREAD) places.look(epi);
  for (;;) {
    multiply(c0);
    c0 += U * stride;
    if (c0 >= whole) break;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) w_off[nt] += U * w_jump;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) a_off[mt] += U * a_jump;
    issue(c0);
  }
  // K's partial chunk, for the wave whose turn it is (widths that are no multiple of 64 bytes: one more trip to memory for them):
  // a group beyond K reads the last one inside, its weights are cleared
  if (rest != 0 && wave == whole % WAVES && split == whole / WAVES % splits) {
    const int keep = g * ELEMS < rest ? -1 : 0, inside = (rest / ELEMS - 1 - g) * 16 & ~keep;
    const int4v zero = {0, 0, 0, 0};
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int n = nt * 16 + i16, last = n_end - n_base - 1;
      const int4v w = from(w_base, (Offset)(n < last ? n : last) * o.w_pitch * PITCHES + (Offset)whole * o.w_step + g * 16 + inside);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const int m = mt * 16 + i16 < M ? mt * 16 + i16 : M - 1;
        const int4v a = NORM ? *reinterpret_cast<const int4v*>(normed + m * normed_pitch + whole * 64 + g * 16 + inside)
                             : from(a_base, (Offset)m * o.a_pitch * PITCHES + (Offset)whole * o.a_step + g * 16 + inside);
        Mma<T>::block16(acc[mt][nt], keep ? w : zero, a);
      }
    }
  }
  if constexpr (OWN_PLACES && SPREAD) places.put(wave, tables);
  if constexpr (OWN_SINES) pairs.work();
  // lane holds D[i][j]: i = 4 g + r the column, j = i16 the row.  (The groups lie 80 floats apart, or 72 where a lane reads four: what
  // sixteen lanes' quads, or 64 lanes' values of a block, are read from is then in 64 different banks.)
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
      *reinterpret_cast<floatx4*>(&red[wave][mt * NT + nt][g][i16 * 4]) = acc[mt][nt];
  __syncthreads();
  if (out_m < M) {                          // (whole quads of lanes: the turned pairs are together)
    const float* part = &red[0][out_m / 16 * NT + column / 16][column % 16 / 4][out_m % 16 * 4 + column % 4];
    typedef __attribute__((__vector_size__(VALUES * sizeof(float)))) float floats;
    float v[VALUES];
    floats share[WAVES];
#pragma unroll
    for (int w = 0; w < WAVES; ++w) share[w] = *reinterpret_cast<const floats*>(part + w * (MT * NT * 4 * GROUP_PITCH));
#pragma unroll
    for (int i = 0; i < VALUES; ++i) {
      v[i] = 0.f;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) v[i] += share[w][i];
      v[i] += add[i];
    }
    if constexpr (NINTH && KIND == EPILOGUE_TURN) {
#pragma unroll
      for (int p = 0; p < pairs.PAIRS; ++p) pairs.turn[p] = tables.turn[out_m][(column >> 1) + p];
    }
    epilogue_values<T, KIND>(epi, n_end, out_m, n_base + column, column, v, split, tables, pairs.turn);
  }
}

static int check_operands(const char* who, int elems, const void* A, int64_t lda, const void* W, int M, int N,
                          int K, const Epilogue& e, int splits) {
  if (N <= 0 || K <= 0) BT_REFUSE("%s: N %d and K %d must be positive", who, N, K);
  if (K % elems != 0 || lda % elems != 0)
    BT_REFUSE("%s: K %d and the row pitch %lld must be multiples of %d (16-byte loads)", who, K, (long long)lda, elems);
  if (((uintptr_t)A & 15) || ((uintptr_t)W & 15)) BT_REFUSE("%s: operands must be 16-byte aligned", who);
  if (e.mode < 0 || e.mode > 6 || e.out == nullptr) BT_REFUSE("%s: bad epilogue", who);
  if (e.mode == EPI_F32_ACT && (!e.out2 || e.n_q <= 0 || e.n_q >= N || e.n_q % 4 != 0))
    BT_REFUSE("%s: %d of %d columns in 32-bit, the others activated: a multiple of four, and a place for each", who, e.n_q, N);
  if (e.mode == EPI_TURN && (e.turn.pitch <= 0 || e.turn.pitch % 4 != 0 || N % e.turn.pitch != 0 || e.turn.at < 0 || e.turn.at % 2 != 0 ||
                             e.turn.dim <= 0 || e.turn.dim % 2 != 0 || e.turn.at + e.turn.dim > e.turn.pitch || !e.tok_pos || !e.turn.inv_freq || e.bias))
    BT_REFUSE("%s: heads of %d columns (a multiple of four) in %d, turned in neighbouring pairs from %d on (%d columns, both even), without a bias",
              who, e.turn.pitch, N, e.turn.at, e.turn.dim);
  if (splits < 1 || (splits > 1 && e.mode != EPI_F32))
    BT_REFUSE("%s: K can be split %d ways only into 32-bit partial sums", who, splits);
  if (e.out_rows != 0 && ((e.mode != EPI_STORE && e.mode != EPI_ACT && e.mode != EPI_F32_ACT) || e.out_rows < M))
    BT_REFUSE("%s: a chunk-major output of %d rows for %d rows (stored or activated results only)", who, e.out_rows, M);
  if (e.mode == EPI_QKV) {
    if (e.kv.head_dim <= 0 || e.kv.head_dim % 16 != 0)
      BT_REFUSE("%s: head size %d must be a multiple of 16", who, e.kv.head_dim);
    if (e.n_q % 16 != 0 || e.n_kv != e.kv.kv_heads * e.kv.head_dim || e.n_q + 2 * e.n_kv != N)
      BT_REFUSE("%s: fused projection of %d columns does not split into %d query and 2 x %d key/value columns",
                who, N, e.n_q, e.n_kv);
    if (!e.tok_seq || !e.tok_pos || !e.kv.blocks || !e.kv.keys || !e.kv.values)
      BT_REFUSE("%s: the key/value scatter needs token and cache tables", who);
  }
  return BT_OK;
}

template <typename T, int BM, int BN, int WM, int WN>
static void launch_tile(hipStream_t stream, const T* A, int64_t lda, const T* W, int M, int N, int K,
                        const Epilogue& epi, int splits) {
  int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  size_t lds = (size_t)2 * (BM + BN) * TILE_ROW_BYTES;
  auto kernel = gemm_tile_kernel<T, BM, BN, WM, WN>;
  if (lds > 64 * 1024)
    (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  hipLaunchKernelGGL(kernel, dim3(tiles_m * tiles_n, 1, splits), dim3(WM * WN * 64), lds, stream, A, lda, W, M, N,
                     K, epi, tiles_m, tiles_n);
}

// Rows of tiles that make a run of tiles of one XCD about square.
static int tile_group(int tiles_m, int tiles_n, int splits, int bm, int bn) {
  const int rows = (int)(sqrtf((float)tiles_m * tiles_n * splits / 8 * bn / bm) + 0.5f);
  return rows < 1 ? 1 : rows;
}

template <int BM, int BN, int WM, int WN, int STAGES, typename T>
static int launch_pipe(hipStream_t s, const T* a, int64_t lda, const T* w, int M, int N, int K, const Epilogue& epi, int splits) {
  typedef TilePipe<T, BM, BN, WM, WN, STAGES> Pipe;
  auto kernel = gemm_tile_pipe_kernel<T, BM, BN, WM, WN, STAGES>;
  const size_t stages = (size_t)STAGES * Pipe::STAGE_BYTES, scratch = (size_t)WM * WN * tile_scratch_bytes<Pipe::TM, Pipe::TN>();
  const size_t lds = stages > scratch ? stages : scratch;
  static bool raised = false;
  if (!raised) {
    hipError_t err = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err != hipSuccess) BT_REFUSE("gemm_tile: cannot get %zu bytes of LDS: %s", lds, hipGetErrorString(err));
    raised = true;
  }
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  hipLaunchKernelGGL(kernel, dim3(tiles_m * tiles_n, 1, splits), dim3(WM * WN * 64), lds, s, a, lda, w, M, N, K, epi, tiles_m,
                     tiles_n, tile_group(tiles_m, tiles_n, splits, BM, BN));
  return bt_check_launch("gemm_tile");
}

template <int BM, int BN, int WM, int WN, int SA, int SW, typename T>
static int launch_blocks(hipStream_t s, const T* a, int64_t lda, const T* w, int M, int N, int K, const Epilogue& epi, int splits) {
  typedef BlockPipe<T, BM, BN, WM, WN, SA, SW> Pipe;
  auto kernel = gemm_tile_blocks_kernel<T, BM, BN, WM, WN, SA, SW>;
  static_assert(WM * WN * block_scratch_bytes<Pipe::TM, Pipe::TN>() <= Pipe::BYTES, "the epilogue's rows fit into the stages");
  static bool raised = false;
  if (!raised) {
    hipError_t err = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, Pipe::BYTES);
    if (err != hipSuccess) BT_REFUSE("gemm_tile: cannot get %d bytes of LDS: %s", Pipe::BYTES, hipGetErrorString(err));
    raised = true;
  }
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  hipLaunchKernelGGL(kernel, dim3(tiles_m * tiles_n, 1, splits), dim3(WM * WN * 64), Pipe::BYTES, s, a, lda, w, M, N, K, epi, tiles_m,
                     tiles_n, tile_group(tiles_m, tiles_n, splits, BM, BN));
  return bt_check_launch("gemm_tile");
}

template <int BM, int BN, int WM, int WN>
static int launch_parts_form(hipStream_t s, const float* a, int64_t lda, const float* w, int M, int N, int K,
                             const Epilogue& epi, int splits) {
  auto kernel = gemm_tile_parts_kernel<BM, BN, WM, WN>;
  const size_t lds = (size_t)3 * 3 * (BM + BN) * 64;
  static bool raised = false;
  if (!raised) {
    hipError_t err = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err != hipSuccess) BT_REFUSE("gemm_tile: cannot get %zu bytes of LDS: %s", lds, hipGetErrorString(err));
    raised = true;
  }
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  hipLaunchKernelGGL(kernel, dim3(tiles_m * tiles_n, 1, splits), dim3(WM * WN * 64), lds, s, a, lda, w, M, N, K, epi, tiles_m,
                     tiles_n, tile_group(tiles_m, tiles_n, splits, BM, BN));
  return bt_check_launch("gemm_tile");
}

// The forms of the tile kernel for whole tiles of K.
static int launch_form(hipStream_t s, int variant, const bf16_t* a, int64_t lda, const bf16_t* w, int M, int N, int K,
                       const Epilogue& epi, int splits) {
  // A long K with one tile to a unit at most: the LDS is its own, and more tiles on their way hide more of the weights' way from
  // memory (cold weights, us: 200 x 1600 x 6400 28.1 -> 24.8; a shorter K pays for the longer start: 290 x 2048 x 1024 6.6 -> 7.3,
  // and prompts of 220 tokens at width 1,024, whose K is 2,048 at most, 1,009 -> 1,017).
  const bool alone = K / TILE_K / splits >= 48 && (int64_t)((M + 63) / 64) * ((N + 63) / 64) * splits <= 256;
  switch (variant) {
    case 2: return launch_blocks<128, 128, 4, 2, 4, 6>(s, a, lda, w, M, N, K, epi, splits);
    case 3: return launch_blocks<256, 160, 4, 2, 3, 3>(s, a, lda, w, M, N, K, epi, splits);
    case 4: return launch_pipe<64, 64, 2, 2, 3>(s, a, lda, w, M, N, K, epi, splits);
    case 5:
      if (alone) return launch_pipe<64, 64, 2, 2, 8>(s, a, lda, w, M, N, K, epi, splits);
      return launch_pipe<64, 64, 2, 2, 4>(s, a, lda, w, M, N, K, epi, splits);
    case 7: return launch_blocks<128, 256, 2, 4, 4, 3>(s, a, lda, w, M, N, K, epi, splits);
    case 8: return launch_blocks<64, 96, 4, 2, 8, 6>(s, a, lda, w, M, N, K, epi, splits);
    case 6:                                            // (64 x 128, which are nowhere the fastest, are 128 x 64)
    case 9: return launch_blocks<128, 64, 4, 2, 5, 8>(s, a, lda, w, M, N, K, epi, splits);
    case 10: return launch_blocks<128, 96, 4, 2, 5, 6>(s, a, lda, w, M, N, K, epi, splits);
    case 11: return launch_blocks<128, 160, 4, 2, 4, 4>(s, a, lda, w, M, N, K, epi, splits);
    case 12: return launch_blocks<128, 192, 2, 4, 4, 4>(s, a, lda, w, M, N, K, epi, splits);
    case 13: return launch_blocks<256, 96, 4, 2, 3, 5>(s, a, lda, w, M, N, K, epi, splits);
    case 14: return launch_blocks<256, 128, 4, 2, 3, 4>(s, a, lda, w, M, N, K, epi, splits);
  }
  BT_REFUSE("gemm_tile: unknown form %d", variant);
}
static int launch_form(hipStream_t s, int variant, const float* a, int64_t lda, const float* w, int M, int N, int K,
                       const Epilogue& epi, int splits) {
  switch (variant) {
    case 4:                // (three stages are for units that share their LDS: no rule wants them here)
    case 5: return launch_pipe<64, 64, 2, 2, 4>(s, a, lda, w, M, N, K, epi, splits);
    case 6: return launch_parts_form<128, 64, 4, 2>(s, a, lda, w, M, N, K, epi, splits);
    case 7: return launch_parts_form<128, 128, 2, 4>(s, a, lda, w, M, N, K, epi, splits);
  }
  BT_REFUSE("gemm_tile: unknown form %d", variant);
}

// dtype: 0 float, 1 bfloat16 (the codes of every entry point that takes both).
// variant: 1 = the general form; 2 .. 14 = launch_form's (a form that cannot take the operands is refused; float has the general form, 5 (4 is
// the same), 6 and 7); 0 = of float products the fastest form the operands allow, of bfloat16 ones the tiles of 64 x 64 where they can be
// taken (which form is the fastest is the caller's to say: kernels/library.py, tile_form).
// Float products take the tiles of 64 x 64 or the forms on parts wherever K is a multiple of 32 (the template's tile of 128 x 128
// takes a compute unit 2.4 us for 32 values of K and leaves most units idle where there are few tiles).  While the tiles of
// 64 x 64 have a unit each, they win: 0.65 us for 32 values of K where a tile of 128 x 64 on parts takes 0.73 (65 x 768 x 3072 62
// against 72; 1000 x 768 x 768 18.8 against 21.9).  Beyond, a unit's share comes in whole tiles of the forms on parts, one to a unit
// at a time, and the busiest unit decides: 128 x 128 takes 1.27 to 1.58 times as long as 128 x 64 for twice the work (figures
// with the kernel).
BT_EXPORT int bt_gemm_tile(void* stream, int dtype, const void* A, int64_t lda, const void* W, int M, int N, int K,
                           const Epilogue* epi, int splits, int variant) {
  if (M <= 0) return BT_OK;
  if (dtype != 0 && dtype != 1) BT_REFUSE("gemm_tile: element type %d is neither float nor bfloat16", dtype);
  if (epi->mode == EPI_F32_ACT) BT_REFUSE("gemm_tile: 32-bit and activated columns of one product are the skinny kernel's");
  if (epi->mode == EPI_TURN) BT_REFUSE("gemm_tile: turned columns are the skinny kernel's");
  int rc = check_operands("gemm_tile", dtype == 0 ? 4 : 8, A, lda, W, M, N, K, *epi, splits);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == 0) {
    const float *a = (const float*)A, *w = (const float*)W;
    const bool whole_ok = K % (TILE_ROW_BYTES / 4) == 0 && (int64_t)M * lda * 4 < ((int64_t)1 << 32) && (int64_t)N * K * 4 < ((int64_t)1 << 32);
    if (variant == 2 || variant == 3) BT_REFUSE("gemm_tile: of the variants 1 to 3 float products have the general form only, not variant %d", variant);
    if (variant >= 4 && !whole_ok) BT_REFUSE("gemm_tile: this form needs K %d to be a multiple of 32 and operands below 4 GiB", K);
    if (variant == 0 && whole_ok) {
      const int64_t rows = (M + 127) / 128 * (int64_t)splits;
      const int64_t rounds = (rows * ((N + 63) / 64) + 255) / 256, wide_rounds = (rows * ((N + 127) / 128) + 255) / 256;
      variant = (int64_t)((M + 63) / 64) * ((N + 63) / 64) * splits <= 256 ? 5 : 2 * rounds <= 3 * wide_rounds ? 6 : 7;
    }
    if (variant >= 4) return launch_form(s, variant, a, lda, w, M, N, K, *epi, splits);
    launch_tile<float, 128, 128, 2, 2>(s, (const float*)A, lda, (const float*)W, M, N, K, *epi, splits);
    return bt_check_launch("gemm_tile");
  }
  const bf16_t* a = (const bf16_t*)A;
  const bf16_t* w = (const bf16_t*)W;
  const int64_t four_gib = (int64_t)1 << 32;
  const bool whole_ok = K % TILE_K == 0 && (int64_t)M * lda * 2 < four_gib && (int64_t)N * K * 2 < four_gib;
  if (variant == 0) variant = whole_ok ? 5 : 1;
  if (variant != 1) {
    if (!whole_ok) BT_REFUSE("gemm_tile: this form needs K %d to be a multiple of 64 and operands below 4 GiB", K);
    return launch_form(s, variant, a, lda, w, M, N, K, *epi, splits);
  }
  launch_tile<bf16_t, 128, 128, 2, 2>(s, a, lda, w, M, N, K, *epi, splits);
  return bt_check_launch("gemm_tile");
}

template <typename T>
static void launch_skinny(hipStream_t s, const T* a, int64_t lda, const T* w, int M, int N, int K, const Epilogue& epi,
                          int splits, int columns, int packed, int a_rows) {
  dim3 grid((N + columns - 1) / columns, splits);
  const NormOperand none = {};
  const SkinnyOperands o = skinny_operands<T>(a, lda, w, M, N, K, splits, columns, packed, a_rows);
#define LAUNCH_SKINNY_FORM(MT, NT, U, KIND, AP, WP) \
  hipLaunchKernelGGL((gemm_skinny_kernel<T, MT, NT, U, 8, 0, KIND, AP, WP>), grid, dim3(skinny_threads(8, KIND, MT, NT, U)), 0, s, o, epi, none)
#define LAUNCH_SKINNY(MT, NT, U, AP, WP)                                                          \
  do {                                                                                            \
    if (epi.mode == EPI_TURN) LAUNCH_SKINNY_FORM(MT, NT, U, EPILOGUE_TURN, AP, WP);               \
    else if (epi.mode == EPI_QKV) LAUNCH_SKINNY_FORM(MT, NT, U, EPILOGUE_QKV, AP, WP);            \
    else if (epi.mode == EPI_F32_ACT) LAUNCH_SKINNY_FORM(MT, NT, U, EPILOGUE_TWO, AP, WP);        \
    else LAUNCH_SKINNY_FORM(MT, NT, U, EPILOGUE_COMMON, AP, WP);                                  \
  } while (0)
  // eight loads in flight where a wave has more than four chunks of K to go through (measured at
  // 17 and 32 rows: 6.4 -> 6.1 us and 6.6 -> 6.4 us for 4800 x 1600; with four chunks or fewer
  // the longer batch only adds loads that are skipped, 4.2 -> 4.4 us for 1600 x 1600 in two slices)
  constexpr int chunk = 4 * Mma<T>::ELEMS;
  const int per_wave = (((K + chunk - 1) / chunk + splits - 1) / splits + 7) / 8;
  if (M <= 16) {
    if (per_wave <= 4) {
      if (columns <= 16) LAUNCH_SKINNY(1, 1, 4, 1, 1); else LAUNCH_SKINNY(1, 2, 4, 1, 1);
    } else if (M <= 4) {
      // (up to twelve chunks a wave in one batch: 768 x 3072, one row 4.26 -> 4.04 us; four rows 1024 x 9216 in four slices 6.1 -> 5.7)
      if (columns <= 16 && per_wave > 8 && per_wave <= 12) {
        if (columns == 8) LAUNCH_SKINNY(1, 1, 12, 4, 2); else LAUNCH_SKINNY(1, 1, 12, 4, 1);
      } else if (columns == 8) {
        LAUNCH_SKINNY(1, 1, 8, 4, 2);
      } else if (columns <= 16) {
        LAUNCH_SKINNY(1, 1, 8, 4, 1);
      } else {
        LAUNCH_SKINNY(1, 2, 8, 4, 1);
      }
    } else if (M <= 8) {
      if (columns == 8) LAUNCH_SKINNY(1, 1, 8, 2, 2); else if (columns <= 16) LAUNCH_SKINNY(1, 1, 8, 2, 1); else LAUNCH_SKINNY(1, 2, 8, 2, 1);
    } else {
      if (columns <= 16) LAUNCH_SKINNY(1, 1, 8, 1, 1); else LAUNCH_SKINNY(1, 2, 8, 1, 1);
    }
  } else if (M <= 32) {
    if (per_wave > 4) {
      if (columns <= 16) LAUNCH_SKINNY(2, 1, 8, 1, 1); else LAUNCH_SKINNY(2, 2, 8, 1, 1);
    } else {
      if (columns <= 16) LAUNCH_SKINNY(2, 1, 4, 1, 1); else LAUNCH_SKINNY(2, 2, 4, 1, 1);
    }
  } else {
    if (columns <= 16) LAUNCH_SKINNY(4, 1, 2, 1, 1); else LAUNCH_SKINNY(4, 2, 2, 1, 1);
  }
#undef LAUNCH_SKINNY
#undef LAUNCH_SKINNY_FORM
}

// The same products (and the same sums) where an offset inside the rows or a work-group's columns needs more than 31 bits, in one form:
// a view of rows 2 GiB apart, or K of many millions.  Nobody's step has such a product, so its time was not looked at.
template <typename T>
static void launch_skinny_far(hipStream_t s, const T* a, int64_t lda, const T* w, int M, int N, int K, const Epilogue& epi, int splits,
                              int columns, int packed, int a_rows) {
  dim3 grid((N + columns - 1) / columns, splits);
  const NormOperand none = {};
  const SkinnyOperands o = skinny_operands<T>(a, lda, w, M, N, K, splits, columns, packed, a_rows, true);
#define LAUNCH_FAR(KIND) \
  hipLaunchKernelGGL((gemm_skinny_kernel<T, 4, 2, 2, 8, 0, KIND, 1, 1, 1>), grid, dim3(skinny_threads(8, KIND, 4, 2, 2)), 0, s, o, epi, none)
  if (epi.mode == EPI_TURN) LAUNCH_FAR(EPILOGUE_TURN);
  else if (epi.mode == EPI_QKV) LAUNCH_FAR(EPILOGUE_QKV);
  else if (epi.mode == EPI_F32_ACT) LAUNCH_FAR(EPILOGUE_TWO);
  else LAUNCH_FAR(EPILOGUE_COMMON);
#undef LAUNCH_FAR
}

// The product of the normalised rows of a float32 residual stream (see NormOperand): bfloat16
// weights, up to 16 rows, K up to 2048 and a multiple of 8.
static int launch_skinny_norm(hipStream_t s, const NormOperand& norm, const bf16_t* w, int M, int N, int K,
                              const Epilogue& epi, int splits, int columns, int packed) {
  dim3 grid((N + columns - 1) / columns, splits);
  size_t lds = (size_t)16 * (K * 2 + 16);
  const SkinnyOperands o = skinny_operands<bf16_t>(nullptr, K, w, M, N, K, splits, columns, packed, 0);
#define LAUNCH_NORM(NT, QPL, WP)                                                                               \
  do {                                                                                                         \
    if (epi.mode == EPI_F32_ACT) LAUNCH_NORM_FORM(NT, QPL, EPILOGUE_TWO, WP);    \
    else if (epi.mode == EPI_TURN) LAUNCH_NORM_FORM(NT, QPL, EPILOGUE_TURN, WP);    \
    else if (epi.mode == EPI_QKV) LAUNCH_NORM_FORM(NT, QPL, EPILOGUE_QKV, WP);    \
    else LAUNCH_NORM_FORM(NT, QPL, EPILOGUE_COMMON, WP);    \
  } while (0)
#define LAUNCH_NORM_FORM(NT, QPL, KIND, WP)                                                                        \
  do {                                                                                                         \
    auto kernel = gemm_skinny_kernel<bf16_t, 1, NT, 8, 8, QPL, KIND, 1, WP>;                                                       \
    static size_t granted = 0;    /* statically allocated LDS comes on top: ask for room beyond the default */ \
    if (lds > granted) {                                                                                       \
      hipError_t err = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); \
      if (err != hipSuccess) BT_REFUSE("gemm_skinny: cannot get %zu bytes of LDS: %s", lds, hipGetErrorString(err));   \
      granted = lds;                                                                                           \
    }                                                                                                          \
    hipLaunchKernelGGL(kernel, grid, dim3(skinny_threads(8, KIND, 1, NT, 8)), lds, s, o, epi, norm);                                     \
  } while (0)
  if (K <= 1024) {
    if (columns == 8) LAUNCH_NORM(1, 4, 2); else if (columns <= 16) LAUNCH_NORM(1, 4, 1); else LAUNCH_NORM(2, 4, 1);
  } else {
    if (columns == 8) LAUNCH_NORM(1, 8, 2); else if (columns <= 16) LAUNCH_NORM(1, 8, 1); else LAUNCH_NORM(2, 8, 1);
  }
#undef LAUNCH_NORM
#undef LAUNCH_NORM_FORM
  return BT_OK;
}

// norm: null, or the activations are the normalised rows it describes (then A and lda are ignored)
// a_rows: 0, or A is chunk-major with that many rows (activation_offset in common.h; lda is not used).
// packed_columns: 0, or W is the packed form of the matrix for that many columns per work-group (see
// the kernel), which then is the number of columns a work-group takes.
BT_EXPORT int bt_gemm_skinny(void* stream, int dtype, const void* A, int64_t lda, const void* W, int M, int N, int K,
                             const Epilogue* epi, int splits, int variant, const NormOperand* norm, int packed_columns,
                             int a_rows) {
  if (M <= 0) return BT_OK;
  if (M > 64) BT_REFUSE("gemm_skinny: %d rows, at most 64", M);
  if (dtype != 0 && dtype != 1) BT_REFUSE("gemm_skinny: element type %d is neither float nor bfloat16", dtype);
  const int elems = dtype == 0 ? 4 : 8;
  if (a_rows != 0 && (norm != nullptr || a_rows < M))
    BT_REFUSE("gemm_skinny: chunk-major activations of %d rows for a product of %d rows%s", a_rows, M,
              norm != nullptr ? " that normalises its rows itself" : "");
  if (norm != nullptr) {
    if (dtype != 1 || M > 16 || K > 2048)
      BT_REFUSE("gemm_skinny: the fused norm takes bfloat16 weights, up to 16 rows and K up to 2048 (got %d rows, K %d)", M, K);
    if (!norm->x || !norm->gamma || norm->ldx < K || norm->ldx % 4 != 0 || ((uintptr_t)norm->x & 15) ||
        ((uintptr_t)norm->gamma & 15) || ((uintptr_t)norm->beta & 15) || (norm->kind != 0 && norm->kind != 1))
      BT_REFUSE("gemm_skinny: the rows to normalise, their scale and shift must be 16-byte aligned float32");
    A = W;            // (only its alignment is looked at below)
    lda = K;
  }
  if (epi->mode == EPI_TURN && a_rows != 0) BT_REFUSE("gemm_skinny: turned columns go with row-major activations");
  if (a_rows != 0) lda = K;          // (chunk-major rows have no pitch; K itself is checked)
  int rc = check_operands("gemm_skinny", elems, A, lda, W, M, N, K, *epi, splits);
  if (rc) return rc;
  // 8 to 32 columns per work-group in steps of four (one or two column blocks of the kernel),
  // whichever leaves the busiest compute unit the least to pull: work-groups land on the units in
  // whole rounds.  Variants 8, 12, ... 32 (measurements and tests) force that many.
  static int compute_units = 0;
  if (compute_units == 0) {
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess ||
        hipDeviceGetAttribute(&compute_units, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess)
      compute_units = 256;
  }
  // columns per work-group: the cost of a work-group is what it pulls for one chunk of K (its
  // columns of the weights and the step's rows of the activations) times its chunks, plus a fixed part
  int columns = M <= 16 ? 16 : 32;
  const int packed = packed_columns != 0;
  if (packed) {
    if (packed_columns < 8 || packed_columns > 32 || packed_columns % 4 != 0)
      BT_REFUSE("gemm_skinny: a matrix packed for %d columns per work-group (8, 12, ... 32 are possible)", packed_columns);
    columns = packed_columns;
  } else if (variant >= 8 && variant <= 32 && variant % 4 == 0) {
    columns = variant;
  } else if (variant == 0) {
    const int chunk = 4 * elems;
    const int64_t per = ((K + chunk - 1) / chunk + splits - 1) / splits;
    int64_t best = -1;
    for (int c = 32; c >= 8; c -= 4) {
      int64_t groups = (int64_t)((N + c - 1) / c) * splits;
      int64_t cost = ((groups + compute_units - 1) / compute_units) * (per * (c + M) + 160);
      if (best < 0 || cost < best) { best = cost; columns = c; }
    }
  }
  // where 32 bits of offset do (rows to normalise are read without)
  const int64_t size = 16 / elems, a_bytes = a_rows != 0 ? (int64_t)a_rows * K * size : norm != nullptr ? 0 : ((int64_t)(M - 1) * lda + K) * size;
  const int64_t w_bytes = (int64_t)columns * (K + 4 * elems) * size;
  const bool far = a_bytes >= (int64_t)1 << 31 || w_bytes >= (int64_t)1 << 31;
  if (norm != nullptr) {
    rc = launch_skinny_norm((hipStream_t)stream, *norm, (const bf16_t*)W, M, N, K, *epi, splits, columns, packed);
    if (rc) return rc;
  } else if (far && dtype == 0) {
    launch_skinny_far<float>((hipStream_t)stream, (const float*)A, lda, (const float*)W, M, N, K, *epi, splits, columns, packed, a_rows);
  } else if (far) {
    launch_skinny_far<bf16_t>((hipStream_t)stream, (const bf16_t*)A, lda, (const bf16_t*)W, M, N, K, *epi, splits, columns, packed, a_rows);
  } else if (dtype == 0) {
    launch_skinny<float>((hipStream_t)stream, (const float*)A, lda, (const float*)W, M, N, K, *epi, splits, columns, packed, a_rows);
  } else {
    launch_skinny<bf16_t>((hipStream_t)stream, (const bf16_t*)A, lda, (const bf16_t*)W, M, N, K, *epi, splits, columns, packed, a_rows);
  }
  return bt_check_launch("gemm_skinny");
}

// The same entry points with their arguments as one structure (calls.h), for launch lists.
BT_EXPORT int bt_gemm_tile_call(void* stream, const GemmCall* c) {
  if (c->has_norm || c->a_rows || c->packed_columns)
    BT_REFUSE("gemm_tile: no rows to normalise, no chunk-major rows and no packed weights");
  return bt_gemm_tile(stream, c->dtype, c->A, c->lda, c->W, c->M, c->N, c->K, &c->epi, c->splits, c->variant);
}
BT_EXPORT int bt_gemm_skinny_call(void* stream, const GemmCall* c) {
  return bt_gemm_skinny(stream, c->dtype, c->A, c->lda, c->W, c->M, c->N, c->K, &c->epi, c->splits, c->variant,
                        c->has_norm ? &c->norm : nullptr, c->packed_columns, c->a_rows);
}
