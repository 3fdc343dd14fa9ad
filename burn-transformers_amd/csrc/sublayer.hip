// Kernels for layers that normalise a sublayer's OUTPUT before it joins the residual stream, and
// for activations that are norms themselves.  All statistics and the residual sum are 32-bit.
//   * output norm: x[t] (+)= mult * N(v), v the sublayer's output (the sum of its partial sums and
//     its bias), N an RMS norm, v / sqrt(mean(v^2) + eps) * gamma, or a layer norm,
//     (v - mean) / sqrt(var + eps) * gamma + beta; and a copy of the new x in the products' type
//   * joined rows: [x | y] side by side in the products' type, the operand of a product that reads two streams
//   * an activation in place, behind products whose kernel has none
//   * PolyNorm: a N(z) + b N(z^2) + c N(z^3) + e, N(v) = v / sqrt(mean(v^2) + eps) over a row
#include "host.h"
#include "epilogue.h"

struct OutputNormCall {
  int cast_dtype;        // element type of `cast`: 0 float32, 1 bfloat16
  int n_delta;           // partial sums of the sublayer's output; 0: the stream's own rows are normalised
  int tokens;
  int width;
  int accumulate;        // 1: x += mult * norm(v); 0: x = mult * norm(v)
  int cast_cols;         // columns of `cast` that are written: the new x, then zeros
  float eps;
  float mult;
  float* x;              // [tokens][width] float32 residual stream
  const float* delta;    // [n_delta][..][ldd]
  int64_t delta_stride;  // elements between two partial sums
  int64_t ldd;           // row pitch of a partial sum
  const float* bias;     // [width] or null: added to v
  const float* gamma;    // [width]
  void* cast;            // [tokens][ld_cast] or null
  int64_t ld_cast;
  int kind;              // 0: layer norm (mean taken off, `beta` added), 1: RMS norm
  const float* beta;     // [width] or null
  // The norm that reads the stream next, in the same pass over the row: next_out[t] = norm'(new x[t])
  // (what the next sublayer multiplies by).  next_out null: none.
  void* next_out;        // [tokens][next_ld] in the type `next_dtype`
  int64_t next_ld;
  int next_dtype;
  int next_kind;
  float next_eps;
  const float* next_gamma;
  const float* next_beta;   // or null
};

// y = N'(v) for one element, given the row's statistics
__device__ __forceinline__ float next_norm(const OutputNormCall& c, float v, float mean, float rstd, int col) {
  const float y = (v - mean) * rstd * c.next_gamma[col];
  return c.next_beta ? y + c.next_beta[col] : y;
}

template <typename T>
__global__ void __launch_bounds__(256) output_norm_kernel(OutputNormCall c) {
  extern __shared__ float row_buf[];
  __shared__ __attribute__((aligned(16))) float scratch[32];
  const int t = blockIdx.x;
  float* xr = c.x + (int64_t)t * c.width;
  float partial = 0.f;
  for (int col = threadIdx.x; col < c.width; col += blockDim.x) {
    float v;
    if (c.n_delta == 0) {
      v = xr[col];
    } else {
      v = c.bias ? c.bias[col] : 0.f;
      for (int s = 0; s < c.n_delta; ++s) v += c.delta[s * c.delta_stride + (int64_t)t * c.ldd + col];
    }
    row_buf[col] = v;
    partial += v;
  }
  const float mean = c.kind == 0 ? block_sum<256>(partial, scratch) / (float)c.width : 0.f;
  partial = 0.f;
  for (int col = threadIdx.x; col < c.width; col += blockDim.x) {
    const float d = row_buf[col] - mean;
    partial += d * d;
  }
  const float total = block_sum<256>(partial, scratch);
  const float scale = c.mult / sqrtf(total / (float)c.width + c.eps);
  T* cast = static_cast<T*>(c.cast);
  for (int col = threadIdx.x; col < c.width; col += blockDim.x) {
    float y = (row_buf[col] - mean) * scale * c.gamma[col];
    if (c.beta) y += c.mult * c.beta[col];
    if (c.accumulate) y += xr[col];
    xr[col] = y;
    row_buf[col] = y;         // (a thread's own columns: read back below by the same thread)
    if (cast) cast[(int64_t)t * c.ld_cast + col] = from_float<T>(y);
  }
  if (cast)
    for (int col = c.width + threadIdx.x; col < c.cast_cols; col += blockDim.x)
      cast[(int64_t)t * c.ld_cast + col] = from_float<T>(0.f);
  if (c.next_out) {
    float sum = 0.f;
    if (c.next_kind == 0)
      for (int col = threadIdx.x; col < c.width; col += blockDim.x) sum += row_buf[col];
    const float next_mean = c.next_kind == 0 ? block_sum<256>(sum, scratch) / (float)c.width : 0.f;
    sum = 0.f;
    for (int col = threadIdx.x; col < c.width; col += blockDim.x) sum += (row_buf[col] - next_mean) * (row_buf[col] - next_mean);
    const float next_rstd = 1.0f / sqrtf(block_sum<256>(sum, scratch) / (float)c.width + c.next_eps);
    for (int col = threadIdx.x; col < c.width; col += blockDim.x) {
      const float y = next_norm(c, row_buf[col], next_mean, next_rstd, col);
      if (c.next_dtype == 0) static_cast<float*>(c.next_out)[(int64_t)t * c.next_ld + col] = y;
      else static_cast<bf16_t*>(c.next_out)[(int64_t)t * c.next_ld + col] = (bf16_t)y;
    }
  }
}

// The same for rows of up to 256 * KMAX columns: a thread's columns live in registers and every load
// of a thread (partial sums, bias, the stream, the scale) is issued before the first is used, so a
// row costs one round trip to memory.  A decode step has few rows: one row's latency is its time.
// A thread's columns are KMAX / 4 quads of neighbours, a load for each (QUADS), or lie 256 apart where the rows are no whole
// quads.  What bounds it is the chain of a row: its loads, two sums over the work-group, its stores.  With two partial sums and
// the next norm, one column a load / quads (us, in a HIP graph): 8 rows of 2,048 4.44 / 3.75, of 1,024 3.54 / 3.18; 773 of 2,048
// 7.86 / 7.35; 1,809 of 1,024 with four partial sums 9.28 / 8.89.  Since then shorter sums over a wave (8 rows of 2,048 3.42) and only what is
// there read, the call's fields asked for together (3.24).
template <int KMAX, bool QUADS>
struct RowColumns {
  __device__ __forceinline__ static int column(int k) {
    return QUADS ? 4 * ((int)threadIdx.x + 256 * (k >> 2)) + (k & 3) : (int)threadIdx.x + 256 * k;
  }
  __device__ __forceinline__ static void load(const float* row, int width, float (&v)[KMAX]) {    // (columns beyond the row: a valid place)
    if constexpr (QUADS) {
#pragma unroll
      for (int k = 0; k < KMAX; k += 4) {
        const floatx4 q = *reinterpret_cast<const floatx4*>(row + (column(k) < width ? column(k) : 0));
#pragma unroll
        for (int i = 0; i < 4; ++i) v[k + i] = q[i];
      }
    } else {
#pragma unroll
      for (int k = 0; k < KMAX; ++k) v[k] = row[column(k) < width ? column(k) : 0];
    }
  }
  template <typename O>
  __device__ __forceinline__ static void store(O* row, int width, const float (&v)[KMAX]) {
    if constexpr (QUADS) {
      typedef __attribute__((__vector_size__(4 * sizeof(O)))) O O4;
#pragma unroll
      for (int k = 0; k < KMAX; k += 4)
        if (column(k) < width)
          *reinterpret_cast<O4*>(row + column(k)) = O4{from_float<O>(v[k]), from_float<O>(v[k + 1]), from_float<O>(v[k + 2]), from_float<O>(v[k + 3])};
    } else {
#pragma unroll
      for (int k = 0; k < KMAX; ++k)
        if (column(k) < width) row[column(k)] = from_float<O>(v[k]);
    }
  }
  // The thread's columns that lie 256 apart, of values that are zero beyond the row: what a sum over the row adds up, so that it
  // is the same number whichever way the row was read.  `row`: LDS for 256 * KMAX values; a barrier stands between its users.
  // (8 rows of 2,048, columns 256 apart read one by one / quads through LDS / quads added up as they lie: 4.44 / 3.75 / 3.73 us.)
  __device__ __forceinline__ static void apart(const float (&v)[KMAX], float* row, float (&w)[KMAX]) {
    if constexpr (QUADS) {
#pragma unroll
      for (int k = 0; k < KMAX; k += 4) *reinterpret_cast<floatx4*>(row + column(k)) = floatx4{v[k], v[k + 1], v[k + 2], v[k + 3]};
      __syncthreads();
#pragma unroll
      for (int k = 0; k < KMAX; ++k) w[k] = row[threadIdx.x + 256 * k];
    } else {
#pragma unroll
      for (int k = 0; k < KMAX; ++k) w[k] = v[k];
    }
  }
  // block_sum of what `apart` left (whose barrier stands in place of the one before the sum's own)
  __device__ __forceinline__ static float sum(float partial, float* scratch) {
    if constexpr (!QUADS) return block_sum<256>(partial, scratch);
    partial = wave_sum(partial);
    if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = partial;
    __syncthreads();
    float total = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) total += scratch[i];
    return total;
  }
};

template <typename T, int KMAX, bool QUADS>
__global__ void __launch_bounds__(256) output_norm_small_kernel(OutputNormCall c) {
  typedef RowColumns<KMAX, QUADS> Columns;
  __shared__ __attribute__((aligned(16))) float scratch[32];
  __shared__ __attribute__((aligned(16))) float row_buf[QUADS ? 256 * KMAX : 4];
  const int t = blockIdx.x;
  float* xr = c.x + (int64_t)t * c.width;
  // Every load of a thread is issued before the first is used and none waits for another (columns beyond the row are read from a
  // valid place and dropped).  What is not there is not read: a wave's load of sixteen bytes a lane takes a compute unit 16
  // cycles whatever it brings.  Those behind a branch (the same for every thread) stand first, the sum's own then, and last, in any case, what is
  // used behind the sum: so the wait for the sum's operands counts what is behind them and lets it come meanwhile.
  float v[KMAX], xv[KMAX], g[KMAX], b[KMAX], g2[KMAX], b2[KMAX], part[4][KMAX];
  bool in_row[KMAX];
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    in_row[k] = Columns::column(k) < c.width;
    v[k] = b[k] = b2[k] = g2[k] = part[2][k] = part[3][k] = 0.f;
  }
  // (the call's fields together at the start: the ones a branch asks for would be waited for in it)
  asm volatile("" ::"s"(c.bias), "s"(c.beta), "s"(c.gamma), "s"(c.cast), "s"(c.next_out), "s"(c.next_gamma), "s"(c.next_beta), "s"(c.delta),
               "s"(c.delta_stride), "s"(c.ldd), "s"(c.kind), "s"(c.next_kind));
  const float* row = c.n_delta ? c.delta + (int64_t)t * c.ldd : xr;
  if (c.beta) Columns::load(c.beta, c.width, b);
  if (c.next_out) {
    Columns::load(c.next_gamma, c.width, g2);
    if (c.next_beta) Columns::load(c.next_beta, c.width, b2);
  }
  if (c.n_delta && c.bias) Columns::load(c.bias, c.width, v);
  if (c.n_delta > 2) {
    Columns::load(row + 2 * c.delta_stride, c.width, part[2]);
    Columns::load(row + (c.n_delta > 3 ? 3 : 2) * c.delta_stride, c.width, part[3]);
  }
  Columns::load(row, c.width, part[0]);
  Columns::load(row + (c.n_delta > 1 ? c.delta_stride : 0), c.width, part[1]);
  Columns::load(xr, c.width, xv);
  Columns::load(c.gamma, c.width, g);
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    b[k] = c.beta ? c.mult * b[k] : 0.f;
    v[k] += part[0][k];
    v[k] += c.n_delta > 1 ? part[1][k] : 0.f;
    v[k] += part[2][k];
    v[k] += c.n_delta > 3 ? part[3][k] : 0.f;
  }
  for (int s0 = 4; s0 < c.n_delta; s0 += 4) {              // four partial sums at a time, all their loads together
#pragma unroll
    for (int u = 0; u < 4; ++u) Columns::load(row + (s0 + u < c.n_delta ? s0 + u : c.n_delta - 1) * c.delta_stride, c.width, part[u]);
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int k = 0; k < KMAX; ++k) v[k] += s0 + u < c.n_delta ? part[u][k] : 0.f;
  }
  if (!c.accumulate)
#pragma unroll
    for (int k = 0; k < KMAX; ++k) xv[k] = 0.f;
#pragma unroll
  for (int k = 0; k < KMAX; ++k) v[k] = in_row[k] ? v[k] : 0.f;
  float w[KMAX], partial = 0.f;
  Columns::apart(v, row_buf, w);
  if (c.kind == 0) {          // a layer norm: the mean first, then the squared distances from it
#pragma unroll
    for (int k = 0; k < KMAX; ++k) partial += w[k];
    const float mean = Columns::sum(partial, scratch) / (float)c.width;
#pragma unroll
    for (int k = 0; k < KMAX; ++k) {
      v[k] = in_row[k] ? v[k] - mean : 0.f;
      w[k] = (int)threadIdx.x + 256 * k < c.width ? w[k] - mean : 0.f;
    }
    partial = 0.f;
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < KMAX; ++k) partial += w[k] * w[k];
  const float scale = c.mult / sqrtf(Columns::sum(partial, scratch) / (float)c.width + c.eps);
#pragma unroll
  for (int k = 0; k < KMAX; ++k) v[k] = in_row[k] ? v[k] * scale * g[k] + b[k] + xv[k] : 0.f;
  Columns::store(xr, c.width, v);
  if (T* cast = static_cast<T*>(c.cast)) {
    cast += (int64_t)t * c.ld_cast;
    Columns::store(cast, c.width, v);
    for (int col = c.width + threadIdx.x; col < c.cast_cols; col += blockDim.x) cast[col] = from_float<T>(0.f);
  }
  if (c.next_out) {           // the norm that reads the new row next, from the registers that hold it
    float next_mean = 0.f;
    Columns::apart(v, row_buf, w);
    if (c.next_kind == 0) {
      float sum = 0.f;
#pragma unroll
      for (int k = 0; k < KMAX; ++k) sum += w[k];
      next_mean = Columns::sum(sum, scratch) / (float)c.width;
      __syncthreads();
    }
    float squares = 0.f;
#pragma unroll
    for (int k = 0; k < KMAX; ++k) {
      const float d = (int)threadIdx.x + 256 * k < c.width ? w[k] - next_mean : 0.f;
      squares += d * d;
    }
    const float next_rstd = 1.0f / sqrtf(Columns::sum(squares, scratch) / (float)c.width + c.next_eps);
#pragma unroll
    for (int k = 0; k < KMAX; ++k) v[k] = (v[k] - next_mean) * next_rstd * g2[k] + (c.next_beta ? b2[k] : 0.f);
    if (c.next_dtype == 0) Columns::store(static_cast<float*>(c.next_out) + (int64_t)t * c.next_ld, c.width, v);
    else Columns::store(static_cast<bf16_t*>(c.next_out) + (int64_t)t * c.next_ld, c.width, v);
  }
}

template <typename T>
static void launch_output_norm(hipStream_t stream, const OutputNormCall& c) {
  dim3 grid(c.tokens), block(256);
  const uintptr_t floats = (uintptr_t)c.x | (uintptr_t)c.delta | (uintptr_t)c.bias | (uintptr_t)c.gamma | (uintptr_t)c.beta | (uintptr_t)c.next_gamma |
                           (uintptr_t)c.next_beta;
  const bool quads = c.width % 4 == 0 && (floats & 15) == 0 && c.ldd % 4 == 0 && c.delta_stride % 4 == 0 &&
                     (!c.cast || (c.ld_cast % 4 == 0 && ((uintptr_t)c.cast & (4 * sizeof(T) - 1)) == 0)) &&
                     (!c.next_out || (c.next_ld % 4 == 0 && ((uintptr_t)c.next_out & (c.next_dtype == 0 ? 15 : 7)) == 0));
  if (c.width <= 1024 && quads)
    hipLaunchKernelGGL((output_norm_small_kernel<T, 4, true>), grid, block, 0, stream, c);
  else if (c.width <= 1024)
    hipLaunchKernelGGL((output_norm_small_kernel<T, 4, false>), grid, block, 0, stream, c);
  else if (c.width <= 2048 && quads)
    hipLaunchKernelGGL((output_norm_small_kernel<T, 8, true>), grid, block, 0, stream, c);
  else if (c.width <= 2048)
    hipLaunchKernelGGL((output_norm_small_kernel<T, 8, false>), grid, block, 0, stream, c);
  else
    hipLaunchKernelGGL(output_norm_kernel<T>, grid, block, (size_t)c.width * sizeof(float), stream, c);
}

BT_EXPORT int bt_output_norm_call(void* stream, const OutputNormCall* c) {
  if (c->tokens <= 0) return BT_OK;
  if (c->width <= 0 || c->width > 15360) BT_REFUSE("output_norm: width %d outside 1..15360", c->width);
  if (!c->x || !c->gamma || (c->n_delta > 0 && !c->delta)) BT_REFUSE("output_norm: missing operand");
  if (c->n_delta == 0 && c->accumulate) BT_REFUSE("output_norm: the stream's own rows cannot be added to themselves");
  if (c->kind != 0 && c->kind != 1) BT_REFUSE("output_norm: unknown kind of norm %d", c->kind);
  if (c->next_out && (!c->next_gamma || c->next_ld < c->width || (c->next_kind != 0 && c->next_kind != 1)))
    BT_REFUSE("output_norm: the norm that follows lacks its scale, its kind or room for its rows");
  if (c->cast && (c->cast_cols < c->width || c->ld_cast < c->cast_cols))
    BT_REFUSE("output_norm: a copy of %d columns in rows of %lld does not hold width %d", c->cast_cols,
              (long long)c->ld_cast, c->width);
  if (c->cast_dtype == 0)
    launch_output_norm<float>((hipStream_t)stream, *c);
  else
    launch_output_norm<bf16_t>((hipStream_t)stream, *c);
  return bt_check_launch("output_norm");
}

// out[t] = [x[t] | y[t] | zeros] in the products' type: the operand of a product over two float32
// streams laid side by side (W [x; y] as one product).
struct JoinRowsCall {
  int out_dtype;         // 0 float32, 1 bfloat16
  int tokens;
  int width;             // columns of x and of y
  int out_cols;          // columns of out written: 2 * width, then zeros
  const float* x;        // [tokens][width]
  const float* y;        // [tokens][width]
  void* out;             // [tokens][ldo]
  int64_t ldo;
};

template <typename T>
__global__ void __launch_bounds__(256) join_rows_kernel(JoinRowsCall c) {
  const int t = blockIdx.x;
  T* out = static_cast<T*>(c.out) + (int64_t)t * c.ldo;
  for (int col = threadIdx.x; col < c.out_cols; col += blockDim.x) {
    float v = 0.f;
    if (col < c.width) v = c.x[(int64_t)t * c.width + col];
    else if (col < 2 * c.width) v = c.y[(int64_t)t * c.width + col - c.width];
    out[col] = from_float<T>(v);
  }
}

BT_EXPORT int bt_join_rows_call(void* stream, const JoinRowsCall* c) {
  if (c->tokens <= 0) return BT_OK;
  if (c->width <= 0 || c->out_cols < 2 * c->width || c->ldo < c->out_cols)
    BT_REFUSE("join_rows: rows of %lld columns (%d written) do not hold two of width %d", (long long)c->ldo, c->out_cols, c->width);
  if (!c->x || !c->y || !c->out) BT_REFUSE("join_rows: missing operand");
  if (c->out_dtype == 0)
    hipLaunchKernelGGL(join_rows_kernel<float>, dim3(c->tokens), dim3(256), 0, (hipStream_t)stream, *c);
  else
    hipLaunchKernelGGL(join_rows_kernel<bf16_t>, dim3(c->tokens), dim3(256), 0, (hipStream_t)stream, *c);
  return bt_check_launch("join_rows");
}

struct PolyNormCall {
  int out_dtype;          // 0 float32, 1 bfloat16
  int tokens;
  int columns;            // the row's length: statistics are means over these
  int out_cols;           // columns of `out` that are written: the result, then zeros
  float eps;
  const float* z;         // [tokens][ldz] float32
  int64_t ldz;
  const float* coefficients;  // a, b, c, e
  void* out;              // [tokens][ldo]
  int64_t ldo;
};

// Three sums over a work-group of 256 threads with one meeting of the waves; `scratch` holds 12 floats of LDS, on 16 bytes.
__device__ __forceinline__ void block_sum3(float& a, float& b, float& d, float* scratch) {
  a = wave_sum(a);
  b = wave_sum(b);
  d = wave_sum(d);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane == 0) {
    scratch[wave * 3] = a;
    scratch[wave * 3 + 1] = b;
    scratch[wave * 3 + 2] = d;
  }
  __syncthreads();
  floatx4 part[3];
#pragma unroll
  for (int q = 0; q < 3; ++q) part[q] = reinterpret_cast<const floatx4*>(scratch)[q];
  a = b = d = 0.f;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    a += part[(w * 3) >> 2][(w * 3) & 3];
    b += part[(w * 3 + 1) >> 2][(w * 3 + 1) & 3];
    d += part[(w * 3 + 2) >> 2][(w * 3 + 2) & 3];
  }
}

// What a value adds to the three sums, and its result: written out, so that every kernel rounds alike.
__device__ __forceinline__ void poly_add(float v, float& s2, float& s4, float& s6) {
  const float v2 = v * v;
  s2 = fmaf(v, v, s2);
  s4 = fmaf(v2, v2, s4);
  s6 = fmaf(v2 * v2, v2, s6);
}
__device__ __forceinline__ float poly_value(float v, float a, float b, float d, float e) {
  const float v2 = v * v;
  return fmaf(a, v, fmaf(b, v2, fmaf(d, v2 * v, e)));
}

template <typename T>
__global__ void __launch_bounds__(256) poly_norm_kernel(PolyNormCall c) {
  extern __shared__ float row_buf[];
  __shared__ __attribute__((aligned(16))) float scratch[12];
  const int t = blockIdx.x;
  const float* zr = c.z + (int64_t)t * c.ldz;
  float s2 = 0.f, s4 = 0.f, s6 = 0.f;
  for (int col = threadIdx.x; col < c.columns; col += blockDim.x) {
    const float v = zr[col];
    row_buf[col] = v;
    poly_add(v, s2, s4, s6);
  }
  block_sum3(s2, s4, s6, scratch);
  const float n = (float)c.columns;
  const float a = c.coefficients[0] / sqrtf(s2 / n + c.eps);
  const float b = c.coefficients[1] / sqrtf(s4 / n + c.eps);
  const float d = c.coefficients[2] / sqrtf(s6 / n + c.eps);
  const float e = c.coefficients[3];
  T* out = static_cast<T*>(c.out) + (int64_t)t * c.ldo;
  for (int col = threadIdx.x; col < c.columns; col += blockDim.x) {
    out[col] = from_float<T>(poly_value(row_buf[col], a, b, d, e));
  }
  for (int col = c.columns + threadIdx.x; col < c.out_cols; col += blockDim.x) out[col] = from_float<T>(0.f);
}

// The same for rows of up to 256 * KMAX columns in whole quads: a thread's columns live in registers, all its loads of 16 bytes are on
// their way together, and the sums take the columns in the order above (RowColumns::apart).  What bounds it is memory: 2,048 rows of 4,096 are
// 50 MB, 10 us at the copy's rate.  Measured (us, a column a load / quads): 2,048 rows of 4,096
// 13.7 / 9.8, 1,024 of 8,192 16.2 / 9.9, 8 of 4,096 5.4 / 3.0, 2,048 of 1,024 6.1 / 5.5.
template <typename T, int KMAX>
__global__ void __launch_bounds__(256) poly_norm_quads_kernel(PolyNormCall c) {
  typedef RowColumns<KMAX, true> Columns;
  __shared__ __attribute__((aligned(16))) float row_buf[256 * KMAX];
  __shared__ __attribute__((aligned(16))) float scratch[12];
  const int t = blockIdx.x;
  float v[KMAX], w[KMAX];
  Columns::load(c.z + (int64_t)t * c.ldz, c.columns, v);
  const float p0 = c.coefficients[0], p1 = c.coefficients[1], p2 = c.coefficients[2], e = c.coefficients[3];
  Columns::apart(v, row_buf, w);
  float s2 = 0.f, s4 = 0.f, s6 = 0.f;
#pragma unroll
  for (int k = 0; k < KMAX; ++k) poly_add((int)threadIdx.x + 256 * k < c.columns ? w[k] : 0.f, s2, s4, s6);
  block_sum3(s2, s4, s6, scratch);
  const float n = (float)c.columns;
  const float a = p0 / sqrtf(s2 / n + c.eps), b = p1 / sqrtf(s4 / n + c.eps), d = p2 / sqrtf(s6 / n + c.eps);
#pragma unroll
  for (int k = 0; k < KMAX; ++k) v[k] = poly_value(v[k], a, b, d, e);
  T* out = static_cast<T*>(c.out) + (int64_t)t * c.ldo;
  Columns::store(out, c.columns, v);
  for (int col = c.columns + threadIdx.x; col < c.out_cols; col += blockDim.x) out[col] = from_float<T>(0.f);
}

template <typename T>
static void launch_poly_norm(hipStream_t stream, const PolyNormCall& c) {
  dim3 grid(c.tokens), block(256);
  const bool quads = c.columns % 4 == 0 && c.ldz % 4 == 0 && c.ldo % 4 == 0 && ((uintptr_t)c.z & 15) == 0 && ((uintptr_t)c.out & (4 * sizeof(T) - 1)) == 0;
  if (quads && c.columns <= 1024)
    hipLaunchKernelGGL((poly_norm_quads_kernel<T, 4>), grid, block, 0, stream, c);
  else if (quads && c.columns <= 4096)
    hipLaunchKernelGGL((poly_norm_quads_kernel<T, 16>), grid, block, 0, stream, c);
  else if (quads && c.columns <= 8192)
    hipLaunchKernelGGL((poly_norm_quads_kernel<T, 32>), grid, block, 0, stream, c);
  else
    hipLaunchKernelGGL(poly_norm_kernel<T>, grid, block, (size_t)c.columns * sizeof(float), stream, c);
}

BT_EXPORT int bt_poly_norm_call(void* stream, const PolyNormCall* c) {
  if (c->tokens <= 0) return BT_OK;
  if (c->columns <= 0 || c->columns > 15360) BT_REFUSE("poly_norm: %d columns outside 1..15360", c->columns);
  if (!c->z || !c->coefficients || !c->out) BT_REFUSE("poly_norm: missing operand");
  if (c->out_cols < c->columns || c->ldo < c->out_cols || c->ldz < c->columns)
    BT_REFUSE("poly_norm: rows of %lld and %lld elements do not hold %d (%d) columns", (long long)c->ldz,
              (long long)c->ldo, c->columns, c->out_cols);
  if (c->out_dtype == 0)
    launch_poly_norm<float>((hipStream_t)stream, *c);
  else
    launch_poly_norm<bf16_t>((hipStream_t)stream, *c);
  return bt_check_launch("poly_norm");
}

// RMS norm in equal consecutive parts of a row ("groups"), each over its own root mean square, the whole
// times `gamma`; of a sublayer's output on its way into the stream, or of rows of the stream itself.
//   output (n_delta > 0):  v = scale * (sum of delta + bias) + scale2 * (sum of delta2 + bias2), the second
//       term for layers whose sublayer is two parts side by side; v *= sigmoid(gate) where a gate's
//       logits come with it; x[t] (+)= mult * N(v), and `cast` receives the new x in the products' type.
//   rows (n_delta == 0):   cast[r] = N(x[rows[r]]) (every row in order without `rows`); x stays as it is.
struct GroupNormCall {
  int cast_dtype;         // element type of `cast`: 0 float32, 1 bfloat16
  int tokens;             // rows of this call
  int width;
  int groups;             // equal parts of a row, each with statistics of its own
  int n_delta, n_delta2;
  int accumulate;         // output: 1: x += mult * N(v); 0: x = mult * N(v)
  int cast_cols;          // columns of `cast` that are written: the result, then zeros
  float eps, mult;
  float scale, scale2;    // factors of the two terms
  float* x;               // [..][width] float32 residual stream
  const float* delta;     // [n_delta][..][ldd]
  int64_t delta_stride, ldd;
  const float* bias;      // [width] or null
  const float* delta2;    // [n_delta2][..][ldd2], or null
  int64_t delta2_stride, ldd2;
  const float* bias2;     // [width] or null
  const float* gate;      // [tokens][ld_gate] logits, or null
  int64_t ld_gate;
  const float* gamma;     // [width]
  void* cast;             // [tokens][ld_cast], or null
  int64_t ld_cast;
  const int* rows;        // rows mode: which rows of x, or null
};

template <typename T>
__global__ void __launch_bounds__(256) group_norm_kernel(GroupNormCall c) {
  extern __shared__ float row_buf[];          // [width], then [groups] reciprocal roots
  float* rstd = row_buf + c.width;
  const int t = blockIdx.x;
  const bool from_stream = c.n_delta == 0;
  const int source = from_stream && c.rows ? c.rows[t] : t;
  float* xr = c.x + (int64_t)source * c.width;
  for (int col = threadIdx.x; col < c.width; col += blockDim.x) {
    float v;
    if (from_stream) {
      v = xr[col];
    } else {
      v = c.bias ? c.bias[col] : 0.f;
      for (int s = 0; s < c.n_delta; ++s) v += c.delta[s * c.delta_stride + (int64_t)t * c.ldd + col];
      v *= c.scale;
      if (c.n_delta2 > 0) {
        float w = c.bias2 ? c.bias2[col] : 0.f;
        for (int s = 0; s < c.n_delta2; ++s) w += c.delta2[s * c.delta2_stride + (int64_t)t * c.ldd2 + col];
        v = fmaf(c.scale2, w, v);
      }
      if (c.gate) v *= 1.0f / (1.0f + expf(-c.gate[(int64_t)t * c.ld_gate + col]));
    }
    row_buf[col] = v;
  }
  __syncthreads();
  // a wave takes whole parts, so no sum crosses waves
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const int per = c.width / c.groups;
  for (int g = wave; g < c.groups; g += waves) {
    float squares = 0.f;
    for (int i = lane; i < per; i += 64) squares = fmaf(row_buf[g * per + i], row_buf[g * per + i], squares);
    squares = wave_sum(squares);
    if (lane == 0) rstd[g] = 1.0f / sqrtf(squares / (float)per + c.eps);
  }
  __syncthreads();
  T* cast = static_cast<T*>(c.cast);
  for (int col = threadIdx.x; col < c.width; col += blockDim.x) {
    float y = row_buf[col] * rstd[col / per] * c.gamma[col];
    if (!from_stream) {
      y *= c.mult;
      if (c.accumulate) y += xr[col];
      xr[col] = y;
    }
    if (cast) cast[(int64_t)t * c.ld_cast + col] = from_float<T>(y);
  }
  if (cast)
    for (int col = c.width + threadIdx.x; col < c.cast_cols; col += blockDim.x)
      cast[(int64_t)t * c.ld_cast + col] = from_float<T>(0.f);
}

// The same for rows of up to 256 * KMAX columns: a thread's columns live in registers (RowColumns), every load of a thread (partial
// sums of both terms, biases, the gate, the stream, the scale) is issued before the first is used, and what is not there is not read, so
// a row costs one round trip to memory (a decode step has few rows: one row's latency is its time).  The parts' sums of squares meet in
// LDS, a wave a part, in one order however the row was read.  What bounds it with many rows is memory: a row's 14 bytes a column take
// 6 us of 2,048 rows of 1,024 at the copy's rate.  Measured (us, 2 parts, one partial sum; a column a load and absent operands' places read too / quads):
// 2,048 rows of 1,024 8.3 / 6.5, of 2,048 13.9 / 11.2; 512 of 1,024 4.5 / 3.7; 8 of 2,048 with two 4.9 / 3.8, one of 1,024 3.5 / 2.9.
template <typename T, int KMAX, bool QUADS, int READS>
__global__ void __launch_bounds__(256) group_norm_small_kernel(GroupNormCall c) {
  typedef RowColumns<KMAX, QUADS> Columns;
  extern __shared__ __attribute__((aligned(16))) float row_buf[];       // [width], then [groups] reciprocal roots
  float* rstd = row_buf + c.width;
  const int t = blockIdx.x;
  const bool from_stream = c.n_delta == 0;
  const int source = from_stream && c.rows ? c.rows[t] : t;
  float* xr = c.x + (int64_t)source * c.width;
  float v[KMAX], w[KMAX], xv[KMAX], g[KMAX], gt[KMAX], part[4][KMAX], part2[4][KMAX];
#pragma unroll
  for (int k = 0; k < KMAX; ++k) v[k] = w[k] = gt[k] = part[0][k] = part[1][k] = part[2][k] = part[3][k] = 0.f;
  // (the call's fields together at the start: the ones a branch asks for would be waited for in it)
  asm volatile("" ::"s"(c.bias), "s"(c.bias2), "s"(c.gate), "s"(c.ld_gate), "s"(c.gamma), "s"(c.cast), "s"(c.delta), "s"(c.delta_stride),
               "s"(c.ldd), "s"(c.n_delta2));
  const float* row = from_stream ? xr : c.delta + (int64_t)t * c.ldd;
  const float* row2 = c.delta2 + (int64_t)t * c.ldd2;
  // one to four of a term's partial sums, from the s0-th on; those that are not there count nothing
  auto ask = [&](const float* first, int64_t stride, int s0, int n, float (&to)[4][KMAX]) {
    Columns::load(first + s0 * stride, c.width, to[0]);
    if (s0 + 1 < n) Columns::load(first + (s0 + 1) * stride, c.width, to[1]);
    if (s0 + 2 < n) Columns::load(first + (s0 + 2) * stride, c.width, to[2]);
    if (s0 + 3 < n) Columns::load(first + (s0 + 3) * stride, c.width, to[3]);
  };
  auto add = [&](float (&sum)[KMAX], const float (&from)[4][KMAX], int s0, int n) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int k = 0; k < KMAX; ++k) sum[k] += s0 + u < n ? from[u][k] : 0.f;
  };
  if (c.gate) Columns::load(c.gate + (int64_t)t * c.ld_gate, c.width, gt);
  if (!from_stream && c.bias) Columns::load(c.bias, c.width, v);
  if (c.n_delta2 > 0) {
    if (c.bias2) Columns::load(c.bias2, c.width, w);
    ask(row2, c.delta2_stride, 0, c.n_delta2, part2);
  }
  if (!from_stream) ask(row, c.delta_stride, 0, c.n_delta, part);
  Columns::load(xr, c.width, xv);
  Columns::load(c.gamma, c.width, g);
  if (from_stream) {
#pragma unroll
    for (int k = 0; k < KMAX; ++k) v[k] = xv[k];
  } else {
    add(v, part, 0, c.n_delta);
    for (int s0 = 4; s0 < c.n_delta; s0 += 4) {
      ask(row, c.delta_stride, s0, c.n_delta, part);
      add(v, part, s0, c.n_delta);
    }
#pragma unroll
    for (int k = 0; k < KMAX; ++k) v[k] *= c.scale;
    if (c.n_delta2 > 0) {
      add(w, part2, 0, c.n_delta2);
      for (int s0 = 4; s0 < c.n_delta2; s0 += 4) {
        ask(row2, c.delta2_stride, s0, c.n_delta2, part2);
        add(w, part2, s0, c.n_delta2);
      }
#pragma unroll
      for (int k = 0; k < KMAX; ++k) v[k] = fmaf(c.scale2, w[k], v[k]);
    }
    if (c.gate) {
#pragma unroll
      for (int k = 0; k < KMAX; ++k) v[k] *= 1.0f / (1.0f + expf(-gt[k]));
    }
  }
  Columns::store(row_buf, c.width, v);
  const int per = c.width / c.groups;
  int mine[KMAX];                             // which part a column (of quads: the quad's columns) lies in
#pragma unroll
  for (int k = 0; k < KMAX; ++k) mine[k] = QUADS && k % 4 ? mine[k & ~3] : Columns::column(k) < c.width ? Columns::column(k) / per : 0;
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  for (int p = wave; p < c.groups; p += waves) {
    const float* from = row_buf + p * per;
    float squares = 0.f;
    for (int i = lane; i < per; i += 64 * READS) {       // (so many reads at a time, added up one after the other)
      float x[READS];
#pragma unroll
      for (int u = 0; u < READS; ++u) x[u] = i + 64 * u < per ? from[i + 64 * u] : 0.f;
#pragma unroll
      for (int u = 0; u < READS; ++u) squares = fmaf(x[u], x[u], squares);
    }
    squares = wave_sum(squares);
    if (lane == 0) rstd[p] = 1.0f / sqrtf(squares / (float)per + c.eps);
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    v[k] = v[k] * rstd[mine[k]] * g[k];
    if (!from_stream) {
      v[k] *= c.mult;
      if (c.accumulate) v[k] += xv[k];
    }
  }
  if (!from_stream) Columns::store(xr, c.width, v);
  if (T* cast = static_cast<T*>(c.cast)) {
    cast += (int64_t)t * c.ld_cast;
    Columns::store(cast, c.width, v);
    for (int col = c.width + threadIdx.x; col < c.cast_cols; col += blockDim.x) cast[col] = from_float<T>(0.f);
  }
}

// The same a column a load, for more rows than units hold at once of the kernel above, which takes 204 registers for 2,048 columns read so and 104 for
// 1,024 (512 and 1,024 rows at once): the places of operands that are not there are read too (those of the scale) and the second
// term's sums come behind the first's, in 88 and 44.  Measured (us, the one above / this one): 512 rows of 2,030 6.2 / 6.8, 700 9.6 / 8.0, 2,048 of 1,030 with
// two terms 18.6 / 13.5; 1,024 of 1,022 5.8 / 6.2, 2,048 of 1,020 9.7 / 8.8.
template <typename T, int KMAX>
__global__ void __launch_bounds__(256) group_norm_lean_kernel(GroupNormCall c) {
  extern __shared__ float row_buf[];          // [width], then [groups] reciprocal roots
  float* rstd = row_buf + c.width;
  const int t = blockIdx.x;
  const bool from_stream = c.n_delta == 0;
  const int source = from_stream && c.rows ? c.rows[t] : t;
  float* xr = c.x + (int64_t)source * c.width;
  float v[KMAX], w[KMAX], xv[KMAX], g[KMAX], gt[KMAX];
  int cc[KMAX];
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    const int col = threadIdx.x + 256 * k;
    cc[k] = col < c.width ? col : 0;
  }
  const float* bias = c.bias ? c.bias : c.gamma;           // (read in any case, used only where there is one)
  const float* bias2 = c.bias2 ? c.bias2 : c.gamma;
  const float* gate = c.gate ? c.gate + (int64_t)t * c.ld_gate : c.gamma;
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    g[k] = c.gamma[cc[k]];
    xv[k] = xr[cc[k]];
    v[k] = bias[cc[k]];
    w[k] = bias2[cc[k]];
    gt[k] = gate[cc[k]];
  }
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    v[k] = c.bias ? v[k] : 0.f;
    w[k] = c.bias2 ? w[k] : 0.f;
  }
  if (from_stream) {
#pragma unroll
    for (int k = 0; k < KMAX; ++k) v[k] = xv[k];
  } else {
    const float* row = c.delta + (int64_t)t * c.ldd;
    for (int s0 = 0; s0 < c.n_delta; s0 += 4) {            // four partial sums at a time, all their loads together
      float part[4][KMAX];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int sc = s0 + u < c.n_delta ? s0 + u : c.n_delta - 1;
#pragma unroll
        for (int k = 0; k < KMAX; ++k) part[u][k] = row[sc * c.delta_stride + cc[k]];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int k = 0; k < KMAX; ++k) v[k] += s0 + u < c.n_delta ? part[u][k] : 0.f;
    }
    const float* row2 = c.delta2 + (int64_t)t * c.ldd2;
    for (int s0 = 0; s0 < c.n_delta2; s0 += 4) {
      float part[4][KMAX];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int sc = s0 + u < c.n_delta2 ? s0 + u : c.n_delta2 - 1;
#pragma unroll
        for (int k = 0; k < KMAX; ++k) part[u][k] = row2[sc * c.delta2_stride + cc[k]];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int k = 0; k < KMAX; ++k) w[k] += s0 + u < c.n_delta2 ? part[u][k] : 0.f;
    }
#pragma unroll
    for (int k = 0; k < KMAX; ++k) {
      v[k] *= c.scale;
      if (c.n_delta2 > 0) v[k] = fmaf(c.scale2, w[k], v[k]);
      if (c.gate) v[k] *= 1.0f / (1.0f + expf(-gt[k]));
    }
  }
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    const int col = threadIdx.x + 256 * k;
    if (col < c.width) row_buf[col] = v[k];
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const int per = c.width / c.groups;
  for (int part = wave; part < c.groups; part += waves) {
    float squares = 0.f;
    for (int i = lane; i < per; i += 64) squares = fmaf(row_buf[part * per + i], row_buf[part * per + i], squares);
    squares = wave_sum(squares);
    if (lane == 0) rstd[part] = 1.0f / sqrtf(squares / (float)per + c.eps);
  }
  __syncthreads();
  T* cast = static_cast<T*>(c.cast);
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    const int col = threadIdx.x + 256 * k;
    if (col < c.width) {
      float y = v[k] * rstd[col / per] * g[k];
      if (!from_stream) {
        y *= c.mult;
        if (c.accumulate) y += xv[k];
        xr[col] = y;
      }
      if (cast) cast[(int64_t)t * c.ld_cast + col] = from_float<T>(y);
    }
  }
  if (cast)
    for (int col = c.width + threadIdx.x; col < c.cast_cols; col += blockDim.x)
      cast[(int64_t)t * c.ld_cast + col] = from_float<T>(0.f);
}

template <typename T>
static void launch_group_norm(hipStream_t stream, const GroupNormCall& c) {
  const size_t lds = (size_t)(c.width + c.groups) * sizeof(float);
  dim3 grid(c.tokens), block(256);
  const uintptr_t floats = (uintptr_t)c.x | (uintptr_t)c.delta | (uintptr_t)c.bias | (uintptr_t)c.delta2 | (uintptr_t)c.bias2 | (uintptr_t)c.gate |
                           (uintptr_t)c.gamma;
  const bool quads = c.width / c.groups % 4 == 0 && (floats & 15) == 0 && c.ldd % 4 == 0 && c.delta_stride % 4 == 0 && c.ldd2 % 4 == 0 &&
                     c.delta2_stride % 4 == 0 && c.ld_gate % 4 == 0 &&
                     (!c.cast || (c.ld_cast % 4 == 0 && ((uintptr_t)c.cast & (4 * sizeof(T) - 1)) == 0));
  // no more reads together than a part has (eight for each of 64 parts of 16 columns took 2,048 rows of 1,024 22.1 us, one 17.1;
  // for 16 parts of 64 9.5 / 8.2, for 8 of 128 7.6, four 7.2)
  const int per = c.width / c.groups;
  auto small = [&](auto columns) {
    constexpr int KMAX = decltype(columns)::value;
    auto launch = [&](auto reads) {
      constexpr int READS = decltype(reads)::value;
      if (quads) hipLaunchKernelGGL((group_norm_small_kernel<T, KMAX, true, READS>), grid, block, lds, stream, c);
      else hipLaunchKernelGGL((group_norm_small_kernel<T, KMAX, false, READS>), grid, block, lds, stream, c);
    };
    if (!quads && c.tokens > 4096 / KMAX) hipLaunchKernelGGL((group_norm_lean_kernel<T, KMAX>), grid, block, lds, stream, c);
    else if (per <= 64) launch(Constant<1>());
    else if (per <= 256) launch(Constant<4>());
    else launch(Constant<8>());
  };
  if (c.width <= 1024)
    small(Constant<4>());
  else if (c.width <= 2048)
    small(Constant<8>());
  else
    hipLaunchKernelGGL(group_norm_kernel<T>, grid, block, lds, stream, c);
}

BT_EXPORT int bt_group_norm_call(void* stream, const GroupNormCall* c) {
  if (c->tokens <= 0) return BT_OK;
  if (c->width <= 0 || c->width > 15360) BT_REFUSE("group_norm: width %d outside 1..15360", c->width);
  if (c->groups <= 0 || c->groups > 512 || c->width % c->groups != 0)
    BT_REFUSE("group_norm: %d parts (1..512) must divide width %d", c->groups, c->width);
  if (!c->x || !c->gamma || (c->n_delta > 0 && !c->delta) || (c->n_delta2 > 0 && !c->delta2))
    BT_REFUSE("group_norm: missing operand");
  if (c->n_delta == 0 && (!c->cast || c->n_delta2 > 0 || c->gate))
    BT_REFUSE("group_norm: rows of the stream are normalised into `cast`, with one term and no gate");
  if (c->n_delta < 0 || c->n_delta2 < 0) BT_REFUSE("group_norm: negative counts of partial sums");
  if (c->cast && (c->cast_cols < c->width || c->ld_cast < c->cast_cols))
    BT_REFUSE("group_norm: a copy of %d columns in rows of %lld does not hold width %d", c->cast_cols,
              (long long)c->ld_cast, c->width);
  if (c->gate && c->ld_gate < c->width) BT_REFUSE("group_norm: the gate's rows are shorter than the width");
  if (c->cast_dtype == 0)
    launch_group_norm<float>((hipStream_t)stream, *c);
  else
    launch_group_norm<bf16_t>((hipStream_t)stream, *c);
  return bt_check_launch("group_norm");
}

// logits <- cap * tanh(logits / cap), in place, over float32 rows.
struct SoftCapCall {
  int rows;
  int columns;
  float cap;
  float* logits;          // [rows][ld]
  int64_t ld;
};

__global__ void __launch_bounds__(256) soft_cap_kernel(SoftCapCall c) {
  float* row = c.logits + (int64_t)blockIdx.x * c.ld;
  const float inverse = 1.0f / c.cap;
  for (int col = blockIdx.y * blockDim.x + threadIdx.x; col < c.columns; col += gridDim.y * blockDim.x)
    row[col] = c.cap * tanhf(row[col] * inverse);
}

BT_EXPORT int bt_soft_cap_call(void* stream, const SoftCapCall* c) {
  if (c->rows <= 0) return BT_OK;
  if (c->columns <= 0 || c->ld < c->columns || !c->logits) BT_REFUSE("soft_cap: missing operand or rows too short");
  if (!(c->cap > 0.f)) BT_REFUSE("soft_cap: the cap %g must be positive", (double)c->cap);
  int per_row = (c->columns + 2047) / 2048;
  if (per_row > 64) per_row = 64;
  hipLaunchKernelGGL(soft_cap_kernel, dim3(c->rows, per_row), dim3(256), 0, (hipStream_t)stream, *c);
  return bt_check_launch("soft_cap");
}

// ---------------------------------------------------------------------------------------------
// An activation in place on a product's stored result: behind products whose kernel (the vendor's library) has no such
// epilogue.  Rows of `columns` values, 16 bytes a thread where pitch and width allow.
// ---------------------------------------------------------------------------------------------
struct ActivateCall {
  int dtype;
  int tokens;
  int columns;
  int act;               // Activation (epilogue.h)
  void* rows;            // [tokens][ld]
  int64_t ld;
};

template <typename T>
__global__ void __launch_bounds__(256) activate_kernel(ActivateCall c) {
  constexpr int V = 16 / (int)sizeof(T);
  T* row = static_cast<T*>(c.rows) + (int64_t)blockIdx.y * c.ld;
  const int col = (blockIdx.x * 256 + threadIdx.x) * V;
  if (col >= c.columns) return;
  T v[V];
  const bool whole = col + V <= c.columns && (((uintptr_t)(row + col)) & 15) == 0;
  if (whole)
    *reinterpret_cast<float4*>(v) = *reinterpret_cast<const float4*>(row + col);
  else
    for (int i = 0; i < V; ++i) v[i] = col + i < c.columns ? row[col + i] : from_float<T>(0.f);
#pragma unroll
  for (int i = 0; i < V; ++i) v[i] = from_float<T>(activate<T>(to_float(v[i]), c.act));
  if (whole)
    *reinterpret_cast<float4*>(row + col) = *reinterpret_cast<const float4*>(v);
  else
    for (int i = 0; i < V; ++i)
      if (col + i < c.columns) row[col + i] = v[i];
}

BT_EXPORT int bt_activate_call(void* stream, const ActivateCall* c) {
  if (c->tokens <= 0) return BT_OK;
  if (c->columns <= 0 || !c->rows || c->ld < c->columns || c->act < 0 || c->act > 2)
    BT_REFUSE("activate: %d columns of rows %lld apart, activation %d", c->columns, (long long)c->ld, c->act);
  if (c->tokens > 65535) BT_REFUSE("activate: %d rows in one call, at most 65535", c->tokens);
  const int per = 256 * (c->dtype == 0 ? 4 : 8);
  dim3 grid((c->columns + per - 1) / per, c->tokens), block(256);
  if (c->dtype == 0)
    hipLaunchKernelGGL(activate_kernel<float>, grid, block, 0, (hipStream_t)stream, *c);
  else
    hipLaunchKernelGGL(activate_kernel<bf16_t>, grid, block, 0, (hipStream_t)stream, *c);
  return bt_check_launch("activate");
}
