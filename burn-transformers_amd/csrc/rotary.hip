// Kernels of attention mixers that turn queries and keys by their positions (rotary positions).
//   * head norms and rotation into the cache: behind a fused query/key/value projection that leaves
//     32-bit sums, every query and key head is divided by its root mean square (times a scale
//     shared by the heads), the first `rot_dims` channels of each head are turned by the token's
//     position, queries go to a buffer for the attention kernel and keys and values straight into
//     the paged cache at the token's position.  Queries/keys and values may have different head
//     sizes; the cache keeps heads of one size, and what lies behind a head's own channels is zero.
// Channel i < rot_dims / 2 is paired with channel i + rot_dims / 2 (`pairing` 0, the halves) or channel
// 2 i with channel 2 i + 1 (`pairing` 1, neighbours); the pair (u, v) at position p
// becomes (u cos a - v sin a, v cos a + u sin a), a = p * inv_freq[i], sine and cosine times `amplitude`
// (one where the frequencies are not rescaled; schedules that slow long waves let both grow a little).  With `norm_span` 1 the root mean
// square is taken over a token's WHOLE query (or key) projection, all heads at once, and the scale has
// an entry for every channel of the projection.  The frequencies come as a
// table, so any schedule of them (scaled, interpolated) is the caller's.  Norms, angles and the
// rotation are 32-bit.
// Three more things a mixer may ask for on the way:
//   * `maps` 2: every head has that many query and key parts, laid out part by part behind each other; part m of a
//     query head becomes a query of its own with its channels at m * dim and zeros elsewhere, and a key head's parts
//     lie side by side in ONE cached head, so that several score maps share that head's values;
//   * `values_from_keys`: the values are the projected keys as they are before norm and rotation (the rows then hold no
//     values of their own);
//   * `temp_coef`: queries times 1 + temp_coef * ln(floor((p + 1) / temp_every) + 1), growing with the position p.
#include "host.h"

struct HeadRotaryCall {
  int dtype;              // element type of `q_out` and of the cache: 0 float32, 1 bfloat16
  int tokens;
  int heads, kv_heads;
  int dim, vdim;          // a head's channels of queries and keys, and of values, in `in`
  int rot_dims;           // channels of each query and key head that are turned: even, at most dim; 0: none
  float eps;
  const float* in;        // [tokens][ld] float32: queries (heads * dim), keys (kv_heads * dim), values (kv_heads * vdim)
  int64_t ld;
  const float* q_gamma;   // [dim] ([heads * dim] with norm_span 1) or null: no norm of the queries
  const float* k_gamma;   // [dim] ([kv_heads * dim] with norm_span 1) or null
  const float* inv_freq;  // [rot_dims / 2]
  void* q_out;            // [tokens][ld_q]: head j at columns j * kv.head_dim
  int64_t ld_q;
  const int* tok_seq;
  const int* tok_pos;
  KvView kv;              // kv_heads heads of head_dim >= max(dim, vdim)
  int pairing;            // 0: channel i turns with channel i + rot_dims / 2; 1: channel 2 i with channel 2 i + 1
  int norm_span;          // 0: every head over its own root mean square; 1: the whole projection over one
  float amplitude;        // factor on every sine and cosine
  int maps;               // query and key parts a head: 1 or 2
  int values_from_keys;
  float temp_coef;        // 0: no temperature
  int temp_every;
};

#define HR_WAVES 4
#define HR_MAX_DIM 256
#define HR_AHEAD 8      // columns of a norm over a whole projection that a lane asks for at once

// A decode step has few tokens: what the kernel takes is its chain of trips to memory.  So all that does not depend on another load is asked
// for at the start (the unit's channels, COLS a lane, and their scales; the position, the sequence, the angles), and the table of blocks is read
// while the unit's channels are on their way.
// Measured in a decode step (us, one load after the other / so): 4 tokens, 8 heads on 2 of 128 with norms 4.6 / 3.3, 8 tokens 3.0 to 4.2 / 2.6 to 3.0.
template <typename T, int COLS>
__global__ void __launch_bounds__(HR_WAVES * 64) head_rotary_kernel(HeadRotaryCall c) {
  __shared__ float rows[HR_WAVES][64 * COLS];
  __shared__ float sines[HR_MAX_DIM / 2], cosines[HR_MAX_DIM / 2];      // of the token's position: the same for all its heads
  const int t = blockIdx.x, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n_q = c.heads * c.maps, n_k = c.kv_heads * c.maps;
  const int units = n_q + n_k + c.kv_heads;
  const bool active = blockIdx.y * HR_WAVES + wave < units;             // (the others do the last unit's work and leave before the stores)
  const int unit = active ? blockIdx.y * HR_WAVES + wave : units - 1;   // a query head, then a key head, then a value head
  const bool is_q = unit < n_q, is_k = !is_q && unit < n_q + n_k;
  const int head = is_q ? unit : (is_k ? unit - n_q : unit - n_q - n_k);      // (with maps: the part's number)
  const int n = (is_q || is_k) ? c.dim : c.vdim;
  const int hd = c.kv.head_dim, half = c.rot_dims >> 1;
  float* row = rows[wave];
  const int64_t first = is_q ? (int64_t)head * c.dim
                             : (is_k || c.values_from_keys ? (int64_t)(n_q + head) * c.dim
                                                           : (int64_t)(n_q + n_k) * c.dim + (int64_t)head * c.vdim);
  const float* src = c.in + (int64_t)t * c.ld + first;
  const float* gamma = is_q ? c.q_gamma : (is_k ? c.k_gamma : nullptr);
  const float* scales = gamma ? gamma + (c.norm_span == 1 ? head * c.dim : 0) : src;      // (src: a valid place, not used)
  const int pos = c.tok_pos[t], seq = c.tok_seq[t];
  const int angle = threadIdx.x < half ? threadIdx.x : 0;               // (half is at most 128)
  float v[COLS], g[COLS];
#pragma unroll
  for (int k = 0; k < COLS; ++k) {
    const int col = lane + 64 * k;
    v[k] = src[col < n ? col : 0];
    g[k] = scales[col < n ? col : 0];
  }
  const float freq = half > 0 ? c.inv_freq[angle] : 0.f;
  const int64_t base = kv_block_base(c.kv, seq, pos, is_q ? 0 : is_k ? head / c.maps : head);
  asm volatile("" ::"s"(base));                            // (here, while the unit's channels are on their way, not where the stores use it)
  float squares = 0.f;
#pragma unroll
  for (int k = 0; k < COLS; ++k)
    if (lane + 64 * k < n) squares = fmaf(v[k], v[k], squares);
  if (gamma) {
    int over = n;
    if (c.norm_span == 1) {
      // every wave of a projection adds up the same squares in the same order: the heads agree exactly
      over = (is_q ? n_q : n_k) * c.dim;
      const float* whole = c.in + (int64_t)t * c.ld + (is_q ? 0 : (int64_t)n_q * c.dim);
      squares = 0.f;
      for (int col0 = lane; col0 - lane < over; col0 += 64 * HR_AHEAD) {
        float w[HR_AHEAD];
#pragma unroll
        for (int u = 0; u < HR_AHEAD; ++u) w[u] = whole[col0 + 64 * u < over ? col0 + 64 * u : 0];
#pragma unroll
        for (int u = 0; u < HR_AHEAD; ++u)
          if (col0 + 64 * u < over) squares = fmaf(w[u], w[u], squares);
      }
    }
    const float rstd = 1.0f / sqrtf(wave_sum(squares) / (float)over + c.eps);
#pragma unroll
    for (int k = 0; k < COLS; ++k) v[k] = v[k] * rstd * g[k];
  }
#pragma unroll
  for (int k = 0; k < COLS; ++k) row[lane + 64 * k] = v[k];             // (behind the unit's channels: read by nobody)
  if (threadIdx.x < half) {
    float sn, cs;
    sincosf((float)pos * freq, &sn, &cs);
    sines[threadIdx.x] = sn * c.amplitude;
    cosines[threadIdx.x] = cs * c.amplitude;
  }
  __syncthreads();
  if (!active) return;
  const bool turned = (is_q || is_k) && half > 0;
  T* q_out = static_cast<T*>(c.q_out) + (int64_t)t * c.ld_q + (int64_t)head * hd;
  T* keys = static_cast<T*>(c.kv.keys) + base;
  T* values = static_cast<T*>(c.kv.values) + base;
  const int part = is_q || is_k ? head % c.maps : 0, offset = part * c.dim;    // where the unit's channels start in its row
  const float factor = is_q && c.temp_coef != 0.f ? 1.0f + c.temp_coef * logf((float)((pos + 1) / c.temp_every) + 1.0f) : 1.0f;
  auto store = [&](int col, float v) {
    if (is_q)
      q_out[col] = from_float<T>(v * factor);
    else if (is_k)
      keys[key_offset(hd, pos, col)] = from_float<T>(v);
    else
      values[value_offset(hd, pos, col)] = from_float<T>(v);
  };
  // a lane takes a pair of channels
  if (turned)
    for (int i = lane; i < half; i += 64) {
      const float sn = sines[i], cs = cosines[i];
      const int first = c.pairing == 1 ? 2 * i : i, second = c.pairing == 1 ? 2 * i + 1 : i + half;
      const float u = row[first], v = row[second];
      store(offset + first, u * cs - v * sn);
      store(offset + second, v * cs + u * sn);
    }
  // the channels that are not turned, and zeros around a query's part (behind a key's last part)
  const int done = turned ? c.rot_dims : 0;
  const int from = is_q ? 0 : offset + done, to = is_k && part + 1 < c.maps ? offset + n : hd;
  for (int col = from + lane; col < to; col += 64) {
    const int channel = col - offset;
    if (channel < 0 || channel >= n) store(col, 0.f);
    else if (channel >= done) store(col, row[channel]);
  }
}

// Steps of many tokens: a wave takes one token and HRR_UNITS of its heads, a lane two neighbouring channels of each, so that
// all its rows are asked for at once, the sines are worked out once for the heads (an angle a lane) and nothing waits at a
// barrier.  Taken for rows of whole pairs up to 128 channels.  Measured against the kernel above (us, above / this; 8 heads on 2 of 128, 64
// channels turned, bfloat16, a norm a head): 512 tokens 5.3 / 4.9, 768 6.9 / 5.2, 1,024 8.2 / 5.4, 2,048 13.9 / 7.7.  What is left is the
// sines (the angles reduced in 32 bits) and the values' stores of two bytes: bytes alone would take 3.4 us at 1,809 tokens.
// Taken where there is enough to share: with one norm over all heads, which the kernel above works out once a head, from 128 tokens on
// for rows of 1,024 query channels, and elsewhere, as without such a norm from 768 tokens on, by the heads of all tokens.  The two kernels add a norm's
// squares in different orders (columns 64 apart, pairs 128 apart), so the lines with norms also say which sums a step has: they stay where they are even
// where the kernel above is now the faster one.  Measured (us, the kernel above / this; queries on keys of channels, heads of all tokens in brackets): one norm over all
// heads, 8 on 2 of 128 128 tokens 3.6 / 4.8, 256 4.1 / 4.9, 512 (6,144) 5.6 / 5.0, 6 on 2 of 128 512 (5,120) 5.0 / 5.4, 768 6.4 / 5.9, 4 on 1 of 64 768 (4,608) 4.8 / 4.3, 2 on 1 of
// 128 1,024 (4,096) 4.4 / 4.8, 1,536 (6,144) 5.5 / 5.0, 12 on 12 of 64 128 (4,608) 4.2 / 5.0, 192 (6,912) 5.2 / 5.2, 256 6.3 / 5.4; a norm a head, 2 on 1 of 128 1,280
// (5,120) 4.8 / 4.8, 1,536 (6,144) 5.3 / 4.8, 3 on 1 1,280 (6,400) 6.1 / 5.1, 4 on 4 of 32 512 (6,144) 4.5 / 4.9, 768 5.7 / 5.1; without a norm 2 on 1 of 64 768 (3,072) 3.4 / 3.6, 1,024
// (4,096) 3.7 / 3.7, 1,280 4.2 / 3.9, 1 on 1 of 64 768 (2,304) 3.3 / 3.3, 4 on 1 of 128 768 (4,608) 4.7 / 3.6.
#define HRR_UNITS 4
#define HRR_MIN_TOKENS 768
#define HRR_MIN_TOKENS_WHOLE 128
#define HRR_WHOLE_COLUMNS 1024
#define HRR_MIN_HEADS 4096
#define HRR_MIN_HEADS_WHOLE 6144
#define HRR_MIN_HEADS_NORM 7680

template <typename T>
__global__ void __launch_bounds__(256) head_rotary_rows_kernel(HeadRotaryCall c) {
  typedef __attribute__((__vector_size__(2 * sizeof(T)))) T T2;
  const int lane = threadIdx.x & 63;
  const int t = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  if (t >= c.tokens) return;                               // (a whole wave; there is no barrier)
  const int first_unit = blockIdx.y * HRR_UNITS, n_q = c.heads, n_k = c.kv_heads, units = n_q + 2 * n_k;
  const int ch = 2 * lane, hd = c.kv.head_dim, half = c.rot_dims >> 1;
  const float* in = c.in + (int64_t)t * c.ld;
  float2 x[HRR_UNITS];
#pragma unroll
  for (int i = 0; i < HRR_UNITS; ++i) {
    const int unit = first_unit + i;
    x[i] = make_float2(0.f, 0.f);
    if (unit >= units) continue;
    const bool is_v = unit >= n_q + n_k;
    const int from = !is_v ? unit * c.dim : c.values_from_keys ? (unit - n_k) * c.dim : (n_q + n_k) * c.dim + (unit - n_q - n_k) * c.vdim;
    if (ch < (is_v ? c.vdim : c.dim)) x[i] = *reinterpret_cast<const float2*>(in + from + ch);
  }
  const int pos = c.tok_pos[t];
  const int64_t block_base = first_unit + HRR_UNITS > n_q ? kv_block_base(c.kv, c.tok_seq[t], pos, 0) : 0;
  float q_rstd = 0.f, k_rstd = 0.f;
  if (c.norm_span == 1) {
    auto whole = [&](int from, int all) {
      float squares = 0.f;
      for (int col = ch; col < all; col += 128) {
        const float2 v = *reinterpret_cast<const float2*>(in + from + col);
        squares = fmaf(v.y, v.y, fmaf(v.x, v.x, squares));
      }
      return 1.0f / sqrtf(wave_sum(squares) / (float)all + c.eps);
    };
    if (c.q_gamma && first_unit < n_q) q_rstd = whole(0, n_q * c.dim);
    if (c.k_gamma && first_unit + HRR_UNITS > n_q && first_unit < n_q + n_k) k_rstd = whole(n_q * c.dim, n_k * c.dim);
  }
  // the lane's two channels turn by these (neighbours: both by one); channels that are not turned by nothing
  const bool turned = ch < c.rot_dims, second = c.pairing == 0 && ch >= half;
  float2 sn = make_float2(0.f, 0.f), cs = make_float2(1.f, 1.f);
  if (half > 0 && first_unit < n_q + n_k) {                // (the same for the whole wave; half is at most 64: lane i has angle i)
    float s, co;
    sincosf((float)pos * c.inv_freq[lane < half ? lane : 0], &s, &co);
    s *= c.amplitude;
    co *= c.amplitude;
    const int i = !turned ? 0 : c.pairing == 1 ? lane : second ? ch - half : ch, i1 = c.pairing == 1 ? i : i + 1;
    sn = make_float2(__shfl(s, i, 64), __shfl(s, i1, 64));
    cs = make_float2(__shfl(co, i, 64), __shfl(co, i1, 64));
  }
  const int partner = !turned ? lane : second ? lane - half / 2 : lane + half / 2;
  const float factor = c.temp_coef != 0.f ? 1.0f + c.temp_coef * logf((float)((pos + 1) / c.temp_every) + 1.0f) : 1.0f;
#pragma unroll
  for (int i = 0; i < HRR_UNITS; ++i) {
    const int unit = first_unit + i;
    if (unit >= units) return;
    const bool is_q = unit < n_q, is_v = unit >= n_q + n_k;
    const int head = is_q ? unit : is_v ? unit - n_q - n_k : unit - n_q;
    float2 v = x[i];
    const float* gamma = is_q ? c.q_gamma : is_v ? nullptr : c.k_gamma;
    if (gamma) {
      const float rstd = c.norm_span == 1 ? (is_q ? q_rstd : k_rstd) : 1.0f / sqrtf(wave_sum(fmaf(v.y, v.y, v.x * v.x)) / (float)c.dim + c.eps);
      if (ch < c.dim) {
        const float* g = gamma + (c.norm_span == 1 ? head * c.dim : 0) + ch;
        v.x = v.x * rstd * g[0];
        v.y = v.y * rstd * g[1];
      }
    }
    if (!is_v && half > 0) {
      float2 o;                                            // what each channel turns with, signed
      if (c.pairing == 1) {
        o = make_float2(-v.y, v.x);
      } else {
        o.x = __shfl(v.x, partner, 64);
        o.y = __shfl(v.y, partner, 64);
        if (!second) o = make_float2(-o.x, -o.y);
      }
      if (turned) v = make_float2(v.x * cs.x + o.x * sn.x, v.y * cs.y + o.y * sn.y);
    }
    if (ch >= hd) continue;
    if (is_q) {
      *reinterpret_cast<T2*>(static_cast<T*>(c.q_out) + (int64_t)t * c.ld_q + (int64_t)head * hd + ch) = T2{from_float<T>(v.x * factor), from_float<T>(v.y * factor)};
    } else if (!is_v) {
      *reinterpret_cast<T2*>(static_cast<T*>(c.kv.keys) + block_base + head * c.kv.head_stride + key_offset(hd, pos, ch)) = T2{from_float<T>(v.x), from_float<T>(v.y)};
    } else {
      T* values = static_cast<T*>(c.kv.values) + block_base + head * c.kv.head_stride;
      values[value_offset(hd, pos, ch)] = from_float<T>(v.x);
      values[value_offset(hd, pos, ch + 1)] = from_float<T>(v.y);
    }
  }
}

template <typename T>
static void launch_head_rotary(hipStream_t stream, const HeadRotaryCall& c, int units) {
  dim3 grid(c.tokens, (units + HR_WAVES - 1) / HR_WAVES), block(HR_WAVES * 64);
  const int channels = c.dim > c.vdim ? c.dim : c.vdim;
  if (channels <= 64) hipLaunchKernelGGL((head_rotary_kernel<T, 1>), grid, block, 0, stream, c);
  else if (channels <= 128) hipLaunchKernelGGL((head_rotary_kernel<T, 2>), grid, block, 0, stream, c);
  else hipLaunchKernelGGL((head_rotary_kernel<T, 4>), grid, block, 0, stream, c);
}

BT_EXPORT int bt_head_rotary_call(void* stream, const HeadRotaryCall* c) {
  if (c->tokens <= 0) return BT_OK;
  if (c->heads <= 0 || c->kv_heads <= 0 || c->heads % c->kv_heads != 0)
    BT_REFUSE("head_rotary: %d query heads cannot share %d key/value heads", c->heads, c->kv_heads);
  if (c->dim <= 0 || c->vdim <= 0 || c->dim > HR_MAX_DIM || c->vdim > HR_MAX_DIM)
    BT_REFUSE("head_rotary: head sizes %d and %d outside 1..%d", c->dim, c->vdim, HR_MAX_DIM);
  if ((c->pairing != 0 && c->pairing != 1) || (c->norm_span != 0 && c->norm_span != 1))
    BT_REFUSE("head_rotary: pairing %d and norm_span %d must be 0 or 1", c->pairing, c->norm_span);
  if (c->rot_dims < 0 || c->rot_dims % 2 != 0 || c->rot_dims > c->dim)
    BT_REFUSE("head_rotary: %d turned channels must be even and at most the head size %d", c->rot_dims, c->dim);
  if (c->maps != 1 && c->maps != 2) BT_REFUSE("head_rotary: %d query and key parts a head, 1 or 2 are possible", c->maps);
  if (c->values_from_keys && (c->maps != 1 || c->vdim != c->dim))
    BT_REFUSE("head_rotary: values that are the keys have the keys' size (%d, not %d) and one part a head", c->dim, c->vdim);
  if (c->temp_coef != 0.f && c->temp_every <= 0) BT_REFUSE("head_rotary: a temperature step every %d positions", c->temp_every);
  if (c->kv.kv_heads != c->kv_heads || c->kv.head_dim < c->maps * c->dim || c->kv.head_dim < c->vdim)
    BT_REFUSE("head_rotary: the cache keeps %d heads of %d, the mixer has %d of %d and %d", c->kv.kv_heads,
              c->kv.head_dim, c->kv_heads, c->dim, c->vdim);
  if (c->ld < (int64_t)(c->heads + c->kv_heads) * c->maps * c->dim + (c->values_from_keys ? 0 : (int64_t)c->kv_heads * c->vdim) ||
      c->ld_q < (int64_t)c->heads * c->maps * c->kv.head_dim)
    BT_REFUSE("head_rotary: the rows do not hold the heads");
  if (!c->in || !c->q_out || !c->tok_seq || !c->tok_pos || !c->kv.blocks || !c->kv.keys || !c->kv.values ||
      (c->rot_dims > 0 && !c->inv_freq))
    BT_REFUSE("head_rotary: missing operand");
  const int units = (c->heads + c->kv_heads) * c->maps + c->kv_heads;
  const int hd = c->kv.head_dim;
  const uintptr_t pair = (c->dtype == 0 ? 8 : 4) - 1;      // of two elements of the outputs
  const bool norms = c->q_gamma || c->k_gamma, whole = norms && c->norm_span == 1;
  const bool many = c->tokens >= (whole ? HRR_MIN_TOKENS_WHOLE : HRR_MIN_TOKENS) &&
                    ((whole && (int64_t)c->heads * c->dim >= HRR_WHOLE_COLUMNS) || (int64_t)c->tokens * units >= (whole ? HRR_MIN_HEADS_WHOLE : norms ? HRR_MIN_HEADS_NORM : HRR_MIN_HEADS));
  const bool rows = many && c->maps == 1 && hd <= 128 && hd % 2 == 0 && c->dim % 2 == 0 && c->vdim % 2 == 0 && c->ld % 2 == 0 &&
                    c->ld_q % 2 == 0 && c->kv.block_stride % 2 == 0 && c->kv.head_stride % 2 == 0 && (c->pairing == 1 || c->rot_dims % 4 == 0) && ((uintptr_t)c->in & 7) == 0 &&
                    (((uintptr_t)c->q_out | (uintptr_t)c->kv.keys | (uintptr_t)c->kv.values) & pair) == 0;
  if (rows) {
    const dim3 grid((c->tokens + 3) / 4, (units + HRR_UNITS - 1) / HRR_UNITS);
    if (c->dtype == 0)
      hipLaunchKernelGGL(head_rotary_rows_kernel<float>, grid, dim3(256), 0, (hipStream_t)stream, *c);
    else
      hipLaunchKernelGGL(head_rotary_rows_kernel<bf16_t>, grid, dim3(256), 0, (hipStream_t)stream, *c);
    return bt_check_launch("head_rotary");
  }
  if (c->dtype == 0)
    launch_head_rotary<float>((hipStream_t)stream, *c, units);
  else
    launch_head_rotary<bf16_t>((hipStream_t)stream, *c, units);
  return bt_check_launch("head_rotary");
}
