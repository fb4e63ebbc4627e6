// Row-wise e4m3 quantiser (one power-of-two scale per 128-element row).
// HBM-bound: reads 2 B and writes 1 B per element plus 4 B per row; one 64-lane wave per row
// group, each lane handling 8 consecutive elements (16-byte loads, 8-byte stores).
#include "window.h"

namespace {

__device__ __forceinline__ float wave_max16(float v) {   // max over the 16 lanes sharing a row
  v = fmaxf(v, xor16(v, 1));
  v = fmaxf(v, xor16(v, 2));
  v = fmaxf(v, xor16(v, 4));
  v = fmaxf(v, xor16(v, 8));
  return v;
}

// A weight per row: fp32, or bf16 as it came; AnyWeight times `scale`, rounded to its own type as a tensor operation would
struct F32Weight { const float* p; __device__ float operator[](int64_t i) const { return p[i]; } };
struct AnyWeight {
  const void* p;
  bool bf16;
  float scale;
  __device__ float operator[](int64_t i) const {
    return bf16 ? bf16_bits_to_f32(f32_to_bf16_bits(bf16_bits_to_f32(((const unsigned short*)p)[i]) * scale)) : ((const float*)p)[i] * scale;
  }
};

// cols == 128: 16 lanes per row, 4 rows per wave, 16 rows per 256-thread block.
template <class W>
__device__ __forceinline__ void quant128_rows(unsigned block, const uint4* __restrict__ x, uint2* __restrict__ x8,
                                              float* __restrict__ scale_inv, int64_t rows, float eps, int pow2, W w_in, float w_factor,
                                              float* __restrict__ w_scaled) {
  int64_t row = (int64_t)block * 16 + (threadIdx.x >> 4);
  int sub = threadIdx.x & 15;
  bool live = row < rows;
  uint4 raw = live ? x[row * 16 + sub] : make_uint4(0, 0, 0, 0);
  unsigned w[4] = {raw.x, raw.y, raw.z, raw.w};
  float v[8];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    v[2 * i] = __builtin_bit_cast(float, w[i] << 16);
    v[2 * i + 1] = __builtin_bit_cast(float, w[i] & 0xffff0000u);
  }
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < 8; i++) amax = fmaxf(amax, fabsf(v[i]));
  amax = wave_max16(amax);
  amax = fmaxf(amax, eps);
  float scale = 448.0f / amax;                       // correctly rounded fp32 division
  if (pow2) scale = __builtin_bit_cast(float, __builtin_bit_cast(unsigned, scale) & 0xff800000u);
  float q[8];
#pragma unroll
  for (int i = 0; i < 8; i++) q[i] = fminf(fmaxf(v[i] * scale, -448.0f), 448.0f);  // cvt does not saturate
  int lo = 0, hi = 0;
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], lo, false);
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], lo, true);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(q[4], q[5], hi, false);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(q[6], q[7], hi, true);
  if (live) {
    x8[row * 16 + sub] = make_uint2((unsigned)lo, (unsigned)hi);
    if (sub == 0) {
      const float si = 1.0f / scale;
      scale_inv[row] = si;
      if (w_scaled) w_scaled[row] = (w_in[row] * si) * w_factor;      // two roundings, as two separate multiplications
    }
  }
}

__global__ __launch_bounds__(256) void quant128_kernel(const uint4* __restrict__ x, uint2* __restrict__ x8,
                                                       float* __restrict__ scale_inv, int64_t rows,
                                                       float eps, int pow2, const float* __restrict__ w_in,
                                                       float w_factor, float* __restrict__ w_scaled) {
  quant128_rows(blockIdx.x, x, x8, scale_inv, rows, eps, pow2, F32Weight{w_in}, w_factor, w_scaled);
}

// Hadamard rotation of a 128-element row (Sylvester order, scaled by 128^-0.5, rounded to bf16 as the
// unfused sequence "fp32 product with the Hadamard matrix -> bf16" does) followed by the same
// quantiser.  The butterfly runs over the 7 index bits: 3 inside a lane's 8 elements, 4 across the
// 16 lanes of a row.  Either output may be absent (x8 == nullptr: rotation only; y == nullptr:
// quantised payload only).
template <class W>
__device__ __forceinline__ void rotate_quant128_rows(unsigned block, const uint4* __restrict__ x, uint2* __restrict__ x8,
                                                     float* __restrict__ scale_inv, uint4* __restrict__ y, int64_t rows, float eps, int pow2,
                                                     W w_in, float w_factor, float* __restrict__ w_scaled) {
  int64_t row = (int64_t)block * 16 + (threadIdx.x >> 4);
  int sub = threadIdx.x & 15;
  bool live = row < rows;
  uint4 raw = live ? x[row * 16 + sub] : make_uint4(0, 0, 0, 0);
  unsigned w[4] = {raw.x, raw.y, raw.z, raw.w};
  float v[8];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    v[2 * i] = __builtin_bit_cast(float, w[i] << 16);
    v[2 * i + 1] = __builtin_bit_cast(float, w[i] & 0xffff0000u);
  }
#pragma unroll
  for (int m = 1; m < 8; m <<= 1)
#pragma unroll
    for (int i = 0; i < 8; i++)
      if (!(i & m)) { const float a = v[i], b = v[i | m]; v[i] = a + b; v[i | m] = a - b; }
#pragma unroll
  for (int m = 1; m < 16; m <<= 1)
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const float o = xor16(v[i], m);
      v[i] = (sub & m) ? o - v[i] : v[i] + o;
    }
  unsigned yb[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    yb[i] = cvt_pk_bf16(v[2 * i] * 0.08838834764831845f, v[2 * i + 1] * 0.08838834764831845f);
    v[2 * i] = __builtin_bit_cast(float, yb[i] << 16);
    v[2 * i + 1] = __builtin_bit_cast(float, yb[i] & 0xffff0000u);
  }
  if (live && y) y[row * 16 + sub] = make_uint4(yb[0], yb[1], yb[2], yb[3]);
  if (!x8) return;
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < 8; i++) amax = fmaxf(amax, fabsf(v[i]));
  amax = wave_max16(amax);
  amax = fmaxf(amax, eps);
  float scale = 448.0f / amax;
  if (pow2) scale = __builtin_bit_cast(float, __builtin_bit_cast(unsigned, scale) & 0xff800000u);
  float q[8];
#pragma unroll
  for (int i = 0; i < 8; i++) q[i] = fminf(fmaxf(v[i] * scale, -448.0f), 448.0f);
  int lo = 0, hi = 0;
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], lo, false);
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], lo, true);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(q[4], q[5], hi, false);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(q[6], q[7], hi, true);
  if (live) {
    x8[row * 16 + sub] = make_uint2((unsigned)lo, (unsigned)hi);
    if (sub == 0) {
      const float si = 1.0f / scale;
      scale_inv[row] = si;
      if (w_scaled) w_scaled[row] = (w_in[row] * si) * w_factor;      // two roundings, as two separate multiplications
    }
  }
}

__global__ __launch_bounds__(256) void rotate_quant128_kernel(const uint4* __restrict__ x, uint2* __restrict__ x8,
                                                              float* __restrict__ scale_inv, uint4* __restrict__ y,
                                                              int64_t rows, float eps, int pow2,
                                                              const float* __restrict__ w_in, float w_factor,
                                                              float* __restrict__ w_scaled) {
  rotate_quant128_rows(blockIdx.x, x, x8, scale_inv, y, rows, eps, pow2, F32Weight{w_in}, w_factor, w_scaled);
}

// What the indexer's logits wait for, side by side in one launch: the quantised queries with their weights, the quantised keys, and the
// windows of one sequence.  Each part alone fills a fraction of the chip for a chunk of a prompt, and takes its 3 - 5 us behind the
// other two.  The whole pass, us, as three launches and as one: chunks of a few dozen tokens 76.5 and 68.8, 61 tokens x 64 heads behind
// 20 000 82.2 and 78.0, 1500 behind 6692 1014 and 1010, 3072 queries over compressed keys, forward and backward, 1567 and 1564.
struct InputArgs {
  const uint4 *q, *k;
  uint2 *q8, *k8;
  float *q_scale, *k_scale;
  int64_t q_rows, k_rows;
  AnyWeight w_in;
  float w_factor;
  float* w_scaled;
  unsigned q_blocks, k_blocks;
  float eps;
  int pow2;
  int S, ratio, keys;
  long long offset;
  int *ks, *ke;
};
template <bool ROTATE>
__global__ __launch_bounds__(256) void indexer_inputs_kernel(const InputArgs a) {
  const unsigned b = blockIdx.x;
  if (b < a.q_blocks) {
    if (ROTATE) rotate_quant128_rows(b, a.q, a.q8, a.q_scale, nullptr, a.q_rows, a.eps, a.pow2, a.w_in, a.w_factor, a.w_scaled);
    else quant128_rows(b, a.q, a.q8, a.q_scale, a.q_rows, a.eps, a.pow2, a.w_in, a.w_factor, a.w_scaled);
  } else if (b < a.q_blocks + a.k_blocks) {
    if (ROTATE) rotate_quant128_rows(b - a.q_blocks, a.k, a.k8, a.k_scale, nullptr, a.k_rows, a.eps, a.pow2, F32Weight{nullptr}, 0.f, nullptr);
    else quant128_rows(b - a.q_blocks, a.k, a.k8, a.k_scale, a.k_rows, a.eps, a.pow2, F32Weight{nullptr}, 0.f, nullptr);
  } else {
    const int i = (int)(b - a.q_blocks - a.k_blocks) * 256 + (int)threadIdx.x;
    if (i >= a.S) return;
    const long long end = a.offset + i + 1;
    a.ks[i] = 0;
    a.ke[i] = (int)(a.ratio ? min(max(end / a.ratio, 1ll), (long long)a.keys) : end);
  }
}

// The quantiser over rows that are padded on the way: token t's heads_in rows of dim_in elements become heads_out rows of 128,
// zeros in between (as if the bf16 tensor had been padded first: zero rows get the scale of the epsilon floor, and the
// weight 0).  Weights may be bf16.
__global__ __launch_bounds__(256) void quant_padded_kernel(const unsigned short* __restrict__ x, int heads_in, int dim_in, int heads_out,
                                                           uint2* __restrict__ x8, float* __restrict__ scale_inv, int64_t rows,
                                                           float eps, int pow2, const void* __restrict__ w_in, int w_bf16, float w_factor,
                                                           float* __restrict__ w_scaled) {
  const int64_t row = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
  const int sub = threadIdx.x & 15;
  if (row >= rows) return;               // (the 16 lanes of a row leave together)
  const int64_t tok = row / heads_out;
  const int h = (int)(row % heads_out);
  float v[8];
#pragma unroll
  for (int i = 0; i < 8; i++)
    v[i] = h < heads_in && 8 * sub + i < dim_in ? bf16_bits_to_f32(x[(tok * heads_in + h) * dim_in + 8 * sub + i]) : 0.f;
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < 8; i++) amax = fmaxf(amax, fabsf(v[i]));
  amax = fmaxf(wave_max16(amax), eps);
  float scale = 448.0f / amax;
  if (pow2) scale = __builtin_bit_cast(float, __builtin_bit_cast(unsigned, scale) & 0xff800000u);
  float q[8];
#pragma unroll
  for (int i = 0; i < 8; i++) q[i] = fminf(fmaxf(v[i] * scale, -448.0f), 448.0f);
  int lo = 0, hi = 0;
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], lo, false);
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], lo, true);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(q[4], q[5], hi, false);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(q[6], q[7], hi, true);
  x8[row * 16 + sub] = make_uint2((unsigned)lo, (unsigned)hi);
  if (sub == 0) {
    const float si = 1.0f / scale;
    scale_inv[row] = si;
    if (w_scaled) {
      float w = 0.f;
      if (h < heads_in) {
        const int64_t e = tok * heads_in + h;
        w = w_bf16 ? bf16_bits_to_f32(((const unsigned short*)w_in)[e]) : ((const float*)w_in)[e];
      }
      w_scaled[row] = (w * si) * w_factor;
    }
  }
}

// The front end of 64-channel heads, all of them rotary, as quant_padded_kernel's rows of 128: rotary embedding (split pairs, every
// product and the sum rounded to bf16, as the separate operations of rope_steps_kernel round), Hadamard rotation of 64 elements
// (hadamard_kernel<64>), quantiser; keys (one head, behind their norm) and the windows of one sequence beside the queries in one
// launch.  Six launches of 3 - 6 us, and four nodes of the graph each way, became this one, which 1024 tokens x 4 heads leave bound
// by its launch; the payloads are the same bits.
struct NarrowArgs {
  const uint4 *q, *k;                      // [S, heads, 64], [keys, 64]
  const uint4 *cos_t, *sin_t;              // [>= S, keys][64], bf16
  int heads, heads_out;
  int64_t q_rows, k_rows;                  // q_rows = S heads_out
  uint2 *q8, *k8;
  float *q_scale, *k_scale;
  AnyWeight w_in;
  float w_factor;
  float* w_scaled;
  unsigned q_blocks, k_blocks;
  int S;
  long long offset;
  int *ks, *ke;
};
__global__ __launch_bounds__(256) void indexer_narrow_kernel(const NarrowArgs a) {
#pragma clang fp contract(off)
  if (blockIdx.x >= a.q_blocks + a.k_blocks) {
    const int i = (int)(blockIdx.x - a.q_blocks - a.k_blocks) * 256 + (int)threadIdx.x;
    if (i >= a.S) return;
    a.ks[i] = 0;
    a.ke[i] = (int)(a.offset + i + 1);
    return;
  }
  const bool keys = blockIdx.x >= a.q_blocks;
  const int64_t row = (int64_t)(blockIdx.x - (keys ? a.q_blocks : 0)) * 16 + (threadIdx.x >> 4);
  const int sub = threadIdx.x & 15;
  if (row >= (keys ? a.k_rows : a.q_rows)) return;         // (the 16 lanes of a row leave together)
  const unsigned tok = keys ? (unsigned)row : (unsigned)row / (unsigned)a.heads_out, h = keys ? 0 : (unsigned)row % (unsigned)a.heads_out;
  const bool real = keys || (int)h < a.heads;
  float v[8], c[8], s[8];
  auto load8 = [&](const uint4* p, int64_t i, float (&o)[8]) {
    const uint4 raw = real && sub < 8 ? p[i] : make_uint4(0, 0, 0, 0);
    const unsigned w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
    for (int e = 0; e < 4; e++) {
      o[2 * e] = __builtin_bit_cast(float, w[e] << 16);
      o[2 * e + 1] = __builtin_bit_cast(float, w[e] & 0xffff0000u);
    }
  };
  load8(keys ? a.k : a.q, keys ? row * 8 + sub : ((int64_t)tok * a.heads + h) * 8 + sub, v);
  load8(a.cos_t, (int64_t)tok * 8 + sub, c);
  load8(a.sin_t, (int64_t)tok * 8 + sub, s);
  auto round_bf16 = [](float (&t)[8]) {
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      const unsigned u = cvt_pk_bf16(t[i], t[i + 1]);
      t[i] = __builtin_bit_cast(float, u << 16);
      t[i + 1] = __builtin_bit_cast(float, u & 0xffff0000u);
    }
  };
  float o[8];                              // element e of lane s pairs with element e of lane s ^ 4
#pragma unroll
  for (int i = 0; i < 8; i++) {
    o[i] = xor16(v[i], 4);
    o[i] = (sub < 4 ? -o[i] : o[i]) * s[i];
    v[i] = v[i] * c[i];
  }
  round_bf16(v);
  round_bf16(o);
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = v[i] + o[i];
  round_bf16(v);
#pragma unroll
  for (int m = 1; m < 8; m <<= 1)
#pragma unroll
    for (int i = 0; i < 8; i++)
      if (!(i & m)) { const float x = v[i], y = v[i | m]; v[i] = x + y; v[i | m] = x - y; }
#pragma unroll
  for (int m = 1; m < 8; m <<= 1)
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const float x = xor16(v[i], m);
      v[i] = (sub & m) ? x - v[i] : v[i] + x;
    }
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = v[i] * 0.125f;
  round_bf16(v);
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < 8; i++) amax = fmaxf(amax, fabsf(v[i]));
  amax = fmaxf(wave_max16(amax), 1e-12f);
  const float scale = __builtin_bit_cast(float, __builtin_bit_cast(unsigned, 448.0f / amax) & 0xff800000u);
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = fminf(fmaxf(v[i] * scale, -448.0f), 448.0f);
  int lo = 0, hi = 0;
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], lo, false);
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], lo, true);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(v[4], v[5], hi, false);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(v[6], v[7], hi, true);
  (keys ? a.k8 : a.q8)[row * 16 + sub] = make_uint2((unsigned)lo, (unsigned)hi);
  if (sub == 0) {
    const float si = 1.0f / scale;
    (keys ? a.k_scale : a.q_scale)[row] = si;
    if (!keys) a.w_scaled[row] = ((real ? a.w_in[(int64_t)tok * a.heads + h] : 0.f) * si) * a.w_factor;
  }
}

// The indexer front end behind its projections, one pass over a 128-element row:
//   LN    (key rows)  y = ((x - mean) * rstd) * gamma + beta, statistics in fp32, rounded to bf16
//   ROPE              rotation of the leading 64 elements by the row's position (pairs adjacent or split,
//                     the formula and rounding of rope_rows_kernel in rope.hip), rounded to bf16
//   rotation          Hadamard butterfly * 128^-0.5, rounded to bf16 (as rotate_quant128_kernel)
//   quantiser         power-of-two scale, e4m3 payload, optionally weights * scale_inv * factor
// Every stage rounds where the separate operations round, so the payload is that of the unfused sequence.
// Sums run in a fixed order (a lane's 8 elements in sequence, then the 16 lanes of a row by xor 1, 2, 4, 8).
template <bool LN, int PAIRING, class W>   // PAIRING: -1 no rotary part, 0 adjacent pairs, 1 split pairs (i, i + 32)
__device__ __forceinline__ void front128_rows(
    unsigned block, const uint4* __restrict__ x, int64_t rows, int rows_per_token, const float* __restrict__ ln_w,
    const float* __restrict__ ln_b, float ln_eps, const void* __restrict__ cos_t, const void* __restrict__ sin_t,
    int cs_f32, const int* __restrict__ positions, int batch, int rotate, uint2* __restrict__ x8,
    float* __restrict__ scale_inv, uint4* __restrict__ y, float eps, int pow2, W w_in,
    float w_factor, float* __restrict__ w_scaled) {
#pragma clang fp contract(off)
  const int64_t row = (int64_t)block * 16 + (threadIdx.x >> 4);
  const int sub = threadIdx.x & 15;
  const bool live = row < rows;
  const uint4 raw = live ? x[row * 16 + sub] : make_uint4(0, 0, 0, 0);
  const unsigned w[4] = {raw.x, raw.y, raw.z, raw.w};
  float v[8];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    v[2 * i] = __builtin_bit_cast(float, w[i] << 16);
    v[2 * i + 1] = __builtin_bit_cast(float, w[i] & 0xffff0000u);
  }
  auto row_sum = [&](const float (&t)[8]) {
    float s = t[0];
#pragma unroll
    for (int i = 1; i < 8; i++) s = s + t[i];
#pragma unroll
    for (int m = 1; m < 16; m <<= 1) s = s + xor16(s, m);
    return s;
  };
  auto round_bf16 = [&]() {
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      const unsigned u = cvt_pk_bf16(v[i], v[i + 1]);
      v[i] = __builtin_bit_cast(float, u << 16);
      v[i + 1] = __builtin_bit_cast(float, u & 0xffff0000u);
    }
  };
  if (LN) {
    const float mean = row_sum(v) * 0.0078125f;
    float d[8], d2[8];
#pragma unroll
    for (int i = 0; i < 8; i++) { d[i] = v[i] - mean; d2[i] = d[i] * d[i]; }
    const float var = row_sum(d2) * 0.0078125f;
    const float rstd = 1.0f / sqrtf(var + ln_eps);
    const f32x4 g0 = *(const f32x4*)(ln_w + 8 * sub), g1 = *(const f32x4*)(ln_w + 8 * sub + 4);
    const f32x4 b0 = *(const f32x4*)(ln_b + 8 * sub), b1 = *(const f32x4*)(ln_b + 8 * sub + 4);
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = (d[i] * rstd) * (i < 4 ? g0[i] : g1[i - 4]) + (i < 4 ? b0[i] : b1[i - 4]);
    round_bf16();
  }
  if (PAIRING >= 0) {
    const unsigned tok = (unsigned)row / (unsigned)rows_per_token;       // in 32 bits: a 64-bit division is a long routine
    const int64_t pos = live ? (positions ? positions[tok] : tok / (unsigned)batch) : 0;
    auto table8 = [&](const void* t, int col, float (&o)[8]) {     // 8 consecutive entries of the position's row
      if (cs_f32) {
        const f32x4 a = *(const f32x4*)((const float*)t + pos * 64 + col), b = *(const f32x4*)((const float*)t + pos * 64 + col + 4);
#pragma unroll
        for (int i = 0; i < 4; i++) { o[i] = a[i]; o[4 + i] = b[i]; }
      } else {
        const uint4 a = *(const uint4*)((const unsigned short*)t + pos * 64 + col);
        const unsigned u[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
        for (int i = 0; i < 4; i++) { o[2 * i] = __builtin_bit_cast(float, u[i] << 16); o[2 * i + 1] = __builtin_bit_cast(float, u[i] & 0xffff0000u); }
      }
    };
    if (PAIRING == 0) {
      if (sub < 8) {            // pairs (2i, 2i + 1) inside the lane; cos / sin indexed like the elements
        float c[8], s[8];
        table8(cos_t, 8 * sub, c);
        table8(sin_t, 8 * sub, s);
#pragma unroll
        for (int i = 0; i < 8; i += 2) {
          const float x1 = v[i], x2 = v[i + 1];
          v[i] = x1 * c[i] - x2 * s[i];
          v[i + 1] = x2 * c[i + 1] + x1 * s[i + 1];
        }
      }
    } else {
      float o[8];               // element e of lane s pairs with element e of lane s ^ 4 (lanes 0..7 hold the 64 rotary elements)
#pragma unroll
      for (int i = 0; i < 8; i++) o[i] = xor16(v[i], 4);
      if (sub < 8) {
        float c[8], s[8];
        table8(cos_t, 8 * sub, c);
        table8(sin_t, 8 * sub, s);
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = sub < 4 ? v[i] * c[i] - o[i] * s[i] : v[i] * c[i] + o[i] * s[i];
      }
    }
    round_bf16();
  }
  unsigned yb[4];
  if (rotate) {
#pragma unroll
    for (int m = 1; m < 8; m <<= 1)
#pragma unroll
      for (int i = 0; i < 8; i++)
        if (!(i & m)) { const float a = v[i], b = v[i | m]; v[i] = a + b; v[i | m] = a - b; }
#pragma unroll
    for (int m = 1; m < 16; m <<= 1)
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const float o = xor16(v[i], m);
        v[i] = (sub & m) ? o - v[i] : v[i] + o;
      }
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = v[i] * 0.08838834764831845f;
    round_bf16();
  }
#pragma unroll
  for (int i = 0; i < 4; i++) yb[i] = (__builtin_bit_cast(unsigned, v[2 * i]) >> 16) | (__builtin_bit_cast(unsigned, v[2 * i + 1]) & 0xffff0000u);
  if (live && y) y[row * 16 + sub] = make_uint4(yb[0], yb[1], yb[2], yb[3]);
  if (!x8) return;
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < 8; i++) amax = fmaxf(amax, fabsf(v[i]));
  amax = wave_max16(amax);
  amax = fmaxf(amax, eps);
  float scale = 448.0f / amax;
  if (pow2) scale = __builtin_bit_cast(float, __builtin_bit_cast(unsigned, scale) & 0xff800000u);
  float q[8];
#pragma unroll
  for (int i = 0; i < 8; i++) q[i] = fminf(fmaxf(v[i] * scale, -448.0f), 448.0f);
  int lo = 0, hi = 0;
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], lo, false);
  lo = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], lo, true);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(q[4], q[5], hi, false);
  hi = __builtin_amdgcn_cvt_pk_fp8_f32(q[6], q[7], hi, true);
  if (live) {
    x8[row * 16 + sub] = make_uint2((unsigned)lo, (unsigned)hi);
    if (sub == 0) {
      const float si = 1.0f / scale;
      scale_inv[row] = si;
      if (w_scaled) w_scaled[row] = (w_in[row] * si) * w_factor;
    }
  }
}

template <bool LN, int PAIRING>
__global__ __launch_bounds__(256) void indexer_front128_kernel(
    const uint4* __restrict__ x, int64_t rows, int rows_per_token, const float* __restrict__ ln_w,
    const float* __restrict__ ln_b, float ln_eps, const void* __restrict__ cos_t, const void* __restrict__ sin_t,
    int cs_f32, const int* __restrict__ positions, int batch, int rotate, uint2* __restrict__ x8,
    float* __restrict__ scale_inv, uint4* __restrict__ y, float eps, int pow2, const float* __restrict__ w_in,
    float w_factor, float* __restrict__ w_scaled) {
  front128_rows<LN, PAIRING>(blockIdx.x, x, rows, rows_per_token, ln_w, ln_b, ln_eps, cos_t, sin_t, cs_f32, positions, batch, rotate, x8, scale_inv,
                             y, eps, pow2, F32Weight{w_in}, w_factor, w_scaled);
}

// Both sides' front end and the windows in one launch: the keys first (LayerNorm: the longest chain), then the queries' heads, then the
// windows, of packed sequences too.  With the head weights scaled on the way it takes the place of five launches of 3 - 6 us beside
// the queries' own, and of the scaling's node.
struct FrontArgs {
  const uint4 *q, *k;
  int64_t q_rows, k_rows;
  int heads;
  const float *ln_w, *ln_b;
  float ln_eps;
  const void *cos_t, *sin_t;
  int cs_f32;
  const int *pos_q, *pos_k;
  int batch, rotate;
  uint2 *q8, *k8;
  float *q_scale, *k_scale;
  AnyWeight w_in;
  float w_factor;
  float* w_scaled;
  unsigned k_blocks, q_blocks;
  const void* cu;
  int cu_i64, ncu, S, chunk_offset;
  int *ks, *ke, *total;
};
template <int PAIRING>
__global__ __launch_bounds__(256) void indexer_fronts_kernel(const FrontArgs a) {
  const unsigned b = blockIdx.x;
  if (b < a.k_blocks)
    front128_rows<true, PAIRING>(b, a.k, a.k_rows, 1, a.ln_w, a.ln_b, a.ln_eps, a.cos_t, a.sin_t, a.cs_f32, a.pos_k, a.batch, a.rotate, a.k8, a.k_scale,
                                 nullptr, 1e-12f, 1, F32Weight{nullptr}, 0.f, nullptr);
  else if (b < a.k_blocks + a.q_blocks)
    front128_rows<false, PAIRING>(b - a.k_blocks, a.q, a.q_rows, a.heads, nullptr, nullptr, 0.f, a.cos_t, a.sin_t, a.cs_f32, a.pos_q, a.batch, a.rotate,
                                  a.q8, a.q_scale, nullptr, 1e-12f, 1, a.w_in, a.w_factor, a.w_scaled);
  else if (a.cu_i64)
    window_part((int)(b - a.k_blocks - a.q_blocks), (const long long*)a.cu, a.ncu, a.S, a.chunk_offset, a.ks, a.ke, a.total);
  else
    window_part((int)(b - a.k_blocks - a.q_blocks), (const int*)a.cu, a.ncu, a.S, a.chunk_offset, a.ks, a.ke, a.total);
}

}  // namespace

extern "C" int dsa_rotate_quant_e4m3(const void* x, int64_t rows, int cols, void* x8, float* scale_inv, void* y,
                                     float eps, int pow2, void* stream) {
  DSA_REQUIRE(cols == 128, "dsa_rotate_quant_e4m3: only rows of 128 elements are supported, got %d", cols);
  DSA_REQUIRE(rows >= 0, "dsa_rotate_quant_e4m3: negative row count");
  DSA_REQUIRE(x8 != nullptr || y != nullptr, "dsa_rotate_quant_e4m3: no output requested");
  DSA_REQUIRE(x8 == nullptr || scale_inv != nullptr, "dsa_rotate_quant_e4m3: payload without scales");
  DSA_REQUIRE(((uintptr_t)x % 16) == 0 && ((uintptr_t)x8 % 8) == 0 && ((uintptr_t)y % 16) == 0,
              "dsa_rotate_quant_e4m3: misaligned pointer");
  if (rows == 0) return DSA_OK;
  int64_t blocks = (rows + 15) / 16;
  DSA_REQUIRE(blocks < (1ll << 31), "dsa_rotate_quant_e4m3: too many rows");
  rotate_quant128_kernel<<<dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream>>>(
      (const uint4*)x, (uint2*)x8, scale_inv, (uint4*)y, rows, eps, pow2, nullptr, 0.f, nullptr);
  DSA_CHECK_LAUNCH("dsa_rotate_quant_e4m3");
  return DSA_OK;
}

extern "C" int dsa_indexer_inputs_e4m3(const void* q, int64_t q_rows, const void* k, int64_t k_rows, int rotate, void* q8, float* q_scale, void* k8,
                                       float* k_scale, float eps, int pow2, const void* weights, int weights_bf16, float factor,
                                       float* weight_scaled, int S, int64_t offset, int ratio, int keys, int32_t* ks, int32_t* ke, void* stream) {
  DSA_REQUIRE(q_rows >= 0 && k_rows >= 0 && S >= 0 && ratio >= 0 && keys >= 0, "dsa_indexer_inputs_e4m3: bad sizes");
  DSA_REQUIRE(((uintptr_t)q % 16) == 0 && ((uintptr_t)k % 16) == 0 && ((uintptr_t)q8 % 8) == 0 && ((uintptr_t)k8 % 8) == 0,
              "dsa_indexer_inputs_e4m3: misaligned pointer");
  DSA_REQUIRE(q_rows == 0 || (q && q8 && q_scale && weights && weight_scaled), "dsa_indexer_inputs_e4m3: null pointer");
  DSA_REQUIRE((k_rows == 0 || (k && k8 && k_scale)) && (S == 0 || (ks && ke)), "dsa_indexer_inputs_e4m3: null pointer");
  const int64_t q_blocks = (q_rows + 15) / 16, k_blocks = (k_rows + 15) / 16, blocks = q_blocks + k_blocks + dsa_cdiv(S, 256);
  DSA_REQUIRE(blocks < (1ll << 31), "dsa_indexer_inputs_e4m3: too many rows");
  if (blocks == 0) return DSA_OK;
  const InputArgs a{(const uint4*)q, (const uint4*)k, (uint2*)q8, (uint2*)k8, q_scale, k_scale, q_rows, k_rows, {weights, weights_bf16 != 0, 1.0f}, factor,
                    weight_scaled, (unsigned)q_blocks, (unsigned)k_blocks, eps, pow2, S, ratio, keys, offset, ks, ke};
  if (rotate) indexer_inputs_kernel<true><<<dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream>>>(a);
  else indexer_inputs_kernel<false><<<dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream>>>(a);
  DSA_CHECK_LAUNCH("dsa_indexer_inputs_e4m3");
  return DSA_OK;
}

extern "C" int dsa_indexer_narrow_e4m3(const void* q, int S, int heads, int heads_out, const void* k, int keys, const void* cos, const void* sin,
                                       int positions, void* q8, float* q_scale, void* k8, float* k_scale, const void* weights, int weights_bf16,
                                       float weights_scale, float factor, float* weight_scaled, int64_t offset, int32_t* ks, int32_t* ke,
                                       void* stream) {
  DSA_REQUIRE(S >= 0 && keys >= 0 && heads > 0 && heads <= heads_out && heads_out <= 64, "dsa_indexer_narrow_e4m3: bad sizes");
  DSA_REQUIRE(positions >= S && positions >= keys, "dsa_indexer_narrow_e4m3: cos / sin tables are shorter than the sequence");
  DSA_REQUIRE(((uintptr_t)q % 16) == 0 && ((uintptr_t)k % 16) == 0 && ((uintptr_t)cos % 16) == 0 && ((uintptr_t)sin % 16) == 0 &&
              ((uintptr_t)q8 % 8) == 0 && ((uintptr_t)k8 % 8) == 0, "dsa_indexer_narrow_e4m3: misaligned pointer");
  DSA_REQUIRE((S == 0 && keys == 0) || (cos && sin), "dsa_indexer_narrow_e4m3: null pointer");
  DSA_REQUIRE(S == 0 || (q && q8 && q_scale && weights && weight_scaled && ks && ke), "dsa_indexer_narrow_e4m3: null pointer");
  DSA_REQUIRE(keys == 0 || (k && k8 && k_scale), "dsa_indexer_narrow_e4m3: null pointer");
  const int64_t q_rows = (int64_t)S * heads_out, q_blocks = (q_rows + 15) / 16, k_blocks = (keys + 15) / 16, blocks = q_blocks + k_blocks + dsa_cdiv(S, 256);
  DSA_REQUIRE(q_rows < (1ll << 31), "dsa_indexer_narrow_e4m3: too many rows");
  if (blocks == 0) return DSA_OK;
  const NarrowArgs a{(const uint4*)q, (const uint4*)k, (const uint4*)cos, (const uint4*)sin, heads, heads_out, q_rows, keys, (uint2*)q8, (uint2*)k8,
                     q_scale, k_scale, {weights, weights_bf16 != 0, weights_scale}, factor, weight_scaled, (unsigned)q_blocks, (unsigned)k_blocks, S, offset, ks, ke};
  indexer_narrow_kernel<<<dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream>>>(a);
  DSA_CHECK_LAUNCH("dsa_indexer_narrow_e4m3");
  return DSA_OK;
}

extern "C" int dsa_quant_rowwise_e4m3(const void* x, int64_t rows, int cols, void* x8, float* scale_inv,
                                      float eps, int pow2, void* stream) {
  DSA_REQUIRE(cols == 128, "dsa_quant_rowwise_e4m3: only rows of 128 elements are supported, got %d", cols);
  DSA_REQUIRE(rows >= 0, "dsa_quant_rowwise_e4m3: negative row count");
  DSA_REQUIRE(((uintptr_t)x % 16) == 0 && ((uintptr_t)x8 % 8) == 0, "dsa_quant_rowwise_e4m3: misaligned pointer");
  if (rows == 0) return DSA_OK;
  int64_t blocks = (rows + 15) / 16;
  DSA_REQUIRE(blocks < (1ll << 31), "dsa_quant_rowwise_e4m3: too many rows");
  quant128_kernel<<<dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream>>>(
      (const uint4*)x, (uint2*)x8, scale_inv, rows, eps, pow2, nullptr, 0.f, nullptr);
  DSA_CHECK_LAUNCH("dsa_quant_rowwise_e4m3");
  return DSA_OK;
}

extern "C" int dsa_quant_padded_e4m3(const void* x, int64_t tokens, int heads_in, int dim_in, int heads_out, void* x8, float* scale_inv,
                                     float eps, int pow2, const void* weights, int weights_bf16, float factor, float* weight_scaled,
                                     void* stream) {
  DSA_REQUIRE(tokens >= 0 && heads_in > 0 && heads_in <= heads_out && dim_in > 0 && dim_in <= 128,
              "dsa_quant_padded_e4m3: %d heads of %d elements do not fit %d of 128", heads_in, dim_in, heads_out);
  DSA_REQUIRE(x8 != nullptr && scale_inv != nullptr && (weights == nullptr) == (weight_scaled == nullptr), "dsa_quant_padded_e4m3: null pointer");
  DSA_REQUIRE(((uintptr_t)x8 % 8) == 0, "dsa_quant_padded_e4m3: misaligned pointer");
  const int64_t rows = tokens * heads_out, blocks = (rows + 15) / 16;
  if (rows == 0) return DSA_OK;
  DSA_REQUIRE(blocks < (1ll << 31), "dsa_quant_padded_e4m3: too many rows");
  quant_padded_kernel<<<dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream>>>(
      (const unsigned short*)x, heads_in, dim_in, heads_out, (uint2*)x8, scale_inv, rows, eps, pow2, weights, weights_bf16, factor, weight_scaled);
  DSA_CHECK_LAUNCH("dsa_quant_padded_e4m3");
  return DSA_OK;
}

extern "C" int dsa_quant_rowwise_e4m3_weights(const void* x, int64_t rows, int cols, void* x8, float* scale_inv,
                                              float eps, int pow2, int rotate, const float* weights, float factor,
                                              float* weight_scaled, void* stream) {
  DSA_REQUIRE(cols == 128, "dsa_quant_rowwise_e4m3_weights: only rows of 128 elements are supported, got %d", cols);
  DSA_REQUIRE(rows >= 0, "dsa_quant_rowwise_e4m3_weights: negative row count");
  DSA_REQUIRE(x8 != nullptr && scale_inv != nullptr && weights != nullptr && weight_scaled != nullptr,
              "dsa_quant_rowwise_e4m3_weights: null pointer");
  DSA_REQUIRE(((uintptr_t)x % 16) == 0 && ((uintptr_t)x8 % 8) == 0, "dsa_quant_rowwise_e4m3_weights: misaligned pointer");
  if (rows == 0) return DSA_OK;
  int64_t blocks = (rows + 15) / 16;
  DSA_REQUIRE(blocks < (1ll << 31), "dsa_quant_rowwise_e4m3_weights: too many rows");
  if (rotate)
    rotate_quant128_kernel<<<dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream>>>(
        (const uint4*)x, (uint2*)x8, scale_inv, nullptr, rows, eps, pow2, weights, factor, weight_scaled);
  else
    quant128_kernel<<<dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream>>>(
        (const uint4*)x, (uint2*)x8, scale_inv, rows, eps, pow2, weights, factor, weight_scaled);
  DSA_CHECK_LAUNCH("dsa_quant_rowwise_e4m3_weights");
  return DSA_OK;
}

extern "C" int dsa_indexer_front_e4m3(const void* x, int64_t rows, int cols, int rows_per_token, const float* ln_weight,
                                      const float* ln_bias, float ln_eps, const void* cos, const void* sin,
                                      int cos_sin_f32, int pairing, const int32_t* positions, int batch, int rotate,
                                      void* x8, float* scale_inv, void* y, float eps, int pow2, const float* weights,
                                      float factor, float* weight_scaled, void* stream) {
  DSA_REQUIRE(cols == 128, "dsa_indexer_front_e4m3: only rows of 128 elements are supported, got %d", cols);
  DSA_REQUIRE(rows >= 0 && rows_per_token > 0 && batch > 0, "dsa_indexer_front_e4m3: bad row counts");
  DSA_REQUIRE(pairing >= -1 && pairing <= 1, "dsa_indexer_front_e4m3: pairing must be -1 (no rotary part), 0 or 1");
  DSA_REQUIRE(pairing < 0 || (cos != nullptr && sin != nullptr), "dsa_indexer_front_e4m3: rotary part without cos / sin");
  DSA_REQUIRE((ln_weight == nullptr) == (ln_bias == nullptr), "dsa_indexer_front_e4m3: LayerNorm needs weight and bias");
  DSA_REQUIRE(x8 != nullptr || y != nullptr, "dsa_indexer_front_e4m3: no output requested");
  DSA_REQUIRE(x8 == nullptr || scale_inv != nullptr, "dsa_indexer_front_e4m3: payload without scales");
  DSA_REQUIRE((weights == nullptr) == (weight_scaled == nullptr) && (weights == nullptr || x8 != nullptr),
              "dsa_indexer_front_e4m3: weights and weight_scaled come together, with the payload");
  DSA_REQUIRE(((uintptr_t)x % 16) == 0 && ((uintptr_t)x8 % 8) == 0 && ((uintptr_t)y % 16) == 0 &&
              ((uintptr_t)ln_weight % 16) == 0 && ((uintptr_t)ln_bias % 16) == 0 && ((uintptr_t)cos % 16) == 0 &&
              ((uintptr_t)sin % 16) == 0, "dsa_indexer_front_e4m3: misaligned pointer");
  if (rows == 0) return DSA_OK;
  const int64_t blocks = (rows + 15) / 16;
  DSA_REQUIRE(rows < (1ll << 32), "dsa_indexer_front_e4m3: too many rows");
#define DSA_FRONT_LAUNCH(LN, P) indexer_front128_kernel<LN, P><<<dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream>>>( \
      (const uint4*)x, rows, rows_per_token, ln_weight, ln_bias, ln_eps, cos, sin, cos_sin_f32, positions, batch, rotate, \
      (uint2*)x8, scale_inv, (uint4*)y, eps, pow2, weights, factor, weight_scaled)
  if (ln_weight) {
    if (pairing < 0) DSA_FRONT_LAUNCH(true, -1); else if (pairing == 0) DSA_FRONT_LAUNCH(true, 0); else DSA_FRONT_LAUNCH(true, 1);
  } else {
    if (pairing < 0) DSA_FRONT_LAUNCH(false, -1); else if (pairing == 0) DSA_FRONT_LAUNCH(false, 0); else DSA_FRONT_LAUNCH(false, 1);
  }
#undef DSA_FRONT_LAUNCH
  DSA_CHECK_LAUNCH("dsa_indexer_front_e4m3");
  return DSA_OK;
}

extern "C" int dsa_indexer_fronts_e4m3(const void* q, int S, int heads, const void* k, int keys, const float* ln_weight, const float* ln_bias, float ln_eps,
                                       const void* cos, const void* sin, int cos_sin_f32, int pairing, const int32_t* positions_q,
                                       const int32_t* positions_k, int batch, int rotate, void* q8, float* q_scale, void* k8, float* k_scale,
                                       const void* weights, int weights_bf16, float weights_scale, float factor, float* weight_scaled,
                                       const void* cu, int cu_i64, int ncu, int chunk_offset, int32_t* ks, int32_t* ke, int32_t* total, void* stream) {
  DSA_REQUIRE(S >= 0 && keys >= 0 && heads > 0 && batch > 0 && ncu >= 0, "dsa_indexer_fronts_e4m3: bad sizes");
  DSA_REQUIRE(pairing == 0 || pairing == 1, "dsa_indexer_fronts_e4m3: pairing must be 0 or 1");
  DSA_REQUIRE(cos != nullptr && sin != nullptr && ln_weight != nullptr && ln_bias != nullptr && (cu != nullptr || ncu == 0),
              "dsa_indexer_fronts_e4m3: null pointer");
  DSA_REQUIRE(S == 0 || (q && q8 && q_scale && weights && weight_scaled && ks && ke), "dsa_indexer_fronts_e4m3: null pointer");
  DSA_REQUIRE(keys == 0 || (k && k8 && k_scale), "dsa_indexer_fronts_e4m3: null pointer");
  DSA_REQUIRE(((uintptr_t)q % 16) == 0 && ((uintptr_t)k % 16) == 0 && ((uintptr_t)q8 % 8) == 0 && ((uintptr_t)k8 % 8) == 0 &&
              ((uintptr_t)ln_weight % 16) == 0 && ((uintptr_t)ln_bias % 16) == 0 && ((uintptr_t)cos % 16) == 0 &&
              ((uintptr_t)sin % 16) == 0, "dsa_indexer_fronts_e4m3: misaligned pointer");
  const int64_t q_rows = (int64_t)S * heads, q_blocks = (q_rows + 15) / 16, k_blocks = (keys + 15) / 16;
  DSA_REQUIRE(q_rows < (1ll << 32), "dsa_indexer_fronts_e4m3: too many rows");
  const FrontArgs a{(const uint4*)q, (const uint4*)k, q_rows, keys, heads, ln_weight, ln_bias, ln_eps, cos, sin, cos_sin_f32, positions_q, positions_k, batch,
                    rotate, (uint2*)q8, (uint2*)k8, q_scale, k_scale, {weights, weights_bf16 != 0, weights_scale}, factor, weight_scaled,
                    (unsigned)k_blocks, (unsigned)q_blocks, cu, cu_i64, ncu, S, chunk_offset, ks, ke, total};
  const dim3 grid((unsigned)(k_blocks + q_blocks + dsa_cdiv(S > 0 ? S : 1, 256)));
  if (pairing == 0) indexer_fronts_kernel<0><<<grid, dim3(256), 0, (hipStream_t)stream>>>(a);
  else indexer_fronts_kernel<1><<<grid, dim3(256), 0, (hipStream_t)stream>>>(a);
  DSA_CHECK_LAUNCH("dsa_indexer_fronts_e4m3");
  return DSA_OK;
}
