// Small kernels of the indexer's front end where it runs as separate operations: rotary angles and tables, the rotary embedding
// with the rounding of its bf16 tensor operations, the Hadamard rotation of any power-of-two width.  Each takes the place of
// 4 - 10 elementwise launches of a few microseconds; all are bound by their launch at the sizes that take this way.
#include "dsa_common.h"

namespace {

__device__ __forceinline__ float bf(float x) { return bf16_bits_to_f32(f32_to_bf16_bits(x)); }

// angle[i][c] = (i + offset) * inv_freq[c % half] or its cosine and sine; c < 2 half
template <int WHAT>   // 0 angles, 1 cos / sin in fp32, 2 in bf16
__global__ __launch_bounds__(256) void rotary_table_kernel(const float* __restrict__ inv_freq, int half, int n, float offset, void* __restrict__ a,
                                                           void* __restrict__ b) {
  const long e = (long)blockIdx.x * 256 + threadIdx.x;
  if (e >= (long)n * half) return;
  const int i = (int)(e / half), c = (int)(e % half);
  const float ang = ((float)i + offset) * inv_freq[c];
  const long o = (long)i * 2 * half + c;
  if (WHAT == 0) {
    ((float*)a)[o] = ang;
    ((float*)a)[o + half] = ang;
    return;
  }
  const float cs = cosf(ang), sn = sinf(ang);
  if (WHAT == 1) {
    ((float*)a)[o] = cs; ((float*)a)[o + half] = cs;
    ((float*)b)[o] = sn; ((float*)b)[o + half] = sn;
  } else {
    const unsigned short cb = f32_to_bf16_bits(cs), sb = f32_to_bf16_bits(sn);
    ((unsigned short*)a)[o] = cb; ((unsigned short*)a)[o + half] = cb;
    ((unsigned short*)b)[o] = sb; ((unsigned short*)b)[o + half] = sb;
  }
}

// y = t cos + rotate_half(t) sin over rows [token, head][d], every product and the sum rounded to bf16 (cos and sin as well) as the
// separate operations round; the transpose of that for gradients.  `interleaved`: the pairs of t are adjacent elements (they
// leave split into halves).  token t takes angle row t / batch.
template <bool TRANSPOSE>
__global__ __launch_bounds__(256) void rope_steps_kernel(const unsigned short* __restrict__ x, long x_tok, long x_head, unsigned short* __restrict__ y,
                                                         long y_tok, long y_head, const float* __restrict__ angles, float mscale, int interleaved,
                                                         int batch, long rows, int heads, int half) {
#pragma clang fp contract(off)
  const long e = (long)blockIdx.x * 256 + threadIdx.x;
  if (e >= rows * heads * half) return;
  const int i = (int)(e % half);
  const long rh = e / half, h = rh % heads, t = rh / heads;
  const float* ang = angles + (t / batch) * 2 * half;
  const float c1 = bf(cosf(ang[i]) * mscale), s1 = bf(sinf(ang[i]) * mscale);
  const float c2 = bf(cosf(ang[i + half]) * mscale), s2 = bf(sinf(ang[i + half]) * mscale);
  const long in1 = !TRANSPOSE && interleaved ? 2 * i : i, in2 = !TRANSPOSE && interleaved ? 2 * i + 1 : i + half;
  const long out1 = TRANSPOSE && interleaved ? 2 * i : i, out2 = TRANSPOSE && interleaved ? 2 * i + 1 : i + half;
  const unsigned short* xp = x + t * x_tok + h * x_head;
  const float a = bf16_bits_to_f32(xp[in1]), b = bf16_bits_to_f32(xp[in2]);
  float ya, yb;
  if (!TRANSPOSE) {
    ya = bf(a * c1) + bf(-b * s1);
    yb = bf(b * c2) + bf(a * s2);
  } else {
    ya = bf(a * c1) + bf(b * s2);
    yb = bf(b * c2) + -bf(a * s1);
  }
  unsigned short* yp = y + t * y_tok + h * y_head;
  yp[out1] = f32_to_bf16_bits(ya);
  yp[out2] = f32_to_bf16_bits(yb);
}

// rows of N elements through the Hadamard butterfly (Sylvester order, fp32), times N^-0.5, rounded to bf16: 8 elements per lane
template <int N>
__global__ __launch_bounds__(256) void hadamard_kernel(const uint4* __restrict__ x, uint4* __restrict__ y, long rows, float scale) {
  constexpr int LANES = N / 8;
  const long row = (long)blockIdx.x * (256 / LANES) + threadIdx.x / LANES;
  const int sub = threadIdx.x % LANES;
  const bool live = row < rows;
  const uint4 raw = live ? x[row * LANES + sub] : make_uint4(0, 0, 0, 0);
  const unsigned w[4] = {raw.x, raw.y, raw.z, raw.w};
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
  for (int m = 1; m < LANES; m <<= 1)
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const float o = __shfl_xor(v[i], m, 64);
      v[i] = (sub & m) ? o - v[i] : v[i] + o;
    }
  unsigned o[4];
#pragma unroll
  for (int i = 0; i < 4; i++)
    o[i] = (unsigned)f32_to_bf16_bits(v[2 * i] * scale) | ((unsigned)f32_to_bf16_bits(v[2 * i + 1] * scale) << 16);
  if (live) y[row * LANES + sub] = make_uint4(o[0], o[1], o[2], o[3]);
}

}  // namespace

extern "C" int dsa_rotary_tables(const float* inv_freq, int half, int n, float offset, int what, void* a, void* b, void* stream) {
  DSA_REQUIRE(half > 0 && n >= 0 && what >= 0 && what <= 2, "dsa_rotary_tables: bad sizes");
  DSA_REQUIRE(inv_freq != nullptr && (n == 0 || (a != nullptr && (what == 0 || b != nullptr))), "dsa_rotary_tables: null pointer");
  if (n == 0) return DSA_OK;
  const dim3 grid(dsa_cdiv((long)n * half, 256));
  hipStream_t st = (hipStream_t)stream;
  if (what == 0) rotary_table_kernel<0><<<grid, 256, 0, st>>>(inv_freq, half, n, offset, a, b);
  else if (what == 1) rotary_table_kernel<1><<<grid, 256, 0, st>>>(inv_freq, half, n, offset, a, b);
  else rotary_table_kernel<2><<<grid, 256, 0, st>>>(inv_freq, half, n, offset, a, b);
  DSA_CHECK_LAUNCH("dsa_rotary_tables");
  return DSA_OK;
}

extern "C" int dsa_rope_steps(const void* x, int64_t x_tok, int64_t x_head, void* y, int64_t y_tok, int64_t y_head, const float* angles,
                              float mscale, int interleaved, int batch, int64_t rows, int heads, int d, int transpose, void* stream) {
  DSA_REQUIRE(rows >= 0 && heads > 0 && d > 0 && d % 2 == 0 && batch > 0, "dsa_rope_steps: bad sizes");
  if (rows == 0) return DSA_OK;
  const int64_t n = rows * heads * (d / 2);
  DSA_REQUIRE(n < (1ll << 38), "dsa_rope_steps: too many rows");
  const dim3 grid((unsigned)((n + 255) / 256));
  if (transpose)
    rope_steps_kernel<true><<<grid, 256, 0, (hipStream_t)stream>>>((const unsigned short*)x, x_tok, x_head, (unsigned short*)y, y_tok, y_head, angles,
                                                                   mscale, interleaved, batch, rows, heads, d / 2);
  else
    rope_steps_kernel<false><<<grid, 256, 0, (hipStream_t)stream>>>((const unsigned short*)x, x_tok, x_head, (unsigned short*)y, y_tok, y_head, angles,
                                                                    mscale, interleaved, batch, rows, heads, d / 2);
  DSA_CHECK_LAUNCH("dsa_rope_steps");
  return DSA_OK;
}

extern "C" int dsa_hadamard(const void* x, void* y, int64_t rows, int n, void* stream) {
  DSA_REQUIRE(n == 32 || n == 64 || n == 128 || n == 256 || n == 512, "dsa_hadamard: rows of 32, 64, 128, 256 or 512 elements, got %d", n);
  DSA_REQUIRE(rows >= 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)y % 16) == 0, "dsa_hadamard: misaligned pointer");
  if (rows == 0) return DSA_OK;
  const int64_t blocks = (rows * (n / 8) + 255) / 256;
  DSA_REQUIRE(blocks < (1ll << 31), "dsa_hadamard: too many rows");
  const dim3 grid((unsigned)blocks);
  const float scale = n == 32 ? 0.17677669529663687f : n == 64 ? 0.125f : n == 128 ? 0.08838834764831845f : n == 256 ? 0.0625f : 0.04419417382415922f;
  hipStream_t st = (hipStream_t)stream;
#define DSA_HADAMARD(N) hadamard_kernel<N><<<grid, 256, 0, st>>>((const uint4*)x, (uint4*)y, rows, scale)
  if (n == 32) DSA_HADAMARD(32); else if (n == 64) DSA_HADAMARD(64); else if (n == 128) DSA_HADAMARD(128);
  else if (n == 256) DSA_HADAMARD(256); else DSA_HADAMARD(512);
#undef DSA_HADAMARD
  DSA_CHECK_LAUNCH("dsa_hadamard");
  return DSA_OK;
}
