// Rotation of four rotary pairs of one row, shared by the rotary kernels and the absorption kernels.
#pragma once
#include "dsa_common.h"

namespace rope {

constexpr int ADJ = 0, SPLIT = 1;      // where pair i sits in a row: elements (2i, 2i + 1) or (i, i + emb / 2)

// four consecutive elements of a bf16 or fp32 row (by value: arrays filled under a branch end up in memory)
__device__ __forceinline__ f32x4 load4(const void* base, long idx, int f32) {
  if (f32) return *(const f32x4*)((const float*)base + idx);
  const uint2 v = *(const uint2*)((const unsigned short*)base + idx);
  return f32x4{__builtin_bit_cast(float, v.x << 16), __builtin_bit_cast(float, v.x & 0xffff0000u),
               __builtin_bit_cast(float, v.y << 16), __builtin_bit_cast(float, v.y & 0xffff0000u)};
}

// Four pairs at a time: their values (a, b) in a row, the tables' entries, the rotation
//   y.a = a c1 - b s1, y.b = b c2 + a s2, or its transpose (fp32, products and sums separate IEEE operations),
// and the way back with one rounding to bf16.
struct Quad { f32x4 a, b; };
struct QuadTables { f32x4 c1, c2, s1, s2; };

__device__ __forceinline__ Quad adjacent_pairs(const uint4& v) {
  const unsigned w[4] = {v.x, v.y, v.z, v.w};
  Quad x;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    x.a[k] = __builtin_bit_cast(float, w[k] << 16);
    x.b[k] = __builtin_bit_cast(float, w[k] & 0xffff0000u);
  }
  return x;
}

template <int PAIRING>
__device__ __forceinline__ Quad load_quad(const unsigned short* src, int q, int emb) {
  if (PAIRING == ADJ) return adjacent_pairs(*(const uint4*)(src + 8 * q));
  return Quad{load4(src, 4 * q, 0), load4(src, (emb >> 1) + 4 * q, 0)};
}

template <int PAIRING>   // of the rotated side: destination forward, source in the transpose
__device__ __forceinline__ QuadTables load_tables(const void* cos, const void* sin, int f32, long pos, int q, int emb) {
  const long row = pos * emb;
  if (PAIRING == ADJ) {
    const f32x4 ca = load4(cos, row + 8 * q, f32), cb = load4(cos, row + 8 * q + 4, f32);
    const f32x4 sa = load4(sin, row + 8 * q, f32), sb = load4(sin, row + 8 * q + 4, f32);
    return QuadTables{__builtin_shufflevector(ca, cb, 0, 2, 4, 6), __builtin_shufflevector(ca, cb, 1, 3, 5, 7),
                      __builtin_shufflevector(sa, sb, 0, 2, 4, 6), __builtin_shufflevector(sa, sb, 1, 3, 5, 7)};
  }
  const int half = emb >> 1;
  return QuadTables{load4(cos, row + 4 * q, f32), load4(cos, row + half + 4 * q, f32), load4(sin, row + 4 * q, f32),
                    load4(sin, row + half + 4 * q, f32)};
}

template <bool INVERSE>
__device__ __forceinline__ Quad rotate(const Quad& x, const QuadTables& t) {
#pragma clang fp contract(off)
  Quad y;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    if (!INVERSE) {
      y.a[k] = x.a[k] * t.c1[k] - x.b[k] * t.s1[k];
      y.b[k] = x.b[k] * t.c2[k] + x.a[k] * t.s2[k];
    } else {
      y.a[k] = x.a[k] * t.c1[k] + x.b[k] * t.s2[k];
      y.b[k] = (-x.a[k]) * t.s1[k] + x.b[k] * t.c2[k];
    }
  }
  return y;
}

template <int PAIRING>
__device__ __forceinline__ void store_quad(const Quad& y, unsigned short* dst, int q, int emb) {
  if (PAIRING == ADJ) {
    *(uint4*)(dst + 8 * q) = make_uint4(cvt_pk_bf16(y.a[0], y.b[0]), cvt_pk_bf16(y.a[1], y.b[1]),
                                        cvt_pk_bf16(y.a[2], y.b[2]), cvt_pk_bf16(y.a[3], y.b[3]));
  } else {
    *(uint2*)(dst + 4 * q) = make_uint2(cvt_pk_bf16(y.a[0], y.a[1]), cvt_pk_bf16(y.a[2], y.a[3]));
    *(uint2*)(dst + (emb >> 1) + 4 * q) = make_uint2(cvt_pk_bf16(y.b[0], y.b[1]), cvt_pk_bf16(y.b[2], y.b[3]));
  }
}

template <int IN, int OUT, bool INVERSE>
__device__ __forceinline__ void rotate_quad(const unsigned short* src, unsigned short* dst, int q, int emb, long pos, const void* cos,
                                            const void* sin, int f32) {
  const Quad x = load_quad<IN>(src, q, emb);
  const QuadTables t = load_tables<INVERSE ? IN : OUT>(cos, sin, f32, pos, q, emb);
  store_quad<OUT>(rotate<INVERSE>(x, t), dst, q, emb);
}

}  // namespace rope
