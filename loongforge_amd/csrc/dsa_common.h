// Shared device/host helpers for the gfx950 DSA kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>

#include "../../include/dsa_hip.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x2 __attribute__((ext_vector_type(2)));

#define LDS_PTR(T, p) ((__attribute__((address_space(3))) T*)(p))

// ---- error plumbing (never throws across the C ABI) ------------------------------------
void dsa_set_error(const char* fmt, ...);
#define DSA_FAIL(code, ...) do { dsa_set_error(__VA_ARGS__); return (code); } while (0)
#define DSA_REQUIRE(cond, ...) do { if (!(cond)) DSA_FAIL(DSA_ERR_BAD_ARG, __VA_ARGS__); } while (0)
#define DSA_CHECK_LAUNCH(name) do { hipError_t e_ = hipGetLastError(); \
    if (e_ != hipSuccess) DSA_FAIL(DSA_ERR_LAUNCH, "%s: launch failed: %s", name, hipGetErrorString(e_)); } while (0)

// hipFuncSetAttribute(fn, MaxDynamicSharedMemorySize, bytes), once per kernel and device while `bytes` does not
// grow: the call costs several microseconds of host time, which a short kernel sequence cannot hide.
hipError_t dsa_reserve_lds(const void* fn, size_t bytes);

// ---- small device helpers ----------------------------------------------------------------
__device__ __forceinline__ float bf16_bits_to_f32(unsigned short h) {
  return __builtin_bit_cast(float, ((unsigned)h) << 16);
}
__device__ __forceinline__ unsigned short f32_to_bf16_bits(float f) {   // round-to-nearest-even
  unsigned u = __builtin_bit_cast(unsigned, f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (unsigned short)((u >> 16) | 0x40);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ unsigned pack_bf16x2(float lo, float hi) {
  return (unsigned)f32_to_bf16_bits(lo) | ((unsigned)f32_to_bf16_bits(hi) << 16);
}
// the same rounding in one instruction (v_cvt_pk_bf16_f32)
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ unsigned cvt_pk_bf16(float lo, float hi) {
  const f32x2_t v = {lo, hi};
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2_t));
}
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
// The value of lane ^ m (m = 1, 2, 4 or 8, a constant after unrolling) by moves inside rows of 16 lanes, which must all be
// active: vector instructions that the consumer mostly absorbs, where a shuffle is a trip through LDS.
__device__ __forceinline__ float xor16(float x, int m) {
  const int i = __builtin_bit_cast(int, x);
  int o;
  if (m == 1) o = __builtin_amdgcn_update_dpp(0, i, 0xb1, 0xf, 0xf, true);              // quad_perm [1, 0, 3, 2]
  else if (m == 2) o = __builtin_amdgcn_update_dpp(0, i, 0x4e, 0xf, 0xf, true);         // quad_perm [2, 3, 0, 1]
  else if (m == 4) o = __builtin_amdgcn_update_dpp(0, __builtin_amdgcn_update_dpp(0, i, 0x141, 0xf, 0xf, true), 0x1b, 0xf, 0xf, true);
  else o = __builtin_amdgcn_update_dpp(0, i, 0x128, 0xf, 0xf, true);                    // row_ror:8 (m = 4: i ^ 7, then i ^ 3)
  return __builtin_bit_cast(float, o);
}
// v_permlane32_swap: the upper half-wave of a trades places with the lower half-wave of b.
__device__ __forceinline__ void swap_halves(unsigned& a, unsigned& b) {
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
}
// A 32 x 32 MFMA accumulator gives lane (r, g = lane / 32) the elements 8j + 4g .. +3 (j = 0..3) of row
// segment r: four 8-byte pieces once rounded to bf16.  The two half-waves trade pieces so that the lane
// ends up with elements 8 (jj + g) .. +7 for jj = 0 and jj = 2: two 16-byte values, o[0] and o[1].
// Every lane of the wave must take part.
__device__ __forceinline__ void acc_row_to_16B(const f32x16& acc, float scale, uint4 (&o)[2]) {
  unsigned pc[4][2];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    pc[j][0] = cvt_pk_bf16(acc[4 * j] * scale, acc[4 * j + 1] * scale);
    pc[j][1] = cvt_pk_bf16(acc[4 * j + 2] * scale, acc[4 * j + 3] * scale);
  }
  // four v_permlane32_swap (swap_halves) that do not depend on one another: one wait in front, one behind
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\tv_permlane32_swap_b32 %2, %3\n\tv_permlane32_swap_b32 %4, %5\n\t"
               "v_permlane32_swap_b32 %6, %7\n\ts_nop 1"
               : "+v"(pc[0][0]), "+v"(pc[1][0]), "+v"(pc[0][1]), "+v"(pc[1][1]), "+v"(pc[2][0]), "+v"(pc[3][0]), "+v"(pc[2][1]),
                 "+v"(pc[3][1]));
  o[0] = make_uint4(pc[0][0], pc[0][1], pc[1][0], pc[1][1]);
  o[1] = make_uint4(pc[2][0], pc[2][1], pc[3][0], pc[3][1]);
}
// Order of work for kernels whose workgroups own a compute unit each: workgroup i -> position among n queries in order of decreasing length.
// Taken strictly in that order the 256 workgroups of the first round have the same length, stay in step from round to round, and all
// read a query's operands at the same time, when nothing else uses the memory, and compute at the same time, when the memory idles.  So
// the first `round` workgroups take every so-many-th of the last `ramp` positions, where a causal window grows from nothing to its
// full length, and those from there on find them out of step; the others follow in order, the shortest again at the end.
__device__ __forceinline__ int spread_start(int i, int n, int round, int ramp) {
  const int tail = min(n, max(ramp, 2 * round)), step = tail / round;
  if (step < 2) return i;
  if (i < round) return n - tail + i * step;
  const int j = i - round - (n - tail);                // >= 0: among the tail's positions that are left
  if (j < 0) return i - round;
  if (j >= round * (step - 1)) return n - tail + round + j;
  return n - tail + j + j / (step - 1) + 1;
}
// Transfers from memory to LDS: each lane fetches 16 bytes at gbase + goff; the wave's 64 chunks land at lds_base + 16 * lane.
// (m0 carries the LDS base; nothing else in these kernels uses m0.)  The transfer is counted by the vector-memory counter but invisible to
// the compiler, which therefore never waits for it: callers wait with DSA_WAIT_VMCNT before a barrier.
// gbase may come straight out of v_readfirstlane, and a memory instruction may read what a vector one wrote into scalar registers only five
// wait states later, which the compiler sees to for its own loads alone.  A scalar move waits for the write by itself, and is also the wait
// state between m0 and the transfer.
#define DSA_LDS_TRANSFER(instruction, hint)                                                                                            \
  unsigned long long base;                                                                                                             \
  asm volatile("s_mov_b32 m0, %1\n\ts_mov_b64 %0, %3\n\t" instruction " %2, %0" hint : "=&s"(base) : "s"(lds_base), "v"(goff), "s"(gbase) : "memory")
__device__ __forceinline__ void dma16(unsigned lds_base, unsigned goff, const void* gbase) { DSA_LDS_TRANSFER("global_load_lds_dwordx4", ""); }
// With the non-temporal hint, for what is read once: it then leaves the L2 to the key rows that neighbouring workgroups share.
// Whole 128-byte lines by eight neighbouring lanes: a line that comes in by parts would be fetched for each.
__device__ __forceinline__ void dma16_once(unsigned lds_base, unsigned goff, const void* gbase) { DSA_LDS_TRANSFER("global_load_lds_dwordx4", " nt"); }
__device__ __forceinline__ void dma4(unsigned lds_base, unsigned goff, const void* gbase) { DSA_LDS_TRANSFER("global_load_lds_dword", ""); }
#undef DSA_LDS_TRANSFER
// s_waitcnt with only the vector-memory counter constrained (gfx9 encoding).
#define DSA_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt((((n) & 0xf) | (((n) >> 4) << 14)) | (0x7 << 4) | (0xf << 8))

static inline int dsa_cdiv(long a, long b) { return (int)((a + b - 1) / b); }
