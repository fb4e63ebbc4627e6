// Head-averaged softmax over the selected slots: target[i,t] = mean_h softmax_t(p_out[i,h,:] * c).
// HBM-bound: reads H*K logits per query once.  One workgroup per query; each wave takes heads
// w, w+4, ...; a head's K logits live in registers, so p_out is read exactly once.  Two variants:
// 16-byte loads when the layout allows it, element loads otherwise (the same arithmetic; the partial
// sums of a head are grouped differently, so results agree to fp32 rounding, not bit for bit).
// exp2 is the bare hardware instruction (the arguments are <= 0; results below 2^-126 flush to zero):
// the library routine's range handling costs four more instructions per logit, and this kernel is
// bound by them.
#include "dsa_common.h"

namespace {

constexpr int MAXV = 64;   // slots per lane: supports K <= 4096

// Where the means go: as they are, or (half) rounded to bf16, which a pass over them behind this kernel took 5.2 us for at 3072 x 512.
struct Target {
  float* full;
  unsigned short* half;
  __device__ __forceinline__ void put(int64_t at, float v) const {
    if (half) half[at] = (unsigned short)cvt_pk_bf16(v, v);
    else full[at] = v;
  }
};

template <bool F32>
__device__ __forceinline__ float load_logit(const void* p, int64_t off) {
  if (F32) return ((const float*)p)[off];
  return bf16_bits_to_f32(((const unsigned short*)p)[off]);
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, o > 8 ? __shfl_xor(v, o, 64) : xor16(v, o));
  return v;
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += o > 8 ? __shfl_xor(v, o, 64) : xor16(v, o);
  return v;
}

template <bool F32, int NV>
__global__ __launch_bounds__(256) void attn_dist_kernel(const void* __restrict__ p_out, int H, int K,
                                                        int64_t ld_s, int64_t ld_h, float c2,
                                                        Target target) {
  extern __shared__ float acc_s[];            // [4 waves][K]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t i = blockIdx.x;
  float acc[NV];
#pragma unroll
  for (int v = 0; v < NV; v++) acc[v] = 0.f;
  for (int h = wave; h < H; h += 4) {
    const int64_t base = i * ld_s + h * ld_h;
    float z[NV];
    float mx = -INFINITY;
#pragma unroll
    for (int v = 0; v < NV; v++) {
      int t = v * 64 + lane;
      z[v] = t < K ? load_logit<F32>(p_out, base + t) * c2 : -INFINITY;
      mx = fmaxf(mx, z[v]);
    }
    mx = wave_max(mx);
    if (mx == -INFINITY) continue;            // head with no valid slot contributes nothing
    float sum = 0.f;
#pragma unroll
    for (int v = 0; v < NV; v++) { z[v] = __builtin_amdgcn_exp2f(z[v] - mx); sum += z[v]; }
    sum = wave_sum(sum);
    float inv = 1.0f / sum;
#pragma unroll
    for (int v = 0; v < NV; v++) acc[v] += z[v] * inv;
  }
#pragma unroll
  for (int v = 0; v < NV; v++) { int t = v * 64 + lane; if (t < K) acc_s[wave * K + t] = acc[v]; }
  __syncthreads();
  const float invh = 1.0f / (float)H;
  for (int t = threadIdx.x; t < K; t += 256)
    target.put(i * K + t, ((acc_s[t] + acc_s[K + t]) + (acc_s[2 * K + t] + acc_s[3 * K + t])) * invh);
}

// The same with 16-byte loads: lane l of a wave owns slots 8 (64 v + l) .. +7 of every head.  Needs
// K, the strides and the base address to be multiples of 8 elements, and a positive scale (the row
// maximum is taken on the raw logits).  Logits beyond the memory-side cache are read with the non-temporal hint
// (STREAMED; [8192, 128, 2048] bf16: 0.79 -> 0.76 ms, 5.7 TB/s; 0.1 - 0.2 GB, still cached from the forward that wrote
// them, read no faster with it).
// LIVE: the ids of the slots are given, and of the 32-slot tiles without a valid one (0 <= id < min(Skv, q_start + i + 1)) the logits
// have not been written.  They are -inf without being read: short documents and prefixes then cost what their slots cost.  With the
// forward that writes them, us: [912, 128, 1024] of five documents 132 + 59 -> 85 + 36, [1091, 128, 2048] 307 + 146 -> 230 + 89, [871, 64,
// 2048] of five 86 + 46 -> 41 + 22, [8192, 128, 2048] 3843 + 756 -> 3758 + 706; full lists the same.
template <bool F32, int NC, bool STREAMED, bool LIVE>
__global__ __launch_bounds__(256) void attn_dist_vec_kernel(const void* __restrict__ p_out, int H, int K,
                                                            int64_t ld_s, int64_t ld_h, float c2,
                                                            Target target, const int* __restrict__ ids, int Skv, int q_start) {
  extern __shared__ float acc_s[];            // [4 waves][K]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t i = blockIdx.x;
  bool has[NC];                               // the lane's slots of chunk v have logits
  int chunks = NC;                            // chunks in front of the last one that any lane has
  if constexpr (LIVE) {
    const int last = min((int64_t)Skv - 1, (int64_t)q_start + i);
    chunks = 0;
    int4 a[NC], b[NC];
#pragma unroll
    for (int v = 0; v < NC; v++) {
      const int t = min(8 * (v * 64 + lane), K - 8);
      a[v] = *(const int4*)(ids + i * K + t);
      b[v] = *(const int4*)(ids + i * K + t + 4);
    }
#pragma unroll
    for (int v = 0; v < NC; v++) {
      const int id[8] = {a[v].x, a[v].y, a[v].z, a[v].w, b[v].x, b[v].y, b[v].z, b[v].w};
      bool any = false;
#pragma unroll
      for (int e = 0; e < 8; e++) any |= id[e] >= 0 && id[e] <= last;
      const unsigned long long m = __ballot(any && 8 * (v * 64 + lane) < K);
      has[v] = (m >> (lane & ~3)) & 0xfull;   // four lanes share a tile
      if (m) chunks = v + 1;
    }
  }
  float acc[NC][8];
#pragma unroll
  for (int v = 0; v < NC; v++)
#pragma unroll
    for (int e = 0; e < 8; e++) acc[v][e] = 0.f;
  // raw 16-byte pieces of one head; the next head's are requested before this head's arithmetic
  auto piece = [&](const void* at) {
    const i32x4 v = STREAMED ? __builtin_nontemporal_load((const i32x4*)at) : *(const i32x4*)at;
    return __builtin_bit_cast(uint4, v);
  };
  struct Raw { uint4 a[NC]; uint4 b[NC]; };
  auto fetch = [&](int h, Raw& r) {
    const int64_t base = i * ld_s + h * ld_h;
#pragma unroll
    for (int v = 0; v < NC; v++) {
      const int t = 8 * (v * 64 + lane);
      if (t < K && h < H && (!LIVE || has[v])) {
        if (F32) {
          r.a[v] = piece((const float*)p_out + base + t);
          r.b[v] = piece((const float*)p_out + base + t + 4);
        } else {
          r.a[v] = piece((const unsigned short*)p_out + base + t);
        }
      }
    }
  };
  // one head: its softmax numerators, their sum, and the accumulation of the normalised values
  auto head = [&](const Raw& cur) {
    float z[NC][8];
    float mx = -INFINITY;
#pragma unroll
    for (int v = 0; v < NC; v++) {
      if (LIVE && v >= chunks) break;
      const int t = 8 * (v * 64 + lane);
      if (t < K && (!LIVE || has[v])) {
        if (F32) {
          const unsigned w[8] = {cur.a[v].x, cur.a[v].y, cur.a[v].z, cur.a[v].w, cur.b[v].x, cur.b[v].y, cur.b[v].z, cur.b[v].w};
#pragma unroll
          for (int e = 0; e < 8; e++) z[v][e] = __builtin_bit_cast(float, w[e]);
        } else {
          const unsigned w[4] = {cur.a[v].x, cur.a[v].y, cur.a[v].z, cur.a[v].w};
#pragma unroll
          for (int e = 0; e < 4; e++) {
            z[v][2 * e] = __builtin_bit_cast(float, w[e] << 16);
            z[v][2 * e + 1] = __builtin_bit_cast(float, w[e] & 0xffff0000u);
          }
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; e++) z[v][e] = -INFINITY;
      }
#pragma unroll
      for (int e = 0; e < 8; e++) mx = fmaxf(mx, z[v][e]);
    }
    mx = wave_max(mx);
    if (mx == -INFINITY) return;              // head with no valid slot contributes nothing
    // the (positive) scale enters through one fused multiply-add per logit: exp2(z c2 - max(z) c2)
    const float off = -mx * c2;
    float sum = 0.f;
#pragma unroll
    for (int v = 0; v < NC; v++) {
      if (LIVE && v >= chunks) break;
#pragma unroll
      for (int e = 0; e < 8; e++) { z[v][e] = __builtin_amdgcn_exp2f(fmaf(z[v][e], c2, off)); sum += z[v][e]; }
    }
    sum = wave_sum(sum);
    const float inv = 1.0f / sum;
#pragma unroll
    for (int v = 0; v < NC; v++) {
      if (LIVE && v >= chunks) break;
#pragma unroll
      for (int e = 0; e < 8; e++) acc[v][e] += z[v][e] * inv;
    }
  };
  // two buffers take turns (no register copies): while one head is worked on, the next is on its way
  Raw r0, r1;
  fetch(wave, r0);
  for (int h = wave; h < H; h += 8) {
    fetch(h + 4, r1);
    head(r0);
    if (h + 4 < H) {
      fetch(h + 8, r0);
      head(r1);
    }
  }
#pragma unroll
  for (int v = 0; v < NC; v++) {
    const int t = 8 * (v * 64 + lane);
    if (t < K) {
      *(f32x4*)(acc_s + wave * K + t) = f32x4{acc[v][0], acc[v][1], acc[v][2], acc[v][3]};
      *(f32x4*)(acc_s + wave * K + t + 4) = f32x4{acc[v][4], acc[v][5], acc[v][6], acc[v][7]};
    }
  }
  __syncthreads();
  const float invh = 1.0f / (float)H;
  for (int t = threadIdx.x; t < K; t += 256)
    target.put(i * K + t, ((acc_s[t] + acc_s[K + t]) + (acc_s[2 * K + t] + acc_s[3 * K + t])) * invh);
}

// Up to 512 slots: a wave works four heads at a time (up to 256 slots eight, two of them side by side in its half-waves), whose maxima
// and sums are reduced together: two steps leave each row of 16 lanes with one head, four more finish all four, where six for each head
// by itself cost as much as the exponentials.  The sums' reciprocals are divided once for four heads.  Issue-bound like the kernel above.
// A lane of a half-wave owns 8 consecutive slots.
// us, that kernel and this: 2077 queries x 64 heads x 512 slots 31 and 26.5, 8192 x 128 x 512 197 and 182 (5.9 TB/s), 7951 x 32 x 256
// 50 and 25, 1192 x 64 x 256 21.0 and 10.8, 1024 x 16 x 256 6.4 and 5.0.
__device__ __forceinline__ void trade_halves(float& x, float& y) {       // the upper half-wave of x against the lower one of y
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(x), "+v"(y));
}
__device__ __forceinline__ void trade_rows(float& x, float& y) {         // rows of 16 lanes 1 and 3 of x against rows 0 and 2 of y
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(x), "+v"(y));
}
// f over the lanes of a wave (HALVES: of each half-wave) for v[0 .. 3]; v[j] comes back in every lane that it is over.
template <bool HALVES, class F, class G>
__device__ __forceinline__ void fold4(float (&v)[4], F f, G last) {
  float a, b;
  if (!HALVES) {                             // row 2 i + k of 16 lanes ends with head 2 k + i
    trade_halves(v[0], v[1]);
    a = f(v[0], v[1]);                       // the lower half-wave has head 0, the upper one head 1
    trade_halves(v[2], v[3]);
    b = f(v[2], v[3]);
    trade_rows(a, b);
    a = f(a, b);
#pragma unroll
    for (int m = 1; m < 16; m <<= 1) a = f(a, xor16(a, m));
    a = last(a);
#pragma unroll
    for (int j = 0; j < 4; j++)
      v[j] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, a), 32 * (j & 1) + 16 * (j >> 1)));
  } else {                                   // rows 0 and 2 end with v[0] (v[2]) of the half-wave, rows 1 and 3 with v[1] (v[3])
    trade_rows(v[0], v[1]);
    a = f(v[0], v[1]);
    trade_rows(v[2], v[3]);
    b = f(v[2], v[3]);
#pragma unroll
    for (int m = 1; m < 16; m <<= 1) { a = f(a, xor16(a, m)); b = f(b, xor16(b, m)); }
    a = last(a);
    b = last(b);
    v[0] = v[1] = a;
    trade_rows(v[0], v[1]);                  // v[0]: rows 0, 0, 2, 2; v[1]: rows 1, 1, 3, 3
    v[2] = v[3] = b;
    trade_rows(v[2], v[3]);
  }
}

template <bool HALVES, bool STREAMED, bool LIVE>
__global__ __launch_bounds__(256) void attn_dist_few_kernel(const unsigned short* __restrict__ p_out, int H, int K, int64_t ld_s, int64_t ld_h, float c2,
                                                            Target target, const int* __restrict__ ids, int Skv, int q_start) {
  extern __shared__ float acc_s[];           // [4 waves][2 half-waves if HALVES][K]
  constexpr int SIDE = HALVES ? 2 : 1;       // heads side by side
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, side = HALVES ? lane >> 5 : 0;
  const int t = 8 * (HALVES ? lane & 31 : lane);
  const int64_t i = blockIdx.x;
  bool has = t < K;
  if constexpr (LIVE) {
    const int last = (int)min((int64_t)Skv - 1, (int64_t)q_start + i);
    const int at = min(t, K - 8);
    const int4 a = *(const int4*)(ids + i * K + at), b = *(const int4*)(ids + i * K + at + 4);
    const int id[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    bool any = false;
#pragma unroll
    for (int e = 0; e < 8; e++) any |= id[e] >= 0 && id[e] <= last;
    const unsigned long long m = __ballot(any && t < K);
    has = (m >> (lane & ~3)) & 0xfull;       // four lanes share a tile
  }
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; e++) acc[e] = 0.f;
  struct Raw { uint4 x[4]; };
  auto fetch = [&](int h0, Raw& r) {         // heads h0 + SIDE j + side; those beyond the last one as the last one, without weight
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const i32x4* at = (const i32x4*)(p_out + i * ld_s + min(h0 + SIDE * j + side, H - 1) * ld_h + t);
      if (has) r.x[j] = __builtin_bit_cast(uint4, STREAMED ? __builtin_nontemporal_load(at) : *at);
    }
  };
  auto heads = [&](int h0, const Raw& r) {
    float z[4][8], m[4], s[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const unsigned w[4] = {r.x[j].x, r.x[j].y, r.x[j].z, r.x[j].w};
#pragma unroll
      for (int e = 0; e < 4; e++) {
        z[j][2 * e] = __builtin_bit_cast(float, w[e] << 16);
        z[j][2 * e + 1] = __builtin_bit_cast(float, w[e] & 0xffff0000u);
      }
      m[j] = z[j][0];
#pragma unroll
      for (int e = 1; e < 8; e++) m[j] = fmaxf(m[j], z[j][e]);
    }
    fold4<HALVES>(m, [](float x, float y) { return fmaxf(x, y); }, [](float x) { return x; });
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const float off = -m[j] * c2;          // (a head with no valid slot contributes nothing below)
      s[j] = 0.f;
#pragma unroll
      for (int e = 0; e < 8; e++) { z[j][e] = __builtin_amdgcn_exp2f(fmaf(z[j][e], c2, off)); s[j] += z[j][e]; }
    }
    fold4<HALVES>(s, [](float x, float y) { return x + y; }, [](float x) { return 1.0f / x; });
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const bool in = h0 + SIDE * j + side < H && m[j] != -INFINITY;
      if (__ballot(!in) == 0ull) {
#pragma unroll
        for (int e = 0; e < 8; e++) acc[e] += z[j][e] * s[j];
      } else if (in) {
#pragma unroll
        for (int e = 0; e < 8; e++) acc[e] += z[j][e] * s[j];
      }
    }
  };
  Raw r0, r1;
#pragma unroll
  for (int j = 0; j < 4; j++) r0.x[j] = r1.x[j] = make_uint4(0xff80ff80u, 0xff80ff80u, 0xff80ff80u, 0xff80ff80u);      // -inf where nothing is read
  constexpr int STEP = 4 * SIDE;             // heads of a wave at a time
  fetch(STEP * wave, r0);
  for (int h = STEP * wave; h < H; h += 8 * STEP) {
    fetch(h + 4 * STEP, r1);
    heads(h, r0);
    if (h + 4 * STEP < H) {
      fetch(h + 8 * STEP, r0);
      heads(h + 4 * STEP, r1);
    }
  }
  if (t < K) {
    float* const own = acc_s + (wave * SIDE + side) * K + t;
    *(f32x4*)own = f32x4{acc[0], acc[1], acc[2], acc[3]};
    *(f32x4*)(own + 4) = f32x4{acc[4], acc[5], acc[6], acc[7]};
  }
  __syncthreads();
  const float invh = 1.0f / (float)H;
  for (int t = threadIdx.x; t < K; t += 256) {
    float part[SIDE];
#pragma unroll
    for (int k = 0; k < SIDE; k++) {
      const float* const a = acc_s + 4 * k * K + t;
      part[k] = (a[0] + a[K]) + (a[2 * K] + a[3 * K]);
    }
    target.put(i * K + t, (HALVES ? part[0] + part[SIDE - 1] : part[0]) * invh);
  }
}

// ids: null, or those whose dead tiles have no logits
template <bool F32>
int launch(const void* p_out, int S, int H, int K, int64_t ld_s, int64_t ld_h, float sm_scale, Target target, const int* ids, int Skv,
           int q_start, hipStream_t st) {
  const float c2 = sm_scale * 1.4426950408889634f;
  size_t smem = (size_t)4 * K * sizeof(float);
  const bool vec = K % 8 == 0 && ld_s % 8 == 0 && ld_h % 8 == 0 && ((uintptr_t)p_out % 32) == 0 && c2 > 0.f;
  if (vec) {
    const int nc = (K + 511) / 512;
    const bool streamed = (int64_t)S * H * K * (F32 ? 4 : 2) > (256ll << 20);
    if constexpr (!F32) {
      if (nc == 1 && H >= 8) {               // fewer heads: a wave's four would be one and its copies
        const bool halves = K <= 256;
        if (halves) smem *= 2;
#define DSA_FEW_LAUNCH(HV, STR, LIVE) \
        attn_dist_few_kernel<HV, STR, LIVE><<<dim3(S), dim3(256), smem, st>>>((const unsigned short*)p_out, H, K, ld_s, ld_h, c2, target, ids, Skv, q_start)
#define DSA_FEW_CASE(HV) \
        if (ids) { if (streamed) DSA_FEW_LAUNCH(HV, true, true); else DSA_FEW_LAUNCH(HV, false, true); } \
        else if (streamed) DSA_FEW_LAUNCH(HV, true, false); else DSA_FEW_LAUNCH(HV, false, false)
        if (halves) { DSA_FEW_CASE(true); } else { DSA_FEW_CASE(false); }
#undef DSA_FEW_CASE
#undef DSA_FEW_LAUNCH
        return 0;
      }
    }
#define DSA_ADV_LAUNCH(N, STR, LIVE) \
    attn_dist_vec_kernel<F32, N, STR, LIVE><<<dim3(S), dim3(256), smem, st>>>(p_out, H, K, ld_s, ld_h, c2, target, ids, Skv, q_start)
#define DSA_ADV_CASE(N) \
    if (nc <= N) { \
      if constexpr (!F32) { \
        if (ids) { \
          if (streamed) DSA_ADV_LAUNCH(N, true, true); else DSA_ADV_LAUNCH(N, false, true); \
          return 0; \
        } \
      } \
      if (streamed) DSA_ADV_LAUNCH(N, true, false); else DSA_ADV_LAUNCH(N, false, false); \
      return 0; \
    }
    DSA_ADV_CASE(1) DSA_ADV_CASE(2) DSA_ADV_CASE(4) DSA_ADV_CASE(8)
#undef DSA_ADV_CASE
#undef DSA_ADV_LAUNCH
  }
  if (ids) return -1;
  int nv = (K + 63) / 64;
#define DSA_AD_CASE(N) \
  if (nv <= N) { attn_dist_kernel<F32, N><<<dim3(S), dim3(256), smem, st>>>(p_out, H, K, ld_s, ld_h, c2, target); return 0; }
  DSA_AD_CASE(1) DSA_AD_CASE(2) DSA_AD_CASE(4) DSA_AD_CASE(8) DSA_AD_CASE(16) DSA_AD_CASE(32) DSA_AD_CASE(64)
#undef DSA_AD_CASE
  return -1;
}

}  // namespace

extern "C" int dsa_attn_dist_as(const void* p_out, int p_out_f32, int S, int H, int K, int64_t ld_s, int64_t ld_h,
                                float sm_scale, void* target, int target_bf16, void* stream) {
  DSA_REQUIRE(S >= 0 && H > 0 && K > 0, "dsa_attn_dist: bad shape S=%d H=%d K=%d", S, H, K);
  DSA_REQUIRE(K <= 64 * MAXV, "dsa_attn_dist: K=%d exceeds the supported maximum %d", K, 64 * MAXV);
  DSA_REQUIRE(ld_h >= K && ld_s >= ld_h, "dsa_attn_dist: bad strides");
  if (S == 0) return DSA_OK;
  const Target to{target_bf16 ? nullptr : (float*)target, target_bf16 ? (unsigned short*)target : nullptr};
  int rc = p_out_f32 ? launch<true>(p_out, S, H, K, ld_s, ld_h, sm_scale, to, nullptr, 0, 0, (hipStream_t)stream)
                     : launch<false>(p_out, S, H, K, ld_s, ld_h, sm_scale, to, nullptr, 0, 0, (hipStream_t)stream);
  DSA_REQUIRE(rc == 0, "dsa_attn_dist: unsupported K");
  DSA_CHECK_LAUNCH("dsa_attn_dist");
  return DSA_OK;
}
extern "C" int dsa_attn_dist(const void* p_out, int p_out_f32, int S, int H, int K, int64_t ld_s, int64_t ld_h,
                             float sm_scale, float* target, void* stream) {
  return dsa_attn_dist_as(p_out, p_out_f32, S, H, K, ld_s, ld_h, sm_scale, target, 0, stream);
}

// Of logits [S, heads of ld_s / K, K] whose tiles without a valid slot have not been written (K % 64 == 0, 32-byte aligned, sm_scale > 0)
int dsa_attn_dist_live(const void* logits, const int32_t* ids, int S, int H, int Skv, int K, int64_t ld_s, int q_start, float sm_scale,
                       float* target, hipStream_t st) {
  return launch<false>(logits, S, H, K, ld_s, K, sm_scale, Target{target, nullptr}, ids, Skv, q_start, st);
}
