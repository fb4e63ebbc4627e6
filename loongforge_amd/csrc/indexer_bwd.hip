// Sparse backward of the lightning-indexer logits for gfx950, deterministic.
//
// For every selected pair (query i, slot t, key j = ids[i,t]) with upstream gradient g[i,t]:
//   r_h = q8[i,h,:] . k8[j,:]            a = g[i,t] * k_scale[j]          m_h = [r_h > 0]
//   d_qw[i,h]   += a * relu(r_h)
//   d_q8[i,h,:] += q_w[i,h] * (a m_h) * k8[j,:]
//   d_k8[j,:]   += a * sum_h m_h * (q_w[i,h] q8[i,h,:])
// The weight of a head and the factor of a pair stand outside the sums they do not depend on, so that what passes from
// the first product to the other two is a mask.
//
// One workgroup of eight waves per query, 128 slots per tile; the waves p and p + 4 (one SIMD) share 32 slots:
//   r        fp8 MFMA, in both waves: with the keys on the columns in wave p, with the heads on the columns in wave p + 4.
//            The accumulator layout of each is the operand layout of the wave's second product, so nothing is
//            transposed through LDS
//   d_k8 row wave p, bf16 MFMA  row^T[d, key] = (q_w Q)^T[d, head] . m[head, key], times a in fp32; the row, rounded to
//            bf16, goes to a pair buffer at the position of a key-sorted order and a second kernel sums every key's
//            rows in fp32 in ascending query order
//   d_q8     wave p + 4, bf16 MFMA  dq^T[d, head] += K^T[d, key] . (a m)[key, head]; K^T by transposing 8-bit LDS reads of the fp8 tile,
//            converted in registers (exact); a as a bf16 pair (hi + lo), so the products lose nothing visible in fp32
// No floating-point atomics: every sum has a fixed order.
// Where queries select a good part of the keys that they see, d_k8 comes from other kernels (by key tiles, below) and all waves here
// sum d_q8.
//
// With rows, at 8192 queries x 2048 slots x 64 heads (whose causal windows go by key tiles), 1.2 - 1.5 ms, and 0.59 for the rows' sums:
// 0.85 for the loop without its row stores (2048 matrix cycles of 3600 per tile and SIMD), most of the rest for the 3.8 GB of rows
// (4.4 TB/s where the row waves run alone).  By key tiles 0.60 + 0.12 + 0.81 + 0.03.  The queries'
// set-up and final sums run alone on their compute unit.  With the slots behind the query's rows, the first transfers behind the keys'
// scales and weights, scales and angles of the final steps out of memory it took 1.45 ms (2077 x 512 x 32 heads 107 us and now 88,
// 3072 x 512 compressed keys x 64 heads 169 and 147).  (2.54 ms for four waves, one per SIMD, that carried m a q_w through LDS as a bf16 pair: 48 transposing
// reads and 40 writes per wave and tile.)  Rows written in slot order instead of scattered: the same; non-temporal: 2.9 ms.
#include "dsa_common.h"
#include "order.h"
#include <type_traits>

namespace {

constexpr int D = 128;
constexpr int TK = 128;                 // slots per tile of the waves that share them (a list's length is a multiple of it)
constexpr int WAVE_BYTES = 32 * D;      // fp8 key rows of a wave's share of a tile
constexpr int THREADS = 512;
constexpr int RED_STRIDE = 132;         // floats per head row of the cross-wave reduction buffers

// The 16-byte chunk c of a 128-byte row r sits in slot c ^ slot_xor(r): eight rows of one parity of any 16 consecutive ones
// use eight different slots (row reads), and the eight rows of a transposing read four different pairs of slots per
// parity: neither kind of read has a bank conflict.
__device__ __forceinline__ int slot_xor(int r) { return ((r >> 2) & 1) | (r & 2) | ((r >> 1) & 4); }

// e4m3 bytes -> bf16 (exact)
__device__ __forceinline__ bf16x8 fp8_to_bf16(const i32x2& w) {
  bf16x8 o;
#pragma unroll
  for (int x = 0; x < 2; x++) {
    const bf16x2 lo = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[x], 1.0f, false);
    const bf16x2 hi = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[x], 1.0f, true);
    o[4 * x] = lo[0]; o[4 * x + 1] = lo[1]; o[4 * x + 2] = hi[0]; o[4 * x + 3] = hi[1];
  }
  return o;
}
typedef _Float16 __attribute__((ext_vector_type(2))) f16x2;
typedef unsigned short __attribute__((ext_vector_type(2))) u16x2;
// LDS by 32-bit address: sums of a lane's offset, a tile's and a constant then stay in the read's own offset field
template <typename T>
__device__ __forceinline__ T lds_read(unsigned addr) { return *(__attribute__((address_space(3))) const T*)(uintptr_t)addr; }
__device__ __forceinline__ i32x2 read_tr8(unsigned addr) {
  return __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) i32x2*)(uintptr_t)addr);
}

// The (q_w Q)^T operand of d-tile dt and k-step kk: lane = d row 32 dt + r, heads 16 kk + 4 g .. and 16 kk + 8 + 4 g .. (the order in
// which an accumulator of scores holds them); the query's fp8 rows lie in LDS with their chunks at c ^ slot_xor(row).
__device__ __forceinline__ uint4 weighted_query(unsigned q_lds, const float* w_s, int lane, int dt, int kk) {
  const int g = lane >> 5, blk = lane >> 4, ii = lane & 15;
  const f32x4 w0 = *(const f32x4*)(w_s + 16 * kk + 4 * g), w1 = *(const f32x4*)(w_s + 16 * kk + 8 + 4 * g);
  const int row = 16 * kk + 8 * (ii >> 3) + 4 * g + ((ii >> 1) & 3);
  const bf16x8 x = fp8_to_bf16(read_tr8(q_lds + row * D + (((2 * dt + (blk & 1)) ^ slot_xor(row)) << 4) + 8 * (ii & 1)));
  unsigned pk[4];
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const f32x4& w = e < 2 ? w0 : w1;
    pk[e] = cvt_pk_bf16((float)x[2 * e] * w[(2 * e) & 3], (float)x[2 * e + 1] * w[(2 * e + 1) & 3]);
  }
  return make_uint4(pk[0], pk[1], pk[2], pk[3]);
}
// The mask [r > 0] of an accumulator of scores (times 2^20: at least 4 where positive, r is a multiple of 2^-18) as the bf16 operand of
// the next product, each entry 0 or 2^-7: the half-precision 1.0 read as bf16, a conversion and a packed clamp for two.
// The clamp is written in C, so that the compiler knows a vector instruction in front of the product and keeps the wait states between.  Of a
// conversion without another use it would become the conversion's own clamp, which does nothing.
__device__ __forceinline__ unsigned mask_pair(float lo, float hi) {
  const auto pk = __builtin_amdgcn_cvt_pkrtz(lo, hi);
  asm volatile("" :: "v"(pk));
  const f16x2 none = {0.f, 0.f}, one = {1.f, 1.f};
  return __builtin_bit_cast(unsigned, __builtin_elementwise_min(__builtin_elementwise_max(__builtin_bit_cast(f16x2, pk), none), one));
}
template <int NHT>
__device__ __forceinline__ void score_masks(const f32x16 (&acc)[NHT], bf16x8 (&mk)[2 * NHT]) {
#pragma unroll
  for (int t = 0; t < NHT; t++)
#pragma unroll
    for (int s = 0; s < 2; s++) {
      unsigned pk[4];
#pragma unroll
      for (int e = 0; e < 4; e++) pk[e] = mask_pair(acc[t][8 * s + 2 * e], acc[t][8 * s + 2 * e + 1]);
      mk[2 * t + s] = __builtin_bit_cast(bf16x8, make_uint4(pk[0], pk[1], pk[2], pk[3]));
    }
}

// ---- what follows the sums: from payload gradients to gradients of the projections' outputs ------------------
// 16 lanes per row, 8 consecutive elements per lane:  / scale (rows on the quantiser's epsilon floor: 0), Hadamard
// rotation (its own transpose), bf16, transposed rotary embedding of the first 64 elements - the steps of the front
// end backwards, rounding where the separate operations round.
struct RowFinish {
  int rotate;                            // 0 none, 1 of all 128 elements, 2 of the leading 64 (heads of 64 channels)
  const void* cos_t;
  const void* sin_t;
  int cs_f32, pairing, batch;            // pairing -1: no rotary part
};

__device__ __forceinline__ float table_entry(const void* t, int is_f32, long i) {
  return is_f32 ? ((const float*)t)[i] : bf16_bits_to_f32(((const unsigned short*)t)[i]);
}
// cs: the token's 64 cosines and 64 sines where they are at hand already, else null
__device__ __forceinline__ void finish_row(float (&v)[8], int sub, float scale_inv, const RowFinish& f, const int* positions, int token,
                                           const float* cs) {
  constexpr float FLOOR = 0x1.8p-48f;
  const bool usable = scale_inv > FLOOR && scale_inv < INFINITY;
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = usable ? v[i] / scale_inv : 0.f;
  if (f.rotate) {
#pragma unroll
    for (int m = 1; m < 8; m <<= 1)
#pragma unroll
      for (int i = 0; i < 8; i++)
        if (!(i & m)) { const float a = v[i], b = v[i | m]; v[i] = a + b; v[i | m] = a - b; }
#pragma unroll
    for (int m = 1; m < 8; m <<= 1)
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const float o = xor16(v[i], m);
        v[i] = (sub & m) ? o - v[i] : v[i] + o;
      }
    if (f.rotate == 1) {
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const float o = xor16(v[i], 8);
        v[i] = (sub & 8) ? o - v[i] : v[i] + o;
      }
    }
    const float norm = f.rotate == 1 ? 0.08838834764831845f : 0.125f;
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] *= norm;
  }
  if (f.pairing >= 0) {
#pragma clang fp contract(off)
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = bf16_bits_to_f32(f32_to_bf16_bits(v[i]));
    const long row = cs ? 0 : (positions ? positions[token] : token / f.batch) * 64l;
    // element e of a pair (a, b):  a' = a cos[e] + b sin[partner],  b' = b cos[e] - a sin[partner]
    float other[8];
    if (f.pairing == 1) {
#pragma unroll
      for (int i = 0; i < 8; i++) other[i] = xor16(v[i], 4);
    } else {
#pragma unroll
      for (int i = 0; i < 8; i++) other[i] = v[i ^ 1];
    }
    if (sub < 8) {
      float c[8], s[8];
      const long co = row + sub * 8, so = f.pairing == 1 ? row + (sub ^ 4) * 8 : co;
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int j = f.pairing == 1 ? i : i ^ 1;
        c[i] = cs ? cs[co + i] : table_entry(f.cos_t, f.cs_f32, co + i);
        s[i] = cs ? cs[64 + so + j] : table_entry(f.sin_t, f.cs_f32, so + j);
      }
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const bool second = f.pairing == 1 ? sub >= 4 : (i & 1);
        const float y = second ? (-other[i]) * s[i] + v[i] * c[i] : v[i] * c[i] + other[i] * s[i];
        v[i] = bf16_bits_to_f32(f32_to_bf16_bits(y));
      }
    }
  }
}

// elements [8 sub, 8 sub + 8) of an output row of `dim` elements, bf16 or fp32
__device__ __forceinline__ void store_row(const float (&v)[8], void* base, int is_f32, size_t row, int dim, int sub) {
  const int c0 = 8 * sub;
  if (c0 >= dim) return;
  if (dim % 8 == 0) {
    if (is_f32) {
      float* p = (float*)base + row * dim + c0;
      *(f32x4*)p = f32x4{v[0], v[1], v[2], v[3]};
      *(f32x4*)(p + 4) = f32x4{v[4], v[5], v[6], v[7]};
    } else {
      *(uint4*)((unsigned short*)base + row * dim + c0) =
          make_uint4(cvt_pk_bf16(v[0], v[1]), cvt_pk_bf16(v[2], v[3]), cvt_pk_bf16(v[4], v[5]), cvt_pk_bf16(v[6], v[7]));
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < 8; i++)
    if (c0 + i < dim) {
      if (is_f32) ((float*)base)[row * dim + c0 + i] = v[i];
      else ((unsigned short*)base)[row * dim + c0 + i] = f32_to_bf16_bits(v[i]);
    }
}

struct BwdArgs {
  const float* gsc;
  const unsigned char* q8;
  const unsigned char* k8;
  const float* k_scale;
  const float* q_w;
  const int* ids;
  const int* dst;
  unsigned short* rows;
  int q0, cnt, Sk, K, dummy_row;         // (dst, rows, dummy_row: only where the workgroups write rows)
  // plain payload gradients (q_scale null) ...
  float* d_q8;                           // [S, HI, 128]
  float* d_qw;                           // [S, HI]
  // ... or finished ones
  const float* q_scale;
  float w_scale;
  RowFinish fin;
  const int* pos_q;
  int heads, dim;                        // of the outputs
  void* d_q; int q_f32;                  // [S, heads, dim]
  void* d_w; int w_f32;                  // [S, heads]
};

// Tiles in a wave's LDS ring: three, two where the slot arrays of a longer list need the room.  (Four for the waves that
// store rows, whose transfers are awaited behind their stores, and two for the others: the same time.)
int bwd_stages(int K) { return K <= 2048 ? 3 : 2; }

// What a workgroup needs to the end lies behind both the loop's arrays and the reduction buffers that take their place: weights [64],
// scales [64], cosines and sines [2][64], last slot.
constexpr size_t KEPT_BYTES = 4 * 64 * 4 + 64;
__host__ __device__ constexpr size_t kept_offset(int HI, int stages, int K, bool rows) {
  const size_t loop = (size_t)stages * (rows ? 8 : 4) * WAVE_BYTES + (size_t)HI * D + (size_t)K * (rows ? 16 : 12);
  const size_t red = (size_t)4 * (rows ? HI : 32) * RED_STRIDE * 4 + 4 * 64 * 4;
  return loop > red ? loop : red;
}
size_t bwd_lds_bytes(int HI, int stages, int K, bool rows) { return kept_offset(HI, stages, K, rows) + KEPT_BYTES; }

// The waves share nothing inside the loop: each brings the 32 key rows of its slots into a ring of its own and there is no
// barrier, so that one wave's vector work runs under the matrix work of the other wave of its SIMD.  The loop is bound by
// vector issue, hence one role per wave (both products in every wave, a half of d or of the heads each, doubles the masks
// and the operand conversions: 1.5 ms at the size above), a mask of 2^-7 (the half-precision 1.0 read as bf16, made by a
// conversion and a packed clamp for two elements) and slot offsets in the instructions.
//
// ROWS = false: d_k8 is the work of the kernels by key tiles (below).  Four waves sum d_q8 then, in half of a compute unit's LDS (two
// tiles in a ring): one query's set-up and final sums pass under another's loop (8192 queries x 2048 slots 0.53 ms, matrix pipe 59 % busy by
// the counters; 0.60 and 48 % with a front end's final steps; eight waves and a whole compute unit a query 0.825).
template <int NHT, int STAGES, bool ROWS>   // head tiles of 32
__global__ __launch_bounds__(ROWS ? THREADS : THREADS / 2) __attribute__((amdgpu_waves_per_eu(2, 2))) void indexer_bwd_kernel(const BwdArgs A) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  constexpr int HI = 32 * NHT;
  constexpr int NT = ROWS ? THREADS : THREADS / 2, WAVES = NT / 64;
  constexpr int PT = 4 * THREADS / NT;              // slots per thread and round trip
  // [8 waves][STAGES][WAVE_BYTES] fp8 key rows | q8 [HI][128] | a_s [K] f32 | ahl_s [K / 4][4 hi, 4 lo] bf16 | idx_s [K] | dst_s [K] ||
  // w_s [64] | scale_s [64] | cs_s [2][64] | last_s
  unsigned char* qs = smem + WAVES * STAGES * WAVE_BYTES;
  const int K = A.K;
  float* a_s = (float*)(qs + HI * D);
  unsigned short* ahl_s = (unsigned short*)(a_s + K);
  int* idx_s = (int*)(ahl_s + 2 * K);
  int* dst_s = idx_s + K;
  float* w_s = (float*)(smem + kept_offset(HI, STAGES, K, ROWS));
  float *scale_s = w_s + 64, *cs_s = w_s + 128;
  int* last_s = (int*)(w_s + 256);
  float* dw_red = (float*)smem;                     // [4][64], then red [4][HI or 32][RED_STRIDE], reuse the front at the end
  float* red = dw_red + 4 * 64;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave & 3;                          // slots 32 kg .. of a tile
  const int r = lane & 31, g = lane >> 5;
  const int ql = A.cnt - 1 - (int)blockIdx.x;
  const int qi = A.q0 + ql;

  // ---- the query: slots, rows, weights.  Nothing else runs on the compute unit meanwhile, so the chain of round trips to memory is
  // kept short: the slots, the query's rows and weights in one, then the first key rows beside the keys' scales. --------------
  if (tid == 0) *last_s = -1;
  const unsigned char* qrow = A.q8 + (size_t)qi * HI * D;
  const int* ids = A.ids + (size_t)qi * K;
  const float* gsc = A.gsc + (size_t)qi * K;
  const int* dst = ROWS ? A.dst + (size_t)ql * K : nullptr;
  int v[PT], d[PT];
  float gv[PT];
  auto request_slots = [&](int t0) {                // a thread's slots with all their loads in flight
#pragma unroll
    for (int i = 0; i < PT; i++) {
      const int t = min(t0 + i * NT, K - 1);
      v[i] = ids[t];
      gv[i] = gsc[t];
      if (ROWS) d[i] = dst[t];
    }
  };
  request_slots(tid);
  const float w_in = A.q_w[(size_t)qi * HI + min(tid, HI - 1)];
  const float scale_in = A.q_scale ? A.q_scale[(size_t)qi * HI + min(tid, HI - 1)] : 0.f;
  const bool rotary = A.q_scale != nullptr && A.fin.pairing >= 0;
  const long pos = !rotary ? 0 : A.pos_q ? A.pos_q[qi] : qi / A.fin.batch;
  const uint4 q_in = *(const uint4*)(qrow + min(tid, HI * 8 - 1) * 16);
  const uint4 q_in2 = *(const uint4*)(qrow + min(tid + NT, HI * 8 - 1) * 16);
  // Where the key of a slot that counts for nothing is read (its factor is 0): the first slot's key, which the query has selected
  const int spare = (unsigned)ids[0] < (unsigned)A.Sk ? ids[0] : 0;
  __builtin_amdgcn_sched_barrier(0);
  int last = -1;
  for (int t0 = tid; t0 < K; t0 += 4 * THREADS) {   // ids first: the transfers of key rows want nothing else
    if (t0 != tid) {
#pragma unroll
      for (int i = 0; i < PT; i++) v[i] = ids[min(t0 + i * NT, K - 1)];
    }
#pragma unroll
    for (int i = 0; i < PT; i++) {
      const int t = t0 + i * NT;
      const bool ok = v[i] >= 0 && v[i] < A.Sk;
      if (t < K) {
        idx_s[t] = ok ? v[i] : spare;
        if (ok) last = t;
      }
    }
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) last = max(last, __shfl_xor(last, o, 64));
  __syncthreads();                                  // *last_s has been set
  if (lane == 0) atomicMax(last_s, last);
  if (tid < HI) {
    w_s[tid] = w_in;
    scale_s[tid] = scale_in;
  }
  auto keep_query = [&](int c, const uint4& q) {
    if (c < HI * 8) *(uint4*)(qs + (c >> 3) * D + (((c & 7) ^ slot_xor(c >> 3)) << 4)) = q;
  };
  keep_query(tid, q_in);
  if (NT < HI * 8) keep_query(tid + NT, q_in2);
  DSA_WAIT_VMCNT(0);                                // every load so far: what is in flight below are the transfers and the scales
  __syncthreads();
  const int ntile = (*last_s + TK) / TK;            // tiles behind the last valid slot have nothing to add

  // ---- lane-dependent LDS offsets ------------------------------------------------------------------
  const unsigned lds0 = (unsigned)(uintptr_t)smem, ring = lds0 + (unsigned)(wave * STAGES * WAVE_BYTES);
  const unsigned a_lds = lds0 + (unsigned)((unsigned char*)a_s - smem), ahl_lds = lds0 + (unsigned)((unsigned char*)ahl_s - smem),
                 dst_lds = lds0 + (unsigned)((unsigned char*)dst_s - smem), idx_lds = lds0 + (unsigned)((unsigned char*)idx_s - smem);
  unsigned b_off[2][2];      // key row r of the wave's 32, bytes [64 s + 32 g, + 32)
#pragma unroll
  for (int s = 0; s < 2; s++)
#pragma unroll
    for (int x = 0; x < 2; x++) b_off[s][x] = ring + (unsigned)(r * D + (((4 * s + 2 * g + x) ^ slot_xor(r)) << 4));
  const int blk = lane >> 4, ii = lane & 15;
  const int tr_row = 8 * (ii >> 3) + 4 * g + ((ii >> 1) & 3);          // row of a transposing read, + 16 per k-step

  const int gkey = lane >> 3, gsub = lane & 7;
  const unsigned g_off = (unsigned)((gsub ^ slot_xor(gkey)) * 16);     // the lane's chunk of the key row it fetches; rows 8 - 15, 24 - 31: XOR 64
  const unsigned idx_lane = idx_lds + (unsigned)(32 * kg + gkey) * 4;
  auto issue = [&](int n, int stage) {          // four transfers of eight key rows
    const unsigned lb = __builtin_amdgcn_readfirstlane(ring + (unsigned)(stage * WAVE_BYTES));
    const unsigned ia = idx_lane + (unsigned)(n * TK * 4);
#pragma unroll
    for (int c = 0; c < 4; c++) dma16(lb + c * 1024, (lds_read<unsigned>(ia + c * 32) << 7) | (g_off ^ (unsigned)((c & 1) * 64)), A.k8);
  };
  for (int n = 0; n < STAGES - 1 && n < ntile; n++) issue(n, n);
  __builtin_amdgcn_sched_barrier(0);
  // factors and destination rows of the slots and the token's angles, while the first key rows are on their way
  const float cs_in = rotary && tid < 128 ? table_entry(tid < 64 ? A.fin.cos_t : A.fin.sin_t, A.fin.cs_f32, pos * 64 + (tid & 63)) : 0.f;
  for (int t0 = tid; t0 < K; t0 += 4 * THREADS) {
    if (K > 4 * THREADS) request_slots(t0);
    float kv[PT];
#pragma unroll
    for (int i = 0; i < PT; i++) kv[i] = A.k_scale[(v[i] >= 0 && v[i] < A.Sk) ? v[i] : 0];
#pragma unroll
    for (int i = 0; i < PT; i++) {
      const int t = t0 + i * NT;
      if (t < K) {
        const bool ok = v[i] >= 0 && v[i] < A.Sk;
        const float a = ok ? gv[i] * kv[i] : 0.f;
        const unsigned short hi = f32_to_bf16_bits(a);
        a_s[t] = a;
        ahl_s[(t >> 2) * 8 + (t & 3)] = hi;
        ahl_s[(t >> 2) * 8 + 4 + (t & 3)] = f32_to_bf16_bits(a - bf16_bits_to_f32(hi));
        if (ROWS) dst_s[t] = (ok && d[i] >= 0) ? d[i] : A.dummy_row;
      }
    }
  }
  if (tid < 128) cs_s[tid] = cs_in;
  __syncthreads();
  auto key_rows = [&](unsigned stage_off, i32x8 (&bk)[2]) {
#pragma unroll
    for (int s = 0; s < 2; s++) {
      const i32x4 lo = lds_read<i32x4>(b_off[s][0] + stage_off);
      const i32x4 hi = lds_read<i32x4>(b_off[s][1] + stage_off);
      bk[s] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    }
  };
  // fp8 rows of the query, bytes [64 s + 32 g, + 32) of head 32 t + r (they lie in LDS as a tile's rows do)
  i32x8 aq[NHT][2];
  const unsigned q_delta = lds0 + (unsigned)(qs - smem) - ring;
  auto query_rows = [&]() {
#pragma unroll
    for (int t = 0; t < NHT; t++)
#pragma unroll
      for (int s = 0; s < 2; s++) {
        const i32x4 lo = lds_read<i32x4>(b_off[s][0] + q_delta + (unsigned)(t * 32 * D));
        const i32x4 hi = lds_read<i32x4>(b_off[s][1] + q_delta + (unsigned)(t * 32 * D));
        aq[t][s] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      }
  };
  const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

  auto leave_sums = [&](int head, const f32x16 (&acc)[4]) {       // this wave's sums of 32 heads, to rows head .. of its part of red
    constexpr int PER = ROWS ? HI : 32;
#pragma unroll
    for (int dt = 0; dt < 4; dt++) {
      float* rp = red + ((size_t)kg * PER + head + r) * RED_STRIDE + 32 * dt + 4 * g;
#pragma unroll
      for (int j = 0; j < 4; j++)
        *(f32x4*)(rp + 8 * j) = f32x4{acc[dt][4 * j], acc[dt][4 * j + 1], acc[dt][4 * j + 2], acc[dt][4 * j + 3]};
    }
  };
  // ---- sums of 32 heads over the four slot groups, in a fixed order, and what follows them ------------------
  const int sub = tid & 15;
  auto finish_heads = [&](int it, int head) {
    constexpr int PER = ROWS ? HI : 32;
#pragma unroll
    for (int hh = 0; hh < 32; hh += NT / 16) {
      const int h = 32 * it + hh + (tid >> 4);
      float v[8];
#pragma unroll
      for (int x = 0; x < 2; x++) {
        f32x4 p[4];
#pragma unroll
        for (int k = 0; k < 4; k++) p[k] = *(const f32x4*)(red + ((size_t)k * PER + head + hh + (tid >> 4)) * RED_STRIDE + 8 * sub + 4 * x);
#pragma unroll
        for (int e = 0; e < 4; e++) v[4 * x + e] = ((p[0][e] + p[1][e]) + (p[2][e] + p[3][e])) * w_s[h];
      }
      if (A.q_scale == nullptr) {
        store_row(v, A.d_q8, 1, (size_t)qi * HI + h, D, sub);
      } else {
        finish_row(v, sub, scale_s[h], A.fin, nullptr, qi, cs_s);
        if (h < A.heads) store_row(v, A.d_q, A.q_f32, (size_t)qi * A.heads + h, A.dim, sub);
      }
    }
  };

  if (ROWS && wave < 4) {
    // ======== rows of d_k8 ============================================================================
    // (q_w Q)^T operands: lane = d row 32 dt + r, 8 heads of k-step kk = 2 t + s in accumulator order
    bf16x8 qt[4][2 * NHT];
#pragma unroll
    for (int kk = 0; kk < 2 * NHT; kk++)
#pragma unroll
      for (int dt = 0; dt < 4; dt++)
        qt[dt][kk] = __builtin_bit_cast(bf16x8, weighted_query(lds0 + (unsigned)(qs - smem), w_s, lane, dt, kk));
    query_rows();
    unsigned short* const rows = A.rows + 8 * g;
    const unsigned slot_off = (unsigned)(32 * kg + r) * 4;
    i32x8 bk[2];
    float a = 0.f;
    unsigned row = 0;
    // Start of tile n in ring slot st: its rows have landed once at most `behind` operations issued after their transfers
    // are in flight; what the tile's first products need is read.
    auto open_tile = [&](int n, int st) {
      key_rows(st * WAVE_BYTES, bk);
      const unsigned so = slot_off + (unsigned)(n * TK * 4);
      a = lds_read<float>(a_lds + so) * 128.f;
      row = lds_read<unsigned>(dst_lds + so);
    };
    if (ntile > 0) {
      if (ntile >= STAGES - 1) { DSA_WAIT_VMCNT(4 * (STAGES - 2)); } else { DSA_WAIT_VMCNT(0); }
      asm volatile("" ::: "memory");   // no LDS read moves above the wait
      open_tile(0, 0);
    }
    for (int n0 = 0; n0 < ntile; n0 += STAGES)
#pragma unroll
      for (int st = 0; st < STAGES; st++) {
        const int n = n0 + st;
        if (n >= ntile) break;
        // the slot that the tile STAGES - 1 ahead goes to was read one iteration ago (its reads fed that iteration's products)
        if (n + STAGES - 1 < ntile) issue(n + STAGES - 1, (st + STAGES - 1) % STAGES);
        f32x16 acc[NHT];
#pragma unroll
        for (int t = 0; t < NHT; t++) {        // r 2^20: at least 4 where r > 0 (r is a multiple of 2^-18)
          acc[t] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(aq[t][0], bk[0], zero, 0, 0, 0, 147, 0, 127);
          acc[t] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(aq[t][1], bk[1], acc[t], 0, 0, 0, 147, 0, 127);
        }
        const float a_n = a;
        unsigned short* const rowp = rows + (size_t)row * D;
        bf16x8 mk[2 * NHT];
        score_masks<NHT>(acc, mk);
        f32x16 racc[2];
#pragma unroll
        for (int dt = 0; dt < 5; dt++) {       // the products of a d-tile run while the one before it is rounded and stored
          if (dt < 4) {
#pragma unroll
            for (int kk = 0; kk < 2 * NHT; kk++)
              racc[dt & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qt[dt][kk], mk[kk], kk ? racc[dt & 1] : zero, 0, 0, 0);
          }
          if (dt == 3 && n + 1 < ntile) {
            // issued behind the next tile's transfers: four per later tile in flight, eight stores per tile since (four of this one)
            if (n >= STAGES - 2 && n + STAGES - 1 < ntile) { DSA_WAIT_VMCNT(4 * (STAGES - 2) + 8 * (STAGES - 2) + 4); }
            else if (n >= STAGES - 2) { DSA_WAIT_VMCNT(8 * (STAGES - 2) + 4); }
            else { DSA_WAIT_VMCNT(4); }
            asm volatile("" ::: "memory");   // no LDS read moves above the wait
            open_tile(n + 1, (st + 1) % STAGES);
          }
          if (dt > 0) {
            uint4 o[2];
            acc_row_to_16B(racc[(dt - 1) & 1], a_n, o);
            *(uint4*)(rowp + 32 * (dt - 1)) = o[0];
            *(uint4*)(rowp + 32 * (dt - 1) + 16) = o[1];
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    __syncthreads();
  } else {
    // ======== d_q8 and d_qw ===========================================================================
    unsigned kt_off[4];      // K^T operand of d-tile dt (k-step s: 16 s rows on)
#pragma unroll
    for (int dt = 0; dt < 4; dt++)
      kt_off[dt] = ring + (unsigned)(tr_row * D + (((2 * dt + (blk & 1)) ^ slot_xor(tr_row)) << 4) + 8 * (ii & 1));
    f32x16 dq_acc[NHT][4];
    float dw[NHT];           // d_qw of head 32 t + r over the keys of this half-wave
#pragma unroll
    for (int t = 0; t < NHT; t++) {
      dw[t] = 0.f;
#pragma unroll
      for (int dt = 0; dt < 4; dt++) dq_acc[t][dt] = zero;
    }
    const unsigned slot_off = (unsigned)(32 * kg + 4 * g) * 4;
    i32x8 bk[2];
    f32x4 a4[2];             // factors of the keys 16 s + 8 b + 4 g .. + 3 of a k-step: fp32, and as pairs of bf16
    i32x4 hl[2];
    f32x16 acc[NHT];
    unsigned ph[NHT][4], pl[NHT][4];
    i32x2 kr[4];
    auto read_factors = [&](int n, int s) {
      const unsigned so = slot_off + (unsigned)(n * TK * 4 + 64 * s);
#pragma unroll
      for (int b = 0; b < 2; b++) {
        a4[b] = lds_read<f32x4>(a_lds + so + 32 * b);
        hl[b] = lds_read<i32x4>(ahl_lds + so + 32 * b);
      }
    };
    auto read_keys_t = [&](int st, int s) {
#pragma unroll
      for (int dt = 0; dt < 4; dt++) kr[dt] = read_tr8(kt_off[dt] + (unsigned)(st * WAVE_BYTES + s * 16 * D));
    };
    auto coefs = [&](int s, int b, int t) {       // four keys of one head tile
#pragma unroll
      for (int x = 0; x < 2; x++) {
        // relu on the bit patterns; their upper halves, at most 1 each, are the mask that the coefficients are multiplied by
        const float r0 = acc[t][8 * s + 4 * b + 2 * x], r1 = acc[t][8 * s + 4 * b + 2 * x + 1];
        const int p0 = max(__builtin_bit_cast(int, r0), 0), p1 = max(__builtin_bit_cast(int, r1), 0);
        dw[t] = fmaf(a4[b][2 * x], __builtin_bit_cast(float, p0), dw[t]);
        dw[t] = fmaf(a4[b][2 * x + 1], __builtin_bit_cast(float, p1), dw[t]);
        unsigned m = __builtin_amdgcn_perm((unsigned)p1, (unsigned)p0, 0x07060302u);
        asm("v_pk_min_u16 %0, %0, %1" : "+v"(m) : "s"(0x00010001u));
        // (the products in C, so that the compiler keeps their wait states; of a mask that it knew it would make two selects each)
        ph[t][2 * b + x] = __builtin_bit_cast(unsigned, __builtin_bit_cast(u16x2, m) * __builtin_bit_cast(u16x2, (int)hl[b][x]));
        pl[t][2 * b + x] = __builtin_bit_cast(unsigned, __builtin_bit_cast(u16x2, m) * __builtin_bit_cast(u16x2, (int)hl[b][2 + x]));
      }
    };
    if (ntile > 0) {
      if (ntile >= STAGES - 1) { DSA_WAIT_VMCNT(4 * (STAGES - 2)); } else { DSA_WAIT_VMCNT(0); }
      asm volatile("" ::: "memory");
      key_rows(0, bk);
      query_rows();
    }
    for (int n0 = 0; n0 < ntile; n0 += STAGES)
#pragma unroll
      for (int st = 0; st < STAGES; st++) {
        const int n = n0 + st;
        if (n >= ntile) break;
        if (n + STAGES - 1 < ntile) issue(n + STAGES - 1, (st + STAGES - 1) % STAGES);
#pragma unroll
        for (int t = 0; t < NHT; t++) {
          acc[t] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(bk[0], aq[t][0], zero, 0, 0, 0, 127, 0, 127);
          acc[t] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(bk[1], aq[t][1], acc[t], 0, 0, 0, 127, 0, 127);
        }
        read_factors(n, 0);
        __builtin_amdgcn_sched_barrier(0);
        coefs(0, 0, 0);
        coefs(0, 1, 0);
        read_keys_t(st, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (NHT == 2) { coefs(0, 0, NHT - 1); coefs(0, 1, NHT - 1); }
        read_factors(n, 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 2; s++) {
          bf16x8 eh[NHT], el[NHT];
#pragma unroll
          for (int t = 0; t < NHT; t++) {
            eh[t] = __builtin_bit_cast(bf16x8, make_uint4(ph[t][0], ph[t][1], ph[t][2], ph[t][3]));
            el[t] = __builtin_bit_cast(bf16x8, make_uint4(pl[t][0], pl[t][1], pl[t][2], pl[t][3]));
          }
          if (s == 1) {     // the next tile's first operands travel under this tile's last products (behind the last tile: unused)
            if (n + STAGES - 1 < ntile) { DSA_WAIT_VMCNT(4 * (STAGES - 2)); } else { DSA_WAIT_VMCNT(0); }
            asm volatile("" ::: "memory");
            key_rows((st + 1) % STAGES * WAVE_BYTES, bk);
            query_rows();                    // (kept, its 32 registers would not fit beside the sums)
          }
#pragma unroll
          for (int dt = 0; dt < 4; dt++) {
            const bf16x8 kt = fp8_to_bf16(kr[dt]);
#pragma unroll
            for (int t = 0; t < NHT; t++) dq_acc[t][dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kt, eh[t], dq_acc[t][dt], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < NHT; t++) dq_acc[t][dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kt, el[t], dq_acc[t][dt], 0, 0, 0);
            if (s == 0) {                    // the second k-step's coefficients under the first one's products
              if (NHT == 2) coefs(1, dt >> 1, dt & 1);
              else if (dt < 2) coefs(1, dt, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
          }
          if (s == 0) read_keys_t(st, 1);
        }
      }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NHT; t++) {
      const float v = dw[t] + __shfl_xor(dw[t], 32, 64);
      if (g == 0) dw_red[kg * 64 + 32 * t + r] = v;
    }
    if (ROWS) {
#pragma unroll
      for (int t = 0; t < NHT; t++) leave_sums(32 * t, dq_acc[t]);
    } else {
#pragma unroll
      for (int t = 0; t < NHT; t++) {
        if (t) __syncthreads();
        leave_sums(0, dq_acc[t]);
        __syncthreads();
        finish_heads(t, 0);
      }
    }
  }

  if (ROWS) {
    __syncthreads();
#pragma unroll
    for (int it = 0; it < NHT; it++) finish_heads(it, 32 * it);
  }
  if (tid < HI) {
    const float s = (dw_red[tid] + dw_red[64 + tid]) + (dw_red[128 + tid] + dw_red[192 + tid]);
    if (A.q_scale == nullptr) {
      A.d_qw[(size_t)qi * HI + tid] = s;
    } else if (tid < A.heads) {
      const float y = s * scale_s[tid] * A.w_scale;
      if (A.w_f32) ((float*)A.d_w)[(size_t)qi * A.heads + tid] = y;
      else ((unsigned short*)A.d_w)[(size_t)qi * A.heads + tid] = f32_to_bf16_bits(y);
    }
  }
}

// d_k8[key] (+)= sum of the key's bf16 rows in fp32, ascending query order; 16 chunks of 8 columns x RED_GROUPS row groups (row
// r of the segment goes to group r % RED_GROUPS), the groups combined in a fixed order.  A stream of reads, eight rows in
// flight per thread, non-temporal: 8192 keys x 1800 rows 0.59 ms (6.4 TB/s), 768 keys x 1640 rows 0.053 ms.  (Eight groups,
// plain loads and as many rows in flight as the compiler chose: 0.73 and 0.19 ms; with 8 groups 0.57 and 0.057, with 32 0.60
// and 0.055.)
constexpr int RED_GROUPS = 16;
constexpr int RED_FLIGHT = 8;
__global__ __launch_bounds__(16 * RED_GROUPS) void indexer_reduce_kernel(const unsigned short* __restrict__ rows, const int* __restrict__ start,
                                                                     float* __restrict__ d_k8, int accumulate,
                                                                     const int* __restrict__ dup_flag) {
  typedef unsigned u32x4_nt __attribute__((ext_vector_type(4)));
  __shared__ float part[RED_GROUPS][D];
  const int key = blockIdx.x, ch = threadIdx.x & 15, grp = threadIdx.x >> 4;
  const int s0 = start[key], s1 = start[key + 1];
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; e++) acc[e] = 0.f;
  auto add = [&](const u32x4_nt& v) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      acc[2 * e] += __builtin_bit_cast(float, (unsigned)v[e] << 16);
      acc[2 * e + 1] += __builtin_bit_cast(float, (unsigned)v[e] & 0xffff0000u);
    }
  };
  auto row = [&](int rr) { return __builtin_nontemporal_load((const u32x4_nt*)(rows + (size_t)rr * D + 8 * ch)); };
  int rr = s0 + grp;
  for (; rr + (RED_FLIGHT - 1) * RED_GROUPS < s1; rr += RED_FLIGHT * RED_GROUPS) {
    u32x4_nt v[RED_FLIGHT];
#pragma unroll
    for (int u = 0; u < RED_FLIGHT; u++) v[u] = row(rr + u * RED_GROUPS);
#pragma unroll
    for (int u = 0; u < RED_FLIGHT; u++) add(v[u]);
  }
  for (; rr < s1; rr += RED_GROUPS) add(row(rr));
#pragma unroll
  for (int e = 0; e < 8; e++) part[grp][8 * ch + e] = acc[e];
  __syncthreads();
  if (threadIdx.x < D) {
    const int c = threadIdx.x;      // one column per thread
    float s = 0.f;
#pragma unroll
    for (int g = 0; g < RED_GROUPS; g += 4) s += (part[g][c] + part[g + 1][c]) + (part[g + 2][c] + part[g + 3][c]);
    float* p = d_k8 + (size_t)key * D + c;
    if (accumulate) s += *p;
    if (*dup_flag) s = __builtin_nanf("");       // a query row held a repeated id: no sum that misses a term
    *p = s;
  }
}

// ======== d_k8 by key tiles ==========================================================================
// Where a good part of the keys that the queries see is selected, a row per pair through memory (256 bytes written and read, the
// key-sorted order, the sums) costs more than the products with every key of the range: a workgroup then owns 256 keys and a
// chunk of queries, its sums stay in registers, and the pair factors a (0 for a pair that is not selected) come from a dense array.
//   scatter   per query: the factors of its 256-key tiles that hold a selected key, which tiles these are, and the operands of both
//             products in the layout of the matrix instructions
//   keys      per (chunk of queries, 256 keys): d_k8 over the chunk's queries that touch the tile, in ascending order
//   reduce    per key: the chunks' sums in a fixed order
// The sums are fp32 throughout (a row of a pair is not rounded to bf16).
constexpr int KT = 256;                 // keys per tile
constexpr int PIECE_TILES = 16;         // tiles whose factors are scattered in LDS at a time; their marks are one word
constexpr unsigned UNSELECTED = 0x80000000u;       // -0: adds nothing, and is told from a selected pair's factor 0
constexpr int QUERY_BAD = 1, QUERY_DUP = 2;

__host__ __device__ constexpr int operand_bytes(int NHT) { return NHT * 12 * 1024; }   // fp8 rows 4 KB, (q_w Q)^T 8 KB per head tile

struct DenseArgs {
  const float* gsc;
  const unsigned char* q8;
  const unsigned char* k8;
  const float* k_scale;
  const float* q_w;
  const int* ids;
  int q0, cnt, Sk, K;
  int tiles, words, chunk, chunks;      // key tiles, words of marks per query, queries per chunk
  float* factors;                       // [cnt][tiles][KT], written where marked
  unsigned* marks;                      // [cnt][words]
  int* state;                           // [cnt]
  unsigned char* ops;                   // [cnt][operand_bytes]
  float* part;                          // [chunks][tiles][KT][D], written where used
  int* used;                            // [chunks][tiles]: queries summed; negative: a query of the chunk repeats an id
};

// 110 us at 8192 queries x 2048 slots x 64 heads, for 200 MB of operands and 134 MB of factors: three to six workgroups a compute unit,
// each a chain of loads, LDS scatters and barriers (with 32 tiles a piece, half as many workgroups: 139).
template <int NHT>
__global__ __launch_bounds__(256) void indexer_scatter_kernel(const DenseArgs A) {
  constexpr int HI = 32 * NHT, SLOTS = 16;          // K <= 4096
  constexpr unsigned EMPTY = 0xffffffffu;
  __shared__ __attribute__((aligned(16))) unsigned row[PIECE_TILES * KT];
  __shared__ __attribute__((aligned(1024))) unsigned char qs[HI * D];
  __shared__ __attribute__((aligned(16))) float w_s[HI];
  __shared__ int lo_s, hi_s, flags_s;
  __shared__ unsigned marks_s;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ql = blockIdx.x, qi = A.q0 + ql;
  if (tid == 0) { lo_s = 0x7fffffff; hi_s = -1; flags_s = 0; marks_s = 0; }
  const int* ids = A.ids + (size_t)qi * A.K;
  const float* gsc = A.gsc + (size_t)qi * A.K;
  int id[SLOTS];
  unsigned a[SLOTS];
#pragma unroll
  for (int i = 0; i < SLOTS; i++) {
    const int t = tid + 256 * i;
    id[i] = t < A.K ? ids[t] : -1;
    a[i] = t < A.K ? __builtin_bit_cast(unsigned, gsc[t]) : 0u;
  }
  for (int c = tid; c < HI * 8; c += 256) *(uint4*)(qs + (c >> 3) * D + (((c & 7) ^ slot_xor(c >> 3)) << 4)) = *(const uint4*)(A.q8 + (size_t)qi * HI * D + c * 16);
  if (tid < HI) w_s[tid] = A.q_w[(size_t)qi * HI + tid];
  int lo = 0x7fffffff, hi = -1;
#pragma unroll
  for (int i = 0; i < SLOTS; i++) {
    if (id[i] >= A.Sk) id[i] = -1;
    if (id[i] >= 0) {
      float f = __builtin_bit_cast(float, a[i]) * A.k_scale[id[i]];
      a[i] = __builtin_bit_cast(unsigned, f);
      if (a[i] == EMPTY) a[i] = 0x7fc00000u;        // a NaN all the same
      if (a[i] == UNSELECTED) a[i] = 0u;
      lo = min(lo, id[i]);
      hi = max(hi, id[i]);
    }
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    lo = min(lo, __shfl_xor(lo, o, 64));
    hi = max(hi, __shfl_xor(hi, o, 64));
  }
  __syncthreads();
  if (lane == 0) {
    atomicMin(&lo_s, lo);
    atomicMax(&hi_s, hi);
  }
  // ---- operands ------------------------------------------------------------------------------------
  unsigned char* ops = A.ops + (size_t)ql * operand_bytes(NHT) + lane * 16;
  const unsigned q_lds = (unsigned)(uintptr_t)qs;
  const int r = lane & 31, g = lane >> 5;
  for (int b = wave; b < 4 * NHT; b += 4) {         // block (t, s, x): bytes [64 s + 32 g + 16 x, + 16) of head 32 t + r
    const int t = b >> 2, s = (b >> 1) & 1, x = b & 1;
    *(uint4*)(ops + b * 1024) = *(const uint4*)(qs + (32 * t + r) * D + (((4 * s + 2 * g + x) ^ slot_xor(r)) << 4));
  }
  bool bad = false;
  for (int b = wave; b < 8 * NHT; b += 4) {         // block (dt, kk)
    const uint4 v = weighted_query(q_lds, w_s, lane, b / (2 * NHT), b % (2 * NHT));
    const unsigned w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int e = 0; e < 4; e++) bad |= (w[e] & 0x7f80u) == 0x7f80u || (w[e] & 0x7f800000u) == 0x7f800000u;
    *(uint4*)(ops + (4 * NHT + b) * 1024) = v;
  }
  // ---- factors, a piece of the keys at a time ----------------------------------------------------------
  __syncthreads();
  const int first = hi_s < 0 ? A.words : lo_s / (PIECE_TILES * KT), behind = hi_s < 0 ? 0 : hi_s / (PIECE_TILES * KT) + 1;
  bool dup = false;
  for (int p = 0; p < A.words; p++) {
    if (p < first || p >= behind) {
      if (tid == 0) A.marks[(size_t)ql * A.words + p] = 0u;
      continue;
    }
    const int nt = min(PIECE_TILES, A.tiles - p * PIECE_TILES);
    for (int c = tid; c < nt * (KT / 4); c += 256) *(uint4*)(row + 4 * c) = make_uint4(EMPTY, EMPTY, EMPTY, EMPTY);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < SLOTS; i++)
      if (id[i] >= 0 && id[i] / (PIECE_TILES * KT) == p) dup |= atomicExch(row + id[i] % (PIECE_TILES * KT), a[i]) != EMPTY;
    __syncthreads();
    float* out = A.factors + ((size_t)ql * A.tiles + p * PIECE_TILES) * KT + 4 * lane;
    unsigned marks = 0;
    for (int t = wave; t < nt; t += 4) {
      uint4 v = *(const uint4*)(row + t * KT + 4 * lane);
      const bool any = v.x != EMPTY || v.y != EMPTY || v.z != EMPTY || v.w != EMPTY;
      if (__ballot(any) == 0) continue;
      marks |= 1u << t;
      v.x = v.x == EMPTY ? UNSELECTED : v.x;
      v.y = v.y == EMPTY ? UNSELECTED : v.y;
      v.z = v.z == EMPTY ? UNSELECTED : v.z;
      v.w = v.w == EMPTY ? UNSELECTED : v.w;
      *(uint4*)(out + t * KT) = v;
    }
    if (lane == 0 && marks) atomicOr(&marks_s, marks);
    __syncthreads();
    if (tid == 0) {
      A.marks[(size_t)ql * A.words + p] = marks_s;
      marks_s = 0;
    }
  }
  if (bad || dup) atomicOr(&flags_s, (bad ? QUERY_BAD : 0) | (dup ? QUERY_DUP : 0));
  __syncthreads();
  if (tid == 0) A.state[ql] = flags_s;
}

// 1.57 M cycles at 8192 queries x 2048 slots x 64 heads (34 M pairs of query and key in the tiles; 0.81 - 0.85 ms): by the counters the matrix
// pipe is 52 % busy and LDS 27 %.  A wave waits for operands that it asks for one d-tile ahead, and there are no registers for two.  With the
// masks and a query's last sums by themselves instead of under products 1.65 M (inside the training pass 890 us and 849, 3072 x 512 of 768 keys
// 66.5 and 64.2, 32 heads the same); with the sums behind all products of a query and a branch per sum for operands that are not finite 8 % more
// than that, without a query's scores under the products of the one before another 10 %.
// One workgroup of eight waves, 32 keys a wave: scores of the query's heads with the wave's keys on the columns, their masks, the rows
// of the keys, times the pairs' factors into the sums.  Two queries a step; their operands and factors come into a ring of three steps
// by transfers that the waves share out.
constexpr int KEYS_STAGES = 3;
constexpr int MAX_CHUNK = 128;
template <int NHT> constexpr size_t keys_lds_bytes() { return (size_t)KEYS_STAGES * (2 * operand_bytes(NHT) + 8 * 256) + (MAX_CHUNK + 4) * 4; }

template <int NHT>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void indexer_keys_kernel(const DenseArgs A) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  constexpr int OPS = operand_bytes(NHT), STAGE = 2 * OPS + 8 * 256;
  constexpr int PER = OPS / 4096 + 1;               // transfers of a wave per step
  int* list = (int*)(smem + KEYS_STAGES * STAGE);   // [MAX_CHUNK] queries; their number; whether an operand of the chunk is not finite
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, g = lane >> 5;
  // chunk c is an XCD's (c mod 8): the workgroups that read the same queries' operands at the same time share an L2
  const int c = ((int)blockIdx.x >> 3) / A.tiles * 8 + ((int)blockIdx.x & 7), tile = ((int)blockIdx.x >> 3) % A.tiles;
  if (c >= A.chunks) return;
  if (wave == 0) {
    int n = 0;
    bool dup = false, bad = false;
    for (int h = 0; h < A.chunk; h += 64) {
      const int i = h + lane, q = c * A.chunk + i;
      const bool in = i < A.chunk && q < A.cnt;
      const int st = in ? A.state[q] : 0;
      const bool live = in && ((A.marks[(size_t)q * A.words + tile / PIECE_TILES] >> (tile % PIECE_TILES)) & 1u);
      const unsigned long long m = __ballot(live);
      if (live) list[n + __popcll(m & ((1ull << lane) - 1))] = q;
      n += __popcll(m);
      dup |= __ballot(st & QUERY_DUP) != 0;
      bad |= __ballot(st & QUERY_BAD) != 0;
    }
    if (lane == 0) {
      list[MAX_CHUNK] = n;
      list[MAX_CHUNK + 1] = bad;
      A.used[(size_t)c * A.tiles + tile] = dup ? -1 : n;
    }
  }
  __syncthreads();
  const int n = __builtin_amdgcn_readfirstlane(list[MAX_CHUNK]);
  const bool bad = __builtin_amdgcn_readfirstlane(list[MAX_CHUNK + 1]) != 0;
  if (n == 0) return;
  const unsigned lds0 = (unsigned)(uintptr_t)smem;
  const float* fbase = A.factors + ((size_t)c * A.chunk * A.tiles + tile) * KT + 32 * wave;
  int qa, qb;                                       // the two queries of the step that is requested next
  auto look_up = [&](int step) {
    qa = list[min(2 * step, n - 1)];
    qb = list[min(2 * step + 1, n - 1)];
  };
  auto issue = [&](int slot) {
    const int a = __builtin_amdgcn_readfirstlane(qa), b = __builtin_amdgcn_readfirstlane(qb);
    const unsigned base = lds0 + (unsigned)(slot * STAGE);
    const unsigned char* src = A.ops + (size_t)(wave < 4 ? a : b) * OPS + (wave & 3) * (OPS / 4);
    const unsigned dst = base + (unsigned)((wave >> 2) * OPS + (wave & 3) * (OPS / 4));
#pragma unroll
    for (int i = 0; i < PER - 1; i++) dma16(dst + i * 1024, (unsigned)(lane * 16 + i * 1024), src);
    dma4(base + (unsigned)(2 * OPS + wave * 256), (unsigned)(((lane < 32 ? a : b) - c * A.chunk) * A.tiles * (KT * 4) + r * 4), fbase);
  };
  // key row of the lane, bytes [64 s + 32 g, + 32)
  i32x8 bk[2];
  {
    const unsigned char* kp = A.k8 + (size_t)min(tile * KT + 32 * wave + r, A.Sk - 1) * D + 32 * g;
#pragma unroll
    for (int s = 0; s < 2; s++) {
      const i32x4 lo = *(const i32x4*)(kp + 64 * s), hi = *(const i32x4*)(kp + 64 * s + 16);
      bk[s] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    }
  }
  DSA_WAIT_VMCNT(0);                                // from here on only the transfers count
  asm volatile("" : "+v"(bk[0]), "+v"(bk[1]) :: "memory");
  const int steps = (n + 1) >> 1;
  look_up(0);
  issue(0);
  look_up(1);
  if (steps > 1) issue(1);
  look_up(2);
  const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  f32x16 sum[4], acc[NHT], racc[2];
  bf16x8 qt[2][2 * NHT];
  unsigned __attribute__((ext_vector_type(4))) mk[2][2 * NHT];       // of the query in hand and of the next one, in turn
#pragma unroll
  for (int dt = 0; dt < 4; dt++) sum[dt] = zero;
  auto read_query = [&](int t, unsigned ob, i32x8 (&aq)[2]) {
#pragma unroll
    for (int s = 0; s < 2; s++) {
      const i32x4 lo = lds_read<i32x4>(ob + (4 * t + 2 * s) * 1024), hi = lds_read<i32x4>(ob + (4 * t + 2 * s + 1) * 1024);
      aq[s] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    }
  };
  auto scores = [&](int t, const i32x8 (&aq)[2]) {
#pragma unroll
    for (int s = 0; s < 2; s++) acc[t] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(aq[s], bk[s], s ? acc[t] : zero, 0, 0, 0, 147, 0, 127);
  };
  auto read_weighted = [&](int dt, unsigned ob) {
#pragma unroll
    for (int kk = 0; kk < 2 * NHT; kk++) qt[dt & 1][kk] = lds_read<bf16x8>(ob + (4 * NHT + dt * 2 * NHT + kk) * 1024);
  };
  if (steps > 1) { DSA_WAIT_VMCNT(PER); } else { DSA_WAIT_VMCNT(0); }
  asm volatile("s_barrier" ::: "memory");
  unsigned ob = lds0 + (unsigned)(lane * 16);       // operands of the query in hand
#pragma unroll
  for (int t = 0; t < NHT; t++) {
    i32x8 aq[2];
    read_query(t, ob, aq);
    scores(t, aq);
  }
#pragma unroll
  for (int t = 0; t < NHT; t++)
#pragma unroll
    for (int j = 0; j < 8; j++) mk[0][2 * t + (j >> 2)][j & 3] = mask_pair(acc[t][2 * j], acc[t][2 * j + 1]);
  read_weighted(0, ob);
  float before = __builtin_bit_cast(float, UNSELECTED);        // factor of the query whose last d-tile is still to be added
  racc[1] = zero;
  // Scores and masks of the query behind the one in hand are made under the products of the latter (behind the last one: of what lies
  // in the ring, unused), and a query's last sums under the next one's first products.  FINITE: every operand of the chunk is; otherwise
  // infinities and NaN stay with the keys that the query selected.
  auto sweep = [&](auto finite) {
    constexpr bool FINITE = decltype(finite)::value;
    int slot = 0;
    for (int step = 0; step < steps; step++) {
      const int next_slot = slot + 1 < KEYS_STAGES ? slot + 1 : 0;
#pragma unroll
      for (int x = 0; x < 2; x++) {
        if (x == 1 && 2 * step + 1 >= n) break;
        if (x == 1 || 2 * step + 1 >= n) {          // the last query of the step: the next step's operands from here on
          // its transfers have landed, and every read of the step before this one has come back: its slot is filled next
          DSA_WAIT_VMCNT(0);
          asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
          if (step + 2 < steps) issue(slot >= 1 ? slot - 1 : KEYS_STAGES - 1);
          look_up(step + 3);
        }
        const unsigned on = x == 0 ? ob + OPS : lds0 + (unsigned)(next_slot * STAGE + lane * 16);
        const float a = lds_read<float>(lds0 + (unsigned)(slot * STAGE + 2 * OPS + wave * 256 + x * 128 + r * 4));
        // the products of a d-tile run while the one before it is added (the masks' entries are 2^-7)
        auto add = [&](int dt, int e, float f) {
          float v = racc[dt & 1][e];
          if (!FINITE) v = __builtin_bit_cast(unsigned, f) == UNSELECTED ? 0.f : v;
          sum[dt][e] = fmaf(f * 128.f, v, sum[dt][e]);
        };
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int dt = 0; dt < 4; dt++) {
          constexpr int STEP = 16 / (2 * NHT);
          i32x8 aq[2];
          read_weighted((dt + 1) & 3, dt < 3 ? ob : on);
          if (dt < NHT) read_query(dt, on, aq);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int kk = 0; kk < 2 * NHT; kk++) {
            racc[dt & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qt[dt & 1][kk], __builtin_bit_cast(bf16x8, mk[x][kk]), kk ? racc[dt & 1] : zero, 0, 0, 0);
#pragma unroll
            for (int e = STEP * kk; e < STEP * (kk + 1); e++) add(dt > 0 ? dt - 1 : 3, e, dt > 0 ? a : before);
            if (dt >= 2) {                          // (the scores were made by then)
#pragma unroll
              for (int i = 0; i < 2; i++) {
                const int j = 4 * NHT * (dt - 2) + 2 * kk + i, t = j >> 3;
                mk[x ^ 1][j >> 2][j & 3] = mask_pair(acc[t][2 * (j & 7)], acc[t][2 * (j & 7) + 1]);
              }
            }
            __builtin_amdgcn_sched_barrier(0);
          }
          if (dt < NHT) scores(dt, aq);
          __builtin_amdgcn_sched_barrier(0);
        }
        before = a;
        ob = on;
      }
      slot = next_slot;
    }
#pragma unroll
    for (int e = 0; e < 16; e++) {
      float v = racc[1][e];
      if (!FINITE) v = __builtin_bit_cast(unsigned, before) == UNSELECTED ? 0.f : v;
      sum[3][e] = fmaf(before * 128.f, v, sum[3][e]);
    }
  };
  if (bad) sweep(std::false_type()); else sweep(std::true_type());
  float* out = A.part + (((size_t)c * A.tiles + tile) * KT + 32 * wave + r) * D + 4 * g;
#pragma unroll
  for (int dt = 0; dt < 4; dt++)
#pragma unroll
    for (int j = 0; j < 4; j++)
      *(f32x4*)(out + 32 * dt + 8 * j) = f32x4{sum[dt][4 * j], sum[dt][4 * j + 1], sum[dt][4 * j + 2], sum[dt][4 * j + 3]};
}

// d_k8[key] (+)= the sums of the chunks that hold the key: 8 groups of 32 threads, chunk c in group c mod 8, the groups in a fixed order.
__global__ __launch_bounds__(256) void indexer_chunk_sum_kernel(const float* __restrict__ part, const int* __restrict__ used, int chunks, int tiles,
                                                                float* __restrict__ d_k8, int accumulate) {
  __shared__ f32x4 part_s[8][32];
  const int key = blockIdx.x, tile = key / KT, col = threadIdx.x & 31, grp = threadIdx.x >> 5;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  bool dup = false;
#pragma unroll 4
  for (int c = grp; c < chunks; c += 8) {
    const int n = used[(size_t)c * tiles + tile];
    dup |= n < 0;
    if (n > 0) acc += *(const f32x4*)(part + (((size_t)c * tiles + tile) * KT + key % KT) * D + 4 * col);
  }
  part_s[grp][col] = acc;
  dup = __syncthreads_or(dup);
  if (grp == 0) {
    f32x4 s = ((part_s[0][col] + part_s[1][col]) + (part_s[2][col] + part_s[3][col])) +
              ((part_s[4][col] + part_s[5][col]) + (part_s[6][col] + part_s[7][col]));
    float* p = d_k8 + (size_t)key * D + 4 * col;
    if (accumulate) s += *(const f32x4*)p;
    if (dup) s = f32x4{1.f, 1.f, 1.f, 1.f} * __builtin_nanf("");        // a query row held a repeated id: no sum that misses a term
    *(f32x4*)p = s;
  }
}

// Gradients of the keys' projection from the summed payload gradients: the same steps as for the queries, then back
// through the LayerNorm (fp32).  16 lanes per row; a workgroup takes every gridDim-th group of 16 rows and leaves its
// share of the LayerNorm's parameter gradients in part[block][2][128] (summed in block order by the next kernel).
// Bound by its chain of loads, 4 us a group of rows; up to 512 workgroups, one group each up to 8192 keys (with 128 of them 2077 keys
// 11 and now 7.3 us, 8192 keys 22.8 and 10.6; the parameters' sums behind it by 16 groups of threads for 4).
struct KeyArgs {
  const float* d_k8;
  const float* k_scale;
  int Sk;
  RowFinish fin;
  const int* positions;
  const unsigned short* k_in;            // bf16 input of the LayerNorm, or null
  const float* ln_w;
  float ln_eps;
  void* d_k; int k_f32, dim;
  float* part;
};
constexpr int KEY_BLOCKS = 512;

__device__ __forceinline__ float sum16(float v) {
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) v += __shfl_xor(v, o, 64);
  return v;
}

__global__ __launch_bounds__(256) void indexer_key_finish_kernel(const KeyArgs A) {
  __shared__ float red_s[2][16][D];
  const int sub = threadIdx.x & 15, grp = threadIdx.x >> 4;
  float lw[8], dlw[8], dlb[8];
#pragma unroll
  for (int i = 0; i < 8; i++) { lw[i] = A.k_in ? A.ln_w[8 * sub + i] : 0.f; dlw[i] = dlb[i] = 0.f; }
  for (int row0 = blockIdx.x * 16; row0 < A.Sk; row0 += gridDim.x * 16) {
    const int row = min(row0 + grp, A.Sk - 1);
    const bool live = row0 + grp < A.Sk;
    float v[8];
    const f32x4 p0 = *(const f32x4*)(A.d_k8 + (size_t)row * D + 8 * sub), p1 = *(const f32x4*)(A.d_k8 + (size_t)row * D + 8 * sub + 4);
#pragma unroll
    for (int i = 0; i < 4; i++) { v[i] = p0[i]; v[4 + i] = p1[i]; }
    finish_row(v, sub, A.k_scale[row], A.fin, A.positions, row, nullptr);
    if (A.k_in) {
      const uint4 raw = *(const uint4*)(A.k_in + (size_t)row * D + 8 * sub);
      const unsigned w[4] = {raw.x, raw.y, raw.z, raw.w};
      float x[8], dx[8];
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < 8; i++) {
        x[i] = (i & 1) ? __builtin_bit_cast(float, w[i >> 1] & 0xffff0000u) : __builtin_bit_cast(float, w[i >> 1] << 16);
        s += x[i];
      }
      const float mean = sum16(s) * (1.f / D);
      s = 0.f;
#pragma unroll
      for (int i = 0; i < 8; i++) { x[i] -= mean; s += x[i] * x[i]; }
      const float rstd = rsqrtf(sum16(s) * (1.f / D) + A.ln_eps);
      float m1 = 0.f, m2 = 0.f;
#pragma unroll
      for (int i = 0; i < 8; i++) {
        x[i] *= rstd;
        if (live) { dlw[i] += v[i] * x[i]; dlb[i] += v[i]; }
        dx[i] = v[i] * lw[i];
        m1 += dx[i];
        m2 += dx[i] * x[i];
      }
      m1 = sum16(m1) * (1.f / D);
      m2 = sum16(m2) * (1.f / D);
#pragma unroll
      for (int i = 0; i < 8; i++) v[i] = rstd * (dx[i] - m1 - x[i] * m2);
    }
    if (live) store_row(v, A.d_k, A.k_f32, row, A.dim, sub);
  }
  if (!A.k_in) return;
#pragma unroll
  for (int i = 0; i < 8; i++) { red_s[0][grp][8 * sub + i] = dlw[i]; red_s[1][grp][8 * sub + i] = dlb[i]; }
  __syncthreads();
  const int which = threadIdx.x >> 7, c = threadIdx.x & 127;
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < 16; k++) s += red_s[which][k][c];
  A.part[(size_t)blockIdx.x * 2 * D + threadIdx.x] = s;
}

constexpr int LN_GROUPS = 16;
__global__ __launch_bounds__(64 * LN_GROUPS) void indexer_ln_sum_kernel(const float* __restrict__ part, int blocks, float* __restrict__ d_w,
                                                                        float* __restrict__ d_b) {
  __shared__ float red_s[LN_GROUPS][64];
  const int c = blockIdx.x * 64 + (threadIdx.x & 63), grp = threadIdx.x >> 6;      // column of [2][128]
  float s = 0.f;
#pragma unroll 8
  for (int b = grp; b < blocks; b += LN_GROUPS) s += part[(size_t)b * 2 * D + c];
  red_s[grp][threadIdx.x & 63] = s;
  __syncthreads();
  if (grp == 0) {
    s = 0.f;
#pragma unroll
    for (int k = 0; k < LN_GROUPS; k++) s += red_s[k][threadIdx.x];
    if (c < D) d_w[c] = s; else d_b[c - D] = s;
  }
}

struct Plan {
  int chunk, W;
  size_t off_bitmap, off_prefix, off_count, off_start, off_flag, off_dst, off_rows, total;
};
size_t align_up(size_t x) { return (x + 255) & ~(size_t)255; }
Plan layout_plan(int chunk, int Sk, int K) {
  Plan p;
  p.chunk = chunk;
  p.W = (chunk + 31) / 32;
  size_t o = 0;
  p.off_bitmap = o; o = align_up(o + (size_t)Sk * p.W * 4);
  p.off_prefix = o; o = align_up(o + order::prefix_words(chunk, Sk) * 4);
  p.off_count = o; o = align_up(o + (size_t)(Sk + 1) * 4);
  p.off_start = o; o = align_up(o + (size_t)(Sk + 1) * 4);
  p.off_flag = o; o = align_up(o + 4);
  p.off_dst = o; o = align_up(o + (size_t)chunk * K * 4);
  p.off_rows = o; o = align_up(o + ((size_t)chunk * K + 1) * D * 2);
  p.total = o;
  return p;
}
Plan make_plan(int S, int Sk, int K, size_t budget) {
  int chunk = S;
  Plan p = layout_plan(chunk, Sk, K);
  while (p.total > budget && chunk > 64) {
    chunk = (chunk + 1) / 2;
    p = layout_plan(chunk, Sk, K);
  }
  return p;
}
constexpr size_t DEFAULT_BUDGET = (size_t)16 << 30;

struct DensePlan {
  int queries, tiles, words, chunk, chunks;          // queries of a sweep; key tiles; words of marks; queries of a chunk; chunks of a sweep
  float idle;                                        // workgroups of a sweep whose chunk has nothing in their tile
  size_t off_factors, off_marks, off_state, off_ops, off_part, off_used, total;
};
DensePlan dense_layout(int queries, int Hi, int Sk, int seen) {
  DensePlan p;
  p.queries = queries;
  p.tiles = dsa_cdiv(Sk, KT);
  p.words = dsa_cdiv(p.tiles, PIECE_TILES);
  // Queries of a chunk: rounds of 256 workgroups of 7 us and 1.2 us a query (0.65 with one head tile), against 128 KB of sums written and
  // read per workgroup.  Under a causal window a query sees half of `seen` in the mean, and half of a tile besides.  (Chunks of
  // 16 / 32 / 64 / 128, us of the whole call: 1000 queries x 256 slots 73 / 83 / 114 / 177, taken 16; 3072 x 512 of 768 keys
  // 158 / 143 / 170 / 231, 32; 8192 x 2048 1786 / 1505 / 1366 / 1369, 128.)  Beside these a chunk has a workgroup for each tile that it
  // does not touch, in packed sequences most of them, and they outgrow the others with the square of the tokens: without a price for
  // them 262 144 tokens in documents of 1024 x 256 slots take chunks of 24 and 92.6 ms, at 4 ns each chunks of 128 and 40.
  float best = INFINITY;
  for (int chunk : {4, 6, 8, 12, 16, 24, 32, 48, 64, 96, MAX_CHUNK}) {
    const float all = dsa_cdiv(queries, chunk) * (float)p.tiles, live = fminf(dsa_cdiv(queries, chunk) * (seen / (2.f * KT) + 0.5f), all);
    const float us = (live <= 160 ? 1.f : live / 256 + 0.6f) * (7 + chunk * (Hi <= 32 ? 0.65f : 1.2f)) + live * 0.058f + (all - live) * 0.004f;
    if (us < best) {
      best = us;
      p.chunk = chunk;
      p.idle = all - live;
    }
  }
  p.chunks = dsa_cdiv(queries, p.chunk);
  size_t o = 0;
  p.off_factors = o; o = align_up(o + (size_t)queries * p.tiles * KT * 4);
  p.off_marks = o; o = align_up(o + (size_t)queries * p.words * 4);
  p.off_state = o; o = align_up(o + (size_t)queries * 4);
  p.off_ops = o; o = align_up(o + (size_t)queries * operand_bytes(Hi / 32));
  p.off_part = o; o = align_up(o + (size_t)p.chunks * p.tiles * KT * D * 4);
  p.off_used = o; o = align_up(o + (size_t)p.chunks * p.tiles * 4);
  p.total = o;
  return p;
}
// The fewest sweeps over equal parts of the queries that fit the budget; less than 64 queries a sweep is no plan.
DensePlan dense_plan(int S, int Hi, int Sk, int seen, size_t budget) {
  DensePlan p = dense_layout(S, Hi, Sk, seen);
  for (int n = 2; p.total > budget && p.queries > 64; n++) p = dense_layout(dsa_cdiv(S, n), Hi, Sk, seen);
  return p;
}
// What the key tiles may take where the caller does not limit them: as much as the rows would, so that a call needs no more memory for
// being worked this way, or 2 GiB of the 288.  Their factors and sums are as wide as all keys, of which a packed sequence sees few: in one
// sweep 32 768 tokens in documents of 1024 x 256 slots would take 10.1 GiB where the rows take 2.3 (in five 1940 us, 1710 in one).
size_t dense_budget(int S, int Sk, int K) {
  const size_t rows = make_plan(S, Sk, K, DEFAULT_BUDGET).total, least = (size_t)2 << 30;
  return rows > least ? rows : least;
}
// Whether d_k8 is summed by key tiles, by prices in ns a query: the products with a key that the query sees 0.02 (one head tile 0.0104), a
// pair with a row of its own 0.076 more than in d_q8 alone, the key-sorted order's bits 0.00039 per key; the scattered factors and operands
// 2.3 more than the order's launches and 1.9 us a call; 8.6 ns a workgroup without work; 27 us a further sweep.  Fitted to 497 pairs of
// whole calls of 300-131 072 tokens in 1-16 documents, and of compressed keys, x 256-2048 slots: 0.2 % above the better way in the mean,
// 10 % at the worst (2700 x 256 in documents of 675).  us, rows / key tiles, 64 heads: 8192 queries x 2048 slots of a causal window 1822 / 1401,
// 12 000 x 1024 in documents of 4000 1492 / 1188, 3000 x 512 258 / 271, 6000 x 256 in documents of 1500 339 / 363, 8192 x 256 of 2048 compressed keys 445 / 475,
// 32 768 x 2048 in documents of 8192 7550 / 5540, 131 072 x 1024 in documents of 4096 23 800 / 17 900.
bool by_key_tiles(int S, int Hi, int Sk, int K, int seen_keys, const DensePlan& p) {
  const float seen = seen_keys, queries = S, sweeps = dsa_cdiv(S, p.queries);
  const float visible = queries < seen ? seen - 0.5f * queries : 0.5f * seen;       // the window of the last queries, or one that grows from nothing
  const float selected = queries < seen ? fminf(K, visible) : K < seen ? K - 0.5f * K * K / seen : visible;
  const float tiles = (Hi <= 32 ? 0.0104f : 0.02f) * (visible + 0.8f * KT) + 2.3f + (1900.f + 8.6f * sweeps * p.idle + 27000.f * (sweeps - 1)) / queries;
  return tiles < 0.076f * selected + 0.00039f * Sk;
}
constexpr int SPAN_ROWS = -1, SPAN_TILES = -2;       // the way as the caller says
// The way of a call and, if it is the key tiles, their plan.  The plan that a workspace of its own size gets is itself.
bool plan_key_tiles(int S, int Hi, int Sk, int K, int span, size_t budget, DensePlan* p) {
  if (S <= 0 || span == SPAN_ROWS) return false;
  const int seen = span > 0 && span < Sk ? span : Sk;
  if (span != SPAN_TILES) {
    const size_t most = dense_budget(S, Sk, K);
    if (budget > most) budget = most;
  }
  *p = dense_plan(S, Hi, Sk, seen, budget);
  return p->total <= budget && (span == SPAN_TILES || by_key_tiles(S, Hi, Sk, K, seen, *p));
}

}  // namespace

static size_t bwd_workspace(int S, int Hi, int Sk, int K, int span) {
  if (S <= 0 || Sk <= 0 || K <= 0) return 0;
  DensePlan p;
  if (plan_key_tiles(S, Hi <= 32 ? 32 : 64, Sk, K, span, DEFAULT_BUDGET, &p)) return p.total;
  return make_plan(S, Sk, K, DEFAULT_BUDGET).total;
}

extern "C" size_t dsa_indexer_bwd_workspace_bytes(int S, int Hi, int Sk, int K) { return bwd_workspace(S, Hi, Sk, K, 0); }

namespace {

// what dsa_indexer_grads asks for on top of the payload gradients
struct KeyFinish {
  KeyArgs key;
  float* d_ln_w;
  float* d_ln_b;
};

int finish_keys(const char* name, const KeyFinish* kf, int Sk, hipStream_t st) {
  if (!kf) return DSA_OK;
  const int blocks = dsa_cdiv(Sk, 16) < KEY_BLOCKS ? dsa_cdiv(Sk, 16) : KEY_BLOCKS;
  indexer_key_finish_kernel<<<dim3(blocks), dim3(256), 0, st>>>(kf->key);
  if (kf->key.k_in) indexer_ln_sum_kernel<<<dim3(4), dim3(64 * LN_GROUPS), 0, st>>>(kf->key.part, blocks, kf->d_ln_w, kf->d_ln_b);
  DSA_CHECK_LAUNCH("indexer_bwd(keys)");
  return DSA_OK;
}

int run_by_key_tiles(const char* name, BwdArgs A, const DensePlan& p, int S, int Hi, float* d_k8, const KeyFinish* kf, unsigned char* ws, hipStream_t st) {
  const int Sk = A.Sk, K = A.K;
  DenseArgs d = {};
  d.gsc = A.gsc; d.q8 = A.q8; d.k8 = A.k8; d.k_scale = A.k_scale; d.q_w = A.q_w; d.ids = A.ids;
  d.Sk = Sk; d.K = K;
  d.tiles = p.tiles; d.words = p.words; d.chunk = p.chunk;
  d.factors = (float*)(ws + p.off_factors);
  d.marks = (unsigned*)(ws + p.off_marks);
  d.state = (int*)(ws + p.off_state);
  d.ops = ws + p.off_ops;
  d.part = (float*)(ws + p.off_part);
  d.used = (int*)(ws + p.off_used);
  const size_t smem = bwd_lds_bytes(Hi, 2, K, false), smem_keys = Hi == 32 ? keys_lds_bytes<1>() : keys_lds_bytes<2>();
  auto scatter = Hi == 32 ? indexer_scatter_kernel<1> : indexer_scatter_kernel<2>;
  auto keys = Hi == 32 ? indexer_keys_kernel<1> : indexer_keys_kernel<2>;
  auto queries = Hi == 32 ? indexer_bwd_kernel<1, 2, false> : indexer_bwd_kernel<2, 2, false>;
  if (dsa_reserve_lds((const void*)queries, smem) != hipSuccess || dsa_reserve_lds((const void*)keys, smem_keys) != hipSuccess)
    DSA_FAIL(DSA_ERR_LAUNCH, "%s: cannot reserve LDS", name);
  for (int q0 = 0; q0 < S; q0 += p.queries) {
    d.q0 = A.q0 = q0;
    d.cnt = A.cnt = S - q0 < p.queries ? S - q0 : p.queries;
    d.chunks = dsa_cdiv(d.cnt, p.chunk);
    scatter<<<dim3(d.cnt), dim3(256), 0, st>>>(d);
    DSA_CHECK_LAUNCH("indexer_bwd(factors)");
    queries<<<dim3(d.cnt), dim3(THREADS / 2), smem, st>>>(A);
    DSA_CHECK_LAUNCH("indexer_bwd");
    keys<<<dim3(dsa_cdiv(d.chunks, 8) * 8 * p.tiles), dim3(THREADS), smem_keys, st>>>(d);
    DSA_CHECK_LAUNCH("indexer_bwd(key tiles)");
    indexer_chunk_sum_kernel<<<dim3(Sk), dim3(256), 0, st>>>(d.part, d.used, d.chunks, d.tiles, d_k8, q0 > 0);
    DSA_CHECK_LAUNCH("indexer_bwd(chunk sums)");
  }
  return finish_keys(name, kf, Sk, st);
}

int run_bwd(const char* name, BwdArgs A, int S, int Hi, int span, float* d_k8, const KeyFinish* kf, void* workspace, size_t workspace_bytes,
            void* stream) {
  const int Sk = A.Sk, K = A.K;
  DSA_REQUIRE(Hi == 32 || Hi == 64, "%s: head count must be 32 or 64, got %d", name, Hi);
  DSA_REQUIRE(S >= 0 && Sk > 0, "%s: bad sizes S=%d Sk=%d", name, S, Sk);
  DSA_REQUIRE(K > 0 && K % TK == 0 && K <= 4096, "%s: top-k must be a multiple of 128 up to 4096, got %d", name, K);
  DSA_REQUIRE((size_t)Sk * D <= 0xffffffffull, "%s: key array too large", name);
  DSA_REQUIRE(Sk <= order::MAX_KEYS, "%s: at most %d keys are supported, got %d", name, order::MAX_KEYS, Sk);
  DSA_REQUIRE(((uintptr_t)A.q8 % 16) == 0 && ((uintptr_t)A.k8 % 16) == 0 && ((uintptr_t)A.q_w % 16) == 0 &&
              ((uintptr_t)A.d_q8 % 16) == 0 && ((uintptr_t)A.d_q % 16) == 0 && ((uintptr_t)d_k8 % 16) == 0 && ((uintptr_t)workspace % 256) == 0,
              "%s: misaligned pointer", name);
  hipStream_t st = (hipStream_t)stream;
  DensePlan dense;
  if (workspace != nullptr && plan_key_tiles(S, Hi, Sk, K, span, workspace_bytes, &dense))
    return run_by_key_tiles(name, A, dense, S, Hi, d_k8, kf, (unsigned char*)workspace, st);
  Plan p = make_plan(S > 0 ? S : 1, Sk, K, workspace_bytes);
  if (p.total > workspace_bytes || workspace == nullptr)
    DSA_FAIL(DSA_ERR_WORKSPACE, "%s: workspace of %zu bytes is too small (need at least %zu)", name, workspace_bytes, layout_plan(64, Sk, K).total);
  unsigned char* ws = (unsigned char*)workspace;
  unsigned* bitmap = (unsigned*)(ws + p.off_bitmap);
  unsigned* prefix = (unsigned*)(ws + p.off_prefix);
  int* count = (int*)(ws + p.off_count);
  int* start = (int*)(ws + p.off_start);
  int* dup_flag = (int*)(ws + p.off_flag);
  int* dstp = (int*)(ws + p.off_dst);
  A.dst = dstp;
  A.rows = (unsigned short*)(ws + p.off_rows);
  A.dummy_row = p.chunk * K;
  const size_t smem = bwd_lds_bytes(Hi, bwd_stages(K), K, true);
  auto kern = bwd_stages(K) == 3 ? (Hi == 32 ? indexer_bwd_kernel<1, 3, true> : indexer_bwd_kernel<2, 3, true>)
                                 : (Hi == 32 ? indexer_bwd_kernel<1, 2, true> : indexer_bwd_kernel<2, 2, true>);
  if (dsa_reserve_lds((const void*)kern, smem) != hipSuccess) DSA_FAIL(DSA_ERR_LAUNCH, "%s: cannot reserve LDS", name);
  bool first = true;
  order::clear_flag(dup_flag, st);
  for (int q0 = 0; q0 < S; q0 += p.chunk) {
    A.q0 = q0;
    A.cnt = S - q0 < p.chunk ? S - q0 : p.chunk;
    // every id inside [0, Sk) counts: the causal window was already applied when the ids were selected
    order::build(A.ids, q0, A.cnt, K, Sk, 0x3fffffff, bitmap, prefix, count, start, dstp, p.W, order::Room{A.rows, p.total - p.off_rows}, st, dup_flag);
    DSA_CHECK_LAUNCH("indexer_bwd(order)");
    kern<<<dim3(A.cnt), dim3(THREADS), smem, st>>>(A);
    DSA_CHECK_LAUNCH("indexer_bwd");
    indexer_reduce_kernel<<<dim3(Sk), dim3(16 * RED_GROUPS), 0, st>>>(A.rows, start, d_k8, first ? 0 : 1, dup_flag);
    DSA_CHECK_LAUNCH("indexer_bwd(reduce)");
    first = false;
  }
  if (S == 0) order::zero_u32_kernel<<<dim3(256), dim3(256), 0, st>>>((unsigned*)d_k8, (size_t)Sk * D);
  return finish_keys(name, kf, Sk, st);
}

size_t grads_extra_bytes(int Sk) { return align_up((size_t)Sk * D * 4) + align_up((size_t)KEY_BLOCKS * 2 * D * 4); }

}  // namespace

extern "C" int dsa_indexer_bwd(const float* g, const void* q8, const void* k8, const float* k_scale, const float* q_w,
                               const int32_t* ids, int S, int Hi, int Sk, int K, float* d_q8, float* d_k8, float* d_qw,
                               void* workspace, size_t workspace_bytes, void* stream) {
  BwdArgs A = {};
  A.gsc = g; A.q8 = (const unsigned char*)q8; A.k8 = (const unsigned char*)k8; A.k_scale = k_scale; A.q_w = q_w; A.ids = ids;
  A.Sk = Sk; A.K = K; A.d_q8 = d_q8; A.d_qw = d_qw;
  return run_bwd("dsa_indexer_bwd", A, S, Hi, 0, d_k8, nullptr, workspace, workspace_bytes, stream);
}

extern "C" size_t dsa_indexer_grads_span_workspace_bytes(int S, int Hi, int Sk, int K, int span) {
  if (Sk <= 0 || K <= 0) return 0;
  return bwd_workspace(S > 0 ? S : 1, Hi, Sk, K, span) + grads_extra_bytes(Sk);
}
extern "C" size_t dsa_indexer_grads_workspace_bytes(int S, int Hi, int Sk, int K) { return dsa_indexer_grads_span_workspace_bytes(S, Hi, Sk, K, 0); }

extern "C" int dsa_indexer_grads(const float* g, const void* q8, const void* k8, const float* k_scale, const float* q_w,
                                 const int32_t* ids, int S, int Hi, int Sk, int K, const float* q_scale, float w_scale, int rotate,
                                 const void* cos, const void* sin, int tables_f32, int pairing, const int32_t* positions_q,
                                 const int32_t* positions_k, int batch, const void* k_in, const float* ln_w, float ln_eps,
                                 int heads, int dim, void* d_q, int q_f32, void* d_k, int k_f32, void* d_w, int w_f32,
                                 float* d_ln_w, float* d_ln_b, void* workspace, size_t workspace_bytes, void* stream) {
  return dsa_indexer_grads_span(g, q8, k8, k_scale, q_w, ids, S, Hi, Sk, K, 0, q_scale, w_scale, rotate, cos, sin, tables_f32, pairing,
                                positions_q, positions_k, batch, k_in, ln_w, ln_eps, heads, dim, d_q, q_f32, d_k, k_f32, d_w, w_f32, d_ln_w,
                                d_ln_b, workspace, workspace_bytes, stream);
}

extern "C" int dsa_indexer_grads_span(const float* g, const void* q8, const void* k8, const float* k_scale, const float* q_w,
                                      const int32_t* ids, int S, int Hi, int Sk, int K, int span, const float* q_scale, float w_scale, int rotate,
                                      const void* cos, const void* sin, int tables_f32, int pairing, const int32_t* positions_q,
                                      const int32_t* positions_k, int batch, const void* k_in, const float* ln_w, float ln_eps,
                                      int heads, int dim, void* d_q, int q_f32, void* d_k, int k_f32, void* d_w, int w_f32,
                                      float* d_ln_w, float* d_ln_b, void* workspace, size_t workspace_bytes, void* stream) {
  DSA_REQUIRE(heads > 0 && heads <= Hi && dim > 0 && dim <= D, "dsa_indexer_grads: %d heads of %d channels do not fit %d x %d", heads, dim, Hi, D);
  DSA_REQUIRE(q_scale != nullptr, "dsa_indexer_grads: q_scale is missing");
  DSA_REQUIRE(pairing < 0 || (cos != nullptr && sin != nullptr && pairing <= 1 && batch > 0), "dsa_indexer_grads: bad rotary arguments");
  DSA_REQUIRE(k_in == nullptr || (ln_w != nullptr && d_ln_w != nullptr && d_ln_b != nullptr), "dsa_indexer_grads: LayerNorm arguments are missing");
  DSA_REQUIRE(((uintptr_t)d_k % 16) == 0 && ((uintptr_t)k_in % 16) == 0, "dsa_indexer_grads: misaligned pointer");
  const size_t extra = grads_extra_bytes(Sk > 0 ? Sk : 1);
  if (workspace == nullptr || workspace_bytes < extra || ((uintptr_t)workspace % 256) != 0)
    DSA_FAIL(DSA_ERR_WORKSPACE, "dsa_indexer_grads: workspace of %zu bytes is too small or misaligned", workspace_bytes);
  float* d_k8 = (float*)workspace;
  BwdArgs A = {};
  A.gsc = g; A.q8 = (const unsigned char*)q8; A.k8 = (const unsigned char*)k8; A.k_scale = k_scale; A.q_w = q_w; A.ids = ids;
  A.Sk = Sk; A.K = K;
  A.q_scale = q_scale; A.w_scale = w_scale;
  A.fin = RowFinish{rotate == 2 && dim == 64 ? 2 : rotate != 0, cos, sin, tables_f32, pairing, batch};
  A.pos_q = positions_q; A.heads = heads; A.dim = dim;
  A.d_q = d_q; A.q_f32 = q_f32; A.d_w = d_w; A.w_f32 = w_f32;
  KeyFinish kf = {};
  kf.key = KeyArgs{d_k8, k_scale, Sk, A.fin, positions_k, (const unsigned short*)k_in, ln_w, ln_eps, d_k, k_f32, dim,
                   (float*)((unsigned char*)workspace + align_up((size_t)Sk * D * 4))};
  kf.d_ln_w = d_ln_w; kf.d_ln_b = d_ln_b;
  return run_bwd("dsa_indexer_grads", A, S, Hi, span, d_k8, &kf, (unsigned char*)workspace + extra, workspace_bytes - extra, stream);
}
