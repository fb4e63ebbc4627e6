// Sparse MQA-MLA attention forward for gfx950.
//
// The selected latent rows are gathered 32 at a time straight from global memory into LDS
// (global_load_lds, 16 B per lane) in a layout of nine 128-byte groups per key row with an XOR
// swizzle on the 16-byte slot, so both MFMA operand reads below are spread over the LDS banks:
//   S^T[key, head] = KV_tile . Q^T      36 x v_mfma_f32_32x32x16_bf16, A = KV rows from LDS
//                                         (ds_read_b128), B = the wave's Q slice held in registers
//   O^T[dv, head] += V_tile^T . P^T     32 x MFMA, A = LDS transpose reads (ds_read_b64_tr_b16),
//                                         B = the softmaxed S^T accumulators re-used in place
// With S^T a lane owns one head (column), so the online-softmax statistics are per lane and need
// one cross-lane exchange per tile; the accumulator layout of S^T is, up to a fixed permutation
// of the keys inside a tile, the B-operand layout of the second product, so P never touches LDS.
// MFMA-bound: 2*H*(576+512) flop per (query, key) pair against 1152 gathered bytes.
//
// How a workgroup shares a query's heads and slots is the MODE:
//   0  96 or 128 heads, one tile at a time: mla_fwd_wide_kernel, eight waves of up to 256 registers in two roles.
//   3  64 heads, one tile at a time, two workgroups on a compute unit: mla_fwd_half_kernel<2>; 128 heads with up to
//      256 slots as two groups of heads, and any heads with one pair of tiles.
//   4  32 heads, likewise: mla_fwd_half_kernel<1>.
//   1  64 heads, two tiles at a time: waves (stream, b) = (w / 2, w % 2) own heads [32b, 32b + 32)
//      of every other tile; the two streams' sums are merged through LDS at the end.
//   2  32 heads, two tiles at a time: waves (stream, b) compute S^T of the same heads and own half
//      of the value columns.
// Modes 1 and 2 are mla_fwd_kernel: four waves of up to 512 registers, one per SIMD.  They spend 68 / 52 matrix
// instructions per wave on two tiles and are then bound by the gather.  A query's heads may also be spread over several
// workgroups, and its slots over `ksplit` of them (few queries: one workgroup per query would leave most of the 256
// compute units idle); those write unnormalised fp32 sums that mla_fwd_combine_kernel puts together, or, of two ranges in
// modes 1 and 2, the second of their workgroups.
#include <atomic>
#include <chrono>
#include <type_traits>

#include "mla_tile.h"

// attn_dist.hip
int dsa_attn_dist_live(const void* logits, const int32_t* ids, int S, int H, int Skv, int K, int64_t ld_s, int q_start, float sm_scale,
                       float* target, hipStream_t st);

namespace {
using namespace mla;

constexpr int DTILES = DV / 32;              // 16

// S^T MFMAs are issued through inline asm so that their accumulator lives in architectural VGPRs:
// the 256 accumulation registers are exactly the O^T accumulators, and a 17th accumulator tuple
// there would force the register allocator to shuffle tuples between the two register files.
// Back-to-back MFMAs that accumulate into the same registers need no software wait states; the
// consumer of the finished chain does (mfma_chain_done).
__device__ __forceinline__ void mfma_first(f32x16& acc, const bf16x8& a, const bf16x8& b) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(acc) : "v"(a), "v"(b));
}
__device__ __forceinline__ void mfma_next(f32x16& acc, const bf16x8& a, const bf16x8& b) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(a), "v"(b));
}
__device__ __forceinline__ void mfma_chain_done(f32x16& acc) {
  // 8-pass MFMA result -> VALU read needs 11 wait states; leave a margin
  asm volatile("s_nop 15\n\ts_nop 3" : "+v"(acc));
}

struct FwdArgs {
  const __bf16* q; const __bf16* kv; const int* ids;
  __bf16* out; float* lse; void* p_out;
  int S, H, Skv, K, q_start;
  float sm_scale;
  const float* sink;
  int p_skip;
  bool p_all;                                // p_out: tiles without a valid slot are filled with -inf (else left as they are)
  int n_hg, ksplit, k_loc;                   // head groups per query, slot ranges per query, slots of a range
  int span;                                  // modes 1 - 4: neighbouring queries (ranges) on one XCD
  f32x4* part_o; float* part_ml;             // ksplit > 1: sums [S][ksplit][H/32][16][4][64] x 4, (m, l) [S][ksplit][H][2]
  unsigned long long *turn, token;           // two ranges that meet by themselves: [S][n_hg], else null; the call's number
};

// The softmax of a head is taken relative to a reference point, the maximum of the first tile, so the
// O^T accumulators are never rescaled (a rescaling branch in the loop, even one never taken, costs the
// register allocator hundreds of spills).  Where a later tile exceeds it by more than 2^64 (exp2 then nears
// the end of fp32) the wave marks its heads and they are done again relative to the true row maximum: by the workgroup itself behind its
// output, when its accumulators are free, or where the slots are in ranges by the kernel that sums those (the mark is a NaN with a
// payload in the range's statistics).  A kernel for it behind the ones with all slots in one workgroup took 4.5 us also when nothing
// was marked.
constexpr float REDO_ABOVE = 64.0f, REDO_TERM = 0x1p64f;
constexpr unsigned REDO_MARK = 0x7fc0d5a0u;
__device__ __forceinline__ bool is_marked(float x) { return __builtin_bit_cast(unsigned, x) == REDO_MARK; }

// The reference point from a maximum (base 2).  It stays finite where that is -inf: relative to -inf a term would be
// exp2(-inf + inf), while a row whose valid logits are all -inf has the sum 0, a zero output row and lse = +inf.
__device__ __forceinline__ float reference_point(float mx) { return fmaxf(mx, -1e30f); }

struct Final { float o_scale; float inv; float lse; };
// Denominator, output factor and natural-log lse of a head from its reference point m (base 2) and sum l.
// A sink logit is one more term exp(sink) in the denominator with no value row; the reference moves to
// max(m, sink) so that neither term can overflow.  A query without any valid slot gets lse = sink (+inf
// without a sink) and a zero output row.
__device__ __forceinline__ Final finish_head(float m, float l, const float* sink) {
  float o_scale = 1.0f;
  if (sink) {
    const float sk2 = *sink * LOG2E;
    const float nm = fmaxf(m, sk2);
    o_scale = exp2f(m - nm);
    l = l * o_scale + exp2f(sk2 - nm);
    m = nm;
  }
  Final f;
  f.o_scale = o_scale;
  f.inv = l > 0.f ? o_scale / l : 0.f;
  f.lse = l > 0.f ? (m + log2f(l)) * 0.6931471805599453f : INFINITY;
  return f;
}

__device__ __forceinline__ i16x4 read_tr(const unsigned char* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(i16x4, p));
}
__device__ __forceinline__ bf16x8 value_operand(const i16x4& lo, const i16x4& hi) {
  typedef short i16x8 __attribute__((ext_vector_type(8)));
  return __builtin_bit_cast(bf16x8, (i16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}
// maximum of a tile's logits for the lane's head (both half-waves)
__device__ __forceinline__ float tile_max(const f32x16& sacc) {
  float mx = sacc[0];
#pragma unroll
  for (int e = 1; e < 16; e++) mx = fmaxf(mx, sacc[e]);
  return fmaxf(mx, __shfl_xor(mx, 32, 64));
}
// P of a tile relative to `ref` (base 2) as the B operand of the second product; returns the lane's share of the sum
__device__ __forceinline__ float softmax_numerators(const f32x16& sacc, float c2, float ref, bf16x8 (&pb)[2]) {
  float psum = 0.f;
#pragma unroll
  for (int s = 0; s < 2; s++)
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const float pe = __builtin_amdgcn_exp2f(fmaf(sacc[8 * s + e], c2, -ref));
      psum += pe;
      pb[s][e] = (__bf16)pe;
    }
  return psum;
}
// one 32 x 32 block of O^T (lane = head): to the workspace as it lies, or normalised to the lane's output row
__device__ __forceinline__ void store_partial(const f32x16& t, f32x4* p) {
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const f32x4 v = {t[4 * j], t[4 * j + 1], t[4 * j + 2], t[4 * j + 3]};
    p[j * 64] = v;
  }
}
// The same in device scope: written through, for a workgroup on another XCD to read.  (Of assembly the compiler does not know that the data of
// such a store may be written again two wait states later: they are part of it.)
__device__ __forceinline__ void store_partial_through(const f32x16& t, f32x4* p) {
  f32x4 v[4];
#pragma unroll
  for (int j = 0; j < 4; j++) v[j] = f32x4{t[4 * j], t[4 * j + 1], t[4 * j + 2], t[4 * j + 3]};
  asm volatile("global_store_dwordx4 %0, %1, off sc1\n\tglobal_store_dwordx4 %0, %2, off offset:1024 sc1\n\t"
               "global_store_dwordx4 %0, %3, off offset:2048 sc1\n\tglobal_store_dwordx4 %0, %4, off offset:3072 sc1\n\ts_nop 1"
               :: "v"(p), "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]) : "memory");
}
__device__ __forceinline__ void store_out(const f32x16& t, float scale, unsigned short* p) {   // all lanes of the wave
  uint4 o[2];
  acc_row_to_16B(t, scale, o);
  *(uint4*)p = o[0];
  *(uint4*)(p + 16) = o[1];
}
// One 32-head block of a query relative to the true maximum of every head, all slots, one tile at a time: every
// wave computes S^T of the block and sums its own value column tile dt.  For the marked blocks only: simple, and
// light on registers and LDS (one tile, the ids) so that the kernels that carry it stay small.  tid: the thread's number among 256; a
// second half of 512 threads stages and gathers the same again.
template <bool COUNTED>                      // tid is counted anew; else it is threadIdx.x, of 256
__device__ __forceinline__ void redo_block(const FwdArgs& a, int qi, int hb, int dt, f32x16& acc, float& m, float& l, int tid) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int lane = tid & 63, r = lane & 31, g = lane >> 5;
  const int NT = a.K / BI;
  int* idx_s = (int*)(smem + TILE_BYTES);
  unsigned* tmask = (unsigned*)(idx_s + a.K);
  int* tlist = (int*)(tmask + NT);
  __syncthreads();
  int ntiles;
  if constexpr (COUNTED) {
    const int* const ids = a.ids + (size_t)qi * a.K;
    int first[8];
    request_first_ids(ids, 0, a.K, first, tid);
    stage_requested(first, ids, a.K, a.Skv, a.q_start + qi, idx_s, tmask, tid);
    __syncthreads();
    if (tid < 64) list_tiles(NT, tmask, tlist, tlist + NT, tid);
    __syncthreads();
    ntiles = tlist[NT];
  } else {
    ntiles = stage_ids(a.ids, qi, a.K, a.Skv, a.q_start + qi, idx_s, tmask, tlist, tlist + NT);
  }
  const LaneOffsets lo = lane_offsets(tid);
  const bf16x8* qp = (const bf16x8*)(a.q + ((size_t)qi * a.H + hb * 32 + r) * DQK) + g;
  const float c2 = a.sm_scale * LOG2E;
  unsigned v_off[2][2];                      // the wave's value columns: lo.tr_off[s][t][dt & 1]
#pragma unroll
  for (int s = 0; s < 2; s++)
#pragma unroll
    for (int t = 0; t < 2; t++)
      v_off[s][t] = (unsigned)((dt >> 1) * GRP_BYTES) + lo.tr_off[s][t][0] + (unsigned)(dt & 1) * (lo.tr_off[s][t][1] - lo.tr_off[s][t][0]);
  m = -1e30f;
  l = 0.f;
#pragma unroll
  for (int e = 0; e < 16; e++) acc[e] = 0.f;
#pragma unroll 1
  for (int step = 0; step < 2 * ntiles; step++) {            // first sweep: the maximum; second: the sums
    const int tile = tlist[step < ntiles ? step : step - ntiles];
    __syncthreads();
    gather_tile(a.kv, idx_s, tile, (unsigned)(uintptr_t)smem, tid);
    DSA_WAIT_VMCNT(0);
    __syncthreads();
    f32x16 sacc;
#pragma unroll
    for (int e = 0; e < 16; e++) sacc[e] = 0.f;
#pragma unroll 1
    for (int c = 0; c < KSTEPS / 4; c++)
#pragma unroll
      for (int j = 0; j < 4; j++)
        sacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8*)(smem + c * GRP_BYTES + lo.row_off[j]),
                                                       qp[2 * (4 * c + j)], sacc, 0, 0, 0);
    const unsigned mg = tmask[tile] >> (4 * g);
#pragma unroll
    for (int e = 0; e < 16; e++)
      if (!((mg >> (8 * (e >> 2) + (e & 3))) & 1u)) sacc[e] = -INFINITY;
    if (step < ntiles) {
      m = fmaxf(m, tile_max(sacc) * c2);
    } else {
      bf16x8 pb[2];
      l += softmax_numerators(sacc, c2, m, pb);
#pragma unroll
      for (int s = 0; s < 2; s++)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            value_operand(read_tr(smem + v_off[s][0]), read_tr(smem + v_off[s][1])), pb[s], acc, 0, 0, 0);
    }
  }
  l += __shfl_xor(l, 32, 64);
}

__device__ __forceinline__ void write_block(const FwdArgs& a, int qi, int hb, int dt, const f32x16& acc, float m, float l, int tid) {
  const int lane = tid & 63, r = lane & 31, g = lane >> 5;
  const int h = hb * 32 + r;
  const Final fin = finish_head(m, l, a.sink ? a.sink + h : nullptr);
  if (dt == 0 && g == 0) a.lse[(size_t)qi * a.H + h] = fin.lse;
  store_out(acc, fin.inv, (unsigned short*)a.out + ((size_t)qi * a.H + h) * DV + 32 * dt + 8 * g);
}

// The marked ones (bit hb) of a query's head blocks again, by all WAVES waves of the workgroup.
template <int WAVES>
__device__ __forceinline__ void redo_marked(const FwdArgs& a, int qi, unsigned marked, int wave, int lane) {
  const int tid = (wave & 3) * 64 + lane;
#pragma unroll 1
  while (marked) {
    const int hb = __builtin_ctz(marked);
    marked &= marked - 1;
#pragma unroll 1
    for (int dt = wave; dt < DTILES; dt += WAVES) {
      f32x16 acc;
      float m, l;
      redo_block<true>(a, qi, hb, dt, acc, m, l, tid);
      write_block(a, qi, hb, dt, acc, m, l, tid);
    }
  }
}

// The lane counted anew, for what follows the loop over the tiles to hold no register through it.
__device__ __forceinline__ int lane_again() { return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }

// Workgroup -> (unit, head group), a unit being a query, or a slot range of one.  The head groups of a unit gather the same rows:
// they sit eight workgroups apart, i.e. on the same XCD and its L2.  So do `span` neighbouring units: the drafted tokens of a
// sequence have most of their keys in common.
__device__ __forceinline__ int unit_of(const FwdArgs& a, int block, int& hg) {
  const unsigned i = (unsigned)block >> 3, j = i / (unsigned)a.n_hg, t = j / (unsigned)a.span;
  hg = __builtin_amdgcn_readfirstlane(i - j * a.n_hg);
  return __builtin_amdgcn_readfirstlane((t * 8 + (block & 7)) * a.span + (j - t * a.span));
}

template <int MODE, bool SPLIT, int POUT>    // MODE 1, 2; SPLIT: ksplit > 1; POUT: 0 none, 1 bf16, 2 f32
__global__ __launch_bounds__(256, 1) void mla_fwd_kernel(FwdArgs a) {
  constexpr int NDT = MODE == 2 ? DTILES / 2 : DTILES;      // value column tiles of a wave
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, g = lane >> 5;
  const int stream = wave >> 1, sub = wave & 1;
  const int S = a.S, H = a.H, K = a.K, p_skip = a.p_skip;
  const int units = S * (SPLIT ? a.ksplit : 1);              // longest prefixes first, range by range
  int hg;
  const int u = unit_of(a, (int)blockIdx.x, hg);
  if (u >= units) return;
  const int qi = S - 1 - (SPLIT ? u % S : u);
  const int sp = SPLIT ? u / S : 0;
  const int qpos = a.q_start + qi;
  const int k0 = sp * a.k_loc;
  const int KL = min(a.k_loc, K - k0), NT = KL / BI;         // slots and tiles of this range
  const int tile0 = k0 / BI;
  const int hb = MODE == 1 ? 2 * hg + sub : hg;              // 32-head block of the wave

  constexpr int RING = 4 * TILE_BYTES;       // the two tiles at work, the two on their way
  int* idx_s = (int*)(smem + RING);
  unsigned* tmask = (unsigned*)(idx_s + KL);
  int* tlist = (int*)(tmask + NT);
  int* ntile_s = tlist + NT;

  // ---- The ids and Q of the workgroup's heads, requested together so that both come back in one round trip to memory: Q as
  // 32-head blocks in the tiles' layout, where tiles 2 and 3 will lie.  The ids first, so that the list is made and the first tiles start
  // while Q arrives: 200 queries x 32 heads x 512 slots 27.5 -> 26.2 us.  A range of a query is short, its Q comes with it, and there Q
  // goes first (61 queries x 64 heads in two ranges 24.9 us, 25.3 the other way). ----------
  const int* const ids = a.ids + (size_t)qi * K + k0;
  int first[8];
  if (!SPLIT) request_first_ids(ids, 0, KL, first);
  __builtin_amdgcn_sched_barrier(0);
  const unsigned lds0 = (unsigned)(uintptr_t)smem;
  const int h = hb * 32 + r;
  const bool head_ok = h < H;
#pragma unroll
  for (int b = 0; b < (MODE == 1 ? 2 : 1); b++)
    gather_rows(a.q + ((size_t)qi * H + min((MODE == 1 ? 2 * hg + b : hg) * 32, H - 32)) * DQK, lds0 + (unsigned)((2 + b) * TILE_BYTES));
  __builtin_amdgcn_sched_barrier(0);

  // ---- stage the ids, mark valid slots, list the tiles that have any ---------------------
  if (SPLIT) request_first_ids(ids, 0, KL, first);
  const int ntiles = stage_from_first_ids(first, ids, 0, KL, a.Skv, qpos, idx_s, tmask, tlist, ntile_s);
  const int nsteps = (ntiles + 1) / 2;

  // slots of tiles that are never visited still need their -inf in p_out
  // (p_out holds the slots from p_skip on: its rows are K - p_skip wide)
  if (POUT != 0 && a.p_all && head_ok && ntiles < NT) {
    for (int t = 0; t < NT; t++) {
      if (tmask[t] != 0u || (tile0 + t) * BI < p_skip || (t & 1) != stream) continue;
      const size_t pbase = ((size_t)qi * H + h) * (K - p_skip) + (size_t)((tile0 + t) * BI - p_skip) + 16 * g;
      if (POUT == 2) {
        const f32x4 ninf = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
        for (int j = 0; j < 4; j++) *(f32x4*)((float*)a.p_out + pbase + 4 * j) = ninf;
      } else {
        const uint4 ninf = make_uint4(0xff80ff80u, 0xff80ff80u, 0xff80ff80u, 0xff80ff80u);
#pragma unroll
        for (int j = 0; j < 2; j++) *(uint4*)((unsigned short*)a.p_out + pbase + 8 * j) = ninf;
      }
    }
  }

  // ---- gather of tile n of the list into ring slot n % 4; lane-dependent LDS offsets ----
  auto issue = [&](int n) {
    gather_tile(a.kv, idx_s, tlist[min(n, ntiles - 1)], lds0 + (unsigned)((n % 4) * TILE_BYTES));
  };
  // The same gather in single steps (one 128-byte group of the key rows of a tile each), issued between
  // MFMAs: nine transfers in a row hold the wave until the memory pipeline has taken them all (about 520
  // clocks per tile of 4200).
  // (An odd tile count: the last tile is gathered twice and masked out in the second stream.)
  unsigned g_goff[2], g_lb[2];
  auto gather_prepare = [&](int n0) {
#pragma unroll
    for (int s = 0; s < 2; s++) {
      const int n = n0 + s;
      const int gkey = tid >> 3, gsub = tid & 7;
      int kid = idx_s[tlist[min(n, ntiles - 1)] * BI + gkey];
      kid = kid < 0 ? 0 : kid;
      g_goff[s] = (unsigned)kid * (DQK * 2) + (unsigned)((gsub ^ swz(gkey)) * 16);
      g_lb[s] = __builtin_amdgcn_readfirstlane(lds0 + (unsigned)((n % 4) * TILE_BYTES + wave * 1024));
    }
  };
  auto gather_step = [&](int s, int grp) {
    dma16(g_lb[s] + grp * GRP_BYTES, g_goff[s] + grp * 128, a.kv);
  };
  const LaneOffsets lo = lane_offsets();
  const unsigned (&qk_off)[4] = lo.row_off;          // A operand of S^T: row r, 16-byte chunk 2*ks + g
  const unsigned (&pv_off)[2][2][2] = lo.tr_off;     // A operand of O^T: transpose reads, [s][t][dt & 1]

  const float c2 = a.sm_scale * LOG2E;
  float m_ref = -1e30f, l_run = 0.f;
  bf16x8 qreg[KSTEPS];                               // the wave's Q slice, B operand of S^T = KV . Q^T
  f32x16 oacc[NDT];

  // S^T of the tile in stage buffer tb.  Operand reads run four k-steps ahead of the MFMAs; the
  // scheduling fences keep that order (and with it the register budget: Q slice 144 + O^T
  // accumulators 256 of 512 per lane).
  auto qk_tile = [&](const unsigned char* tb, unsigned mask, f32x16& sacc, bool gather) {
    bf16x8 f[4];
#pragma unroll
    for (int ks = 0; ks < 4; ks++) f[ks] = *(const bf16x8*)(tb + (ks >> 2) * GRP_BYTES + qk_off[ks & 3]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ks++) {
      if (ks == 0) mfma_first(sacc, f[0], qreg[0]);
      else mfma_next(sacc, f[ks & 3], qreg[ks]);
      if (ks + 4 < KSTEPS) f[ks & 3] = *(const bf16x8*)(tb + ((ks + 4) >> 2) * GRP_BYTES + qk_off[ks & 3]);
      if (ks % 2 == 1 && gather) gather_step((ks / 2) / 9, (ks / 2) % 9);     // all 18 of the next two tiles
      __builtin_amdgcn_sched_barrier(0);
    }
    mfma_chain_done(sacc);
    // accumulator e of this lane is key 8*(e/4) + 4*g + (e%4) of the tile
    if (mask != 0xffffffffu) {
      const unsigned mg = mask >> (4 * g);
#pragma unroll
      for (int e = 0; e < 16; e++)
        if (!((mg >> (8 * (e >> 2) + (e & 3))) & 1u)) sacc[e] = -INFINITY;
    }
  };

#pragma unroll
  for (int dt = 0; dt < NDT; dt++) {
#pragma unroll
    for (int e = 0; e < 16; e++) oacc[dt][e] = 0.f;
  }
  for (int n = 0; n < 2 && n < 2 * nsteps; n++) issue(n);
  if (nsteps > 0) { DSA_WAIT_VMCNT(18); }
  else { DSA_WAIT_VMCNT(0); }
  __syncthreads();
  {
    const unsigned char* qb = smem + (2 + (MODE == 1 ? sub : 0)) * TILE_BYTES;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ks++) {
      qreg[ks] = *(const bf16x8*)(qb + (ks >> 2) * GRP_BYTES + qk_off[ks & 3]);
      asm volatile("" : "+v"(qreg[ks]));
    }
  }
  bool overflow = false;
  int stores_after = 0;                      // p_out stores a wave issued after the transfers it waits for
  for (int step = 0; step < nsteps; step++) {
    if (POUT != 0 && stores_after == 4) { DSA_WAIT_VMCNT(4); }
    else if (POUT != 0 && stores_after == 2) { DSA_WAIT_VMCNT(2); }
    else { DSA_WAIT_VMCNT(0); }
    __syncthreads();
    const int next0 = 2 * (step + 1);
    const bool more = next0 < ntiles;
    if (more) gather_prepare(next0);
    const int n = 2 * step + stream;
    const bool real = n < ntiles;
    const int tile = tlist[real ? n : ntiles - 1];
    const unsigned mask = real ? tmask[tile] : 0u;
    const unsigned char* tb = smem + (n % 4) * TILE_BYTES;

    f32x16 sacc;
    qk_tile(tb, mask, sacc, more);
    stores_after = 0;
    if (POUT != 0 && head_ok && real && (tile0 + tile) * BI >= p_skip) {
      const size_t prow = ((size_t)qi * H + h) * (K - p_skip) + (size_t)((tile0 + tile) * BI - p_skip);
      if (POUT == 2) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
          f32x4 v = {sacc[4 * j], sacc[4 * j + 1], sacc[4 * j + 2], sacc[4 * j + 3]};
          if (MODE != 2 || (j >> 1) == sub) *(f32x4*)((float*)a.p_out + prow + 4 * g + 8 * j) = v;
        }
      } else {
        // A lane holds keys 8j + 4g .. +3 of its head (j = 0..3): 8-byte pieces.  The two half-waves
        // trade pieces so that each lane ends up with 8 consecutive keys, twice: 16-byte stores.
        uint4 o[2];
        acc_row_to_16B(sacc, 1.0f, o);
        if (MODE != 2 || sub == 0) *(uint4*)((unsigned short*)a.p_out + prow + 8 * g) = o[0];
        if (MODE != 2 || sub == 1) *(uint4*)((unsigned short*)a.p_out + prow + 16 + 8 * g) = o[1];
      }
      stores_after = POUT == 2 ? (MODE == 2 ? 2 : 4) : (MODE == 2 ? 0 : 2);
    }

    // ---- softmax numerators (base 2), one head per lane -----------------------------------
    {
      const float mx = tile_max(sacc) * c2;
      if (step == 0) m_ref = reference_point(mx);     // (a masked-out tile has the maximum -inf)
      overflow |= (mx > m_ref + REDO_ABOVE);
    }
    bf16x8 pb[2];
    l_run += softmax_numerators(sacc, c2, m_ref, pb);
    __builtin_amdgcn_sched_barrier(0);

    // ---- O^T += V^T . P^T -----------------------------------------------------------------
    {
      const unsigned char* vb = tb + (MODE == 2 ? sub * (NDT / 2) * GRP_BYTES : 0);     // the wave's value columns
      i16x4 v[2][2][2];   // [ring][s][t]
#pragma unroll
      for (int dt = 0; dt < 2; dt++)
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
          for (int t = 0; t < 2; t++)
            v[dt][s][t] = read_tr(vb + (dt >> 1) * GRP_BYTES + pv_off[s][t][dt & 1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int dt = 0; dt < NDT; dt++) {
#pragma unroll
        for (int s = 0; s < 2; s++)
          oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(value_operand(v[dt & 1][s][0], v[dt & 1][s][1]), pb[s], oacc[dt], 0, 0, 0);
        if (dt + 2 < NDT) {
#pragma unroll
          for (int s = 0; s < 2; s++)
#pragma unroll
            for (int t = 0; t < 2; t++)
              v[dt & 1][s][t] = read_tr(vb + ((dt + 2) >> 1) * GRP_BYTES + pv_off[s][t][dt & 1]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  float l_tot = l_run + __shfl_xor(l_run, 32, 64);
  bool again = __ballot(overflow) != 0ull;   // the same for all lanes of a wave

  // ---- two streams: their sums are merged through the (now free) tile ring, scaled to the common reference point.  Each stream's
  // wave sends the other's half of the column tiles and finishes its own, so that all four waves store: with the second stream's
  // sums all sent to the first, two waves stored the 131 KB of 64 heads while two had ended. ---------------------------------
  __syncthreads();                         // the last tiles and the id arrays have been read
  static_assert(2 * NDT * 4096 + 1024 + 16 <= RING, "the hand-over fits the tile ring");
  float* ml = (float*)(smem + 2 * NDT * 4096);             // [stream][sub][32][2], behind the waves' boxes
  if (g == 0) {
    ml[((stream * 2 + sub) * 32 + r) * 2] = again ? __builtin_bit_cast(float, REDO_MARK) : m_ref;
    ml[((stream * 2 + sub) * 32 + r) * 2 + 1] = l_tot;
  }
  constexpr int HALF = NDT / 2;
  auto box_of = [&](int to) { return (f32x4*)(smem + (size_t)((to * 2 + sub) * HALF) * 4096) + lane; };
  auto send = [&](auto first, int to) {
    f32x4* const box = box_of(to);
#pragma unroll
    for (int i = 0; i < HALF; i++) store_partial(oacc[decltype(first)::value + i], box + i * 256);
  };
  if (stream == 0) send(std::integral_constant<int, HALF>{}, 1);
  else send(std::integral_constant<int, 0>{}, 0);
  unsigned* const marked_s = (unsigned*)(ml + 256);        // mode 1: the head blocks to be done again
  __syncthreads();
  const float m_o = ml[(((stream ^ 1) * 2 + sub) * 32 + r) * 2], l_o = ml[(((stream ^ 1) * 2 + sub) * 32 + r) * 2 + 1];
  again |= is_marked(m_o);
  if (MODE == 2 && !SPLIT && again) {      // the same for all waves: they have the same heads
#pragma unroll 1
    for (int dt = wave; dt < DTILES; dt += 4) {
      f32x16 acc;
      float m, l;
      redo_block<false>(a, qi, hb, dt, acc, m, l, tid);
      write_block(a, qi, hb, dt, acc, m, l, tid);
    }
    return;
  }
  // the first stream's terms first on both sides: a head's denominator has the same bits in both of its waves
  const float nm = fmaxf(m_ref, m_o);
  const float f_own = __builtin_amdgcn_exp2f(m_ref - nm), f_other = __builtin_amdgcn_exp2f(m_o - nm);
  const float f0 = stream == 0 ? f_own : f_other, f1 = stream == 0 ? f_other : f_own;
  l_tot = fmaf(stream == 0 ? l_tot : l_o, f0, (stream == 0 ? l_o : l_tot) * f1);
  m_ref = nm;

  // ---- epilogue: the wave's column tiles, normalised to out[i,h,:] with lse[i,h], or as they are to the workspace ----
  const bool stats = stream == 0 && g == 0 && (MODE != 2 || sub == 0);
  const int dt0 = MODE == 2 ? sub * NDT : 0;
  auto finish = [&](auto first, auto write) {              // column tiles `first` .. of the wave's, both streams
    constexpr int FIRST = decltype(first)::value;
    const f32x4* const box = box_of(FIRST == 0 ? 0 : 1);
#pragma unroll
    for (int i = 0; i < HALF; i++) {
      f32x16 t;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const f32x4 v = box[(i * 4 + j) * 64];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float own = oacc[FIRST + i][4 * j + e];
          t[4 * j + e] = FIRST == 0 ? fmaf(own, f0, v[e] * f1) : fmaf(v[e], f0, own * f1);
        }
      }
      write(t, FIRST + i);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto finish_mine = [&](auto write) {
    if (stream == 0) finish(std::integral_constant<int, 0>{}, write);
    else finish(std::integral_constant<int, HALF>{}, write);
  };
  if (SPLIT) {
    if (!head_ok && !a.turn) return;         // the same for all lanes of a wave
    const size_t range_ml = (size_t)H * 2, range_o = (size_t)(H / 32) * DTILES * 256;
    float* const part_ml = a.part_ml + ((size_t)qi * a.ksplit * H + h) * 2;
    f32x4* const po = a.part_o + (((size_t)qi * a.ksplit * (H / 32) + hb) * DTILES + dt0) * 256 + lane;
    if (head_ok) {
      if (stats) {
        __hip_atomic_store(part_ml + sp * range_ml, again ? __builtin_bit_cast(float, REDO_MARK) : m_ref, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(part_ml + sp * range_ml + 1, l_tot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      if (!again) finish_mine([&](const f32x16& t, int dt) {
        if (a.turn) store_partial_through(t, po + sp * range_o + dt * 256);
        else store_partial(t, po + sp * range_o + dt * 256);
      });
    }
    if (!a.turn) return;
    // Two ranges: the workgroup that is second to have its sums in memory puts both together.  Whatever the word of the pair held, it
    // holds the call's number once the first has been there.
    unsigned* const second_s = marked_s + 2;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // (a barrier alone does not wait for other waves' stores)
    __syncthreads();
    if (tid == 0) {
      unsigned long long* const word = a.turn + (size_t)qi * a.n_hg + hg;
      const bool second = __hip_atomic_exchange(word, a.token, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == a.token;
      if (second) *word = 0;                 // (the number comes again where a captured launch is replayed)
      *second_s = second;
    }
    __syncthreads();
    if (!__builtin_amdgcn_readfirstlane(*second_s)) return;
    asm volatile("" ::: "memory");
    if (head_ok) {
      const float m_x = __hip_atomic_load(part_ml + (sp ^ 1) * range_ml, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const float l_x = __hip_atomic_load(part_ml + (sp ^ 1) * range_ml + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      again |= is_marked(m_x);               // the same for all heads of a block
      if (!again) {
        const f32x4* const px = po + (sp ^ 1) * range_o;
        const float top = fmaxf(m_ref, m_x), e_own = __builtin_amdgcn_exp2f(m_ref - top), e_x = __builtin_amdgcn_exp2f(m_x - top);
        // the first range's terms first, as mla_fwd_combine_kernel has them
        const Final fin = finish_head(top, sp == 0 ? fmaf(l_x, e_x, l_tot * e_own) : fmaf(l_tot, e_own, l_x * e_x), a.sink ? a.sink + h : nullptr);
        if (stats) a.lse[(size_t)qi * H + h] = fin.lse;
        unsigned short* op = (unsigned short*)a.out + ((size_t)qi * H + h) * DV + 32 * dt0 + 8 * g;
        constexpr int AHEAD = MODE == 1 ? 2 : 4;     // column tiles of the other range on their way
        f32x4 x[AHEAD][4];
        const int first_dt = stream == 0 ? 0 : HALF;
        auto request = [&](int i) {
#pragma unroll
          for (int j = 0; j < 4; j++) {
            const unsigned long long* p8 = (const unsigned long long*)(px + (first_dt + i) * 256 + j * 64);
            const unsigned long long lo = __hip_atomic_load(p8, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), hi = __hip_atomic_load(p8 + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
            x[i % AHEAD][j] = __builtin_bit_cast(f32x4, (u64x2{lo, hi}));
          }
        };
#pragma unroll
        for (int i = 0; i < AHEAD; i++) request(i);
        finish_mine([&](const f32x16& t, int dt) {
          const int i = dt % HALF;
          f32x16 o;
#pragma unroll
          for (int j = 0; j < 4; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
              const float own = t[4 * j + e], y = x[i % AHEAD][j][e];
              o[4 * j + e] = sp == 0 ? fmaf(y, e_x, own * e_own) : fmaf(own, e_own, y * e_x);
            }
          if (i + AHEAD < HALF) request(i + AHEAD);
          store_out(o, fin.inv, op + 32 * dt);
        });
      }
    }
    if (MODE == 2) {
      if (again) {
#pragma unroll 1
        for (int dt = wave; dt < DTILES; dt += 4) {
          f32x16 acc;
          float m, l;
          redo_block<false>(a, qi, hb, dt, acc, m, l, tid);
          write_block(a, qi, hb, dt, acc, m, l, tid);
        }
      }
      return;
    }
  } else if (head_ok && !again) {
    const Final fin = finish_head(m_ref, l_tot, a.sink ? a.sink + h : nullptr);
    if (stats) a.lse[(size_t)qi * H + h] = fin.lse;
    unsigned short* op = (unsigned short*)a.out + ((size_t)qi * H + h) * DV + 32 * dt0 + 8 * g;
    finish_mine([&](const f32x16& t, int dt) { store_out(t, fin.inv, op + 32 * dt); });
  }
  if (MODE == 1) {
    if (stream == 1 && lane == 0) marked_s[sub] = again && head_ok;
    __syncthreads();
    const unsigned marked = __builtin_amdgcn_readfirstlane(marked_s[0] | (marked_s[1] << 1));
    if (marked) redo_marked<4>(a, qi, marked << (2 * hg), wave, lane_again());
  }
}

// ---------------------------------------------------------------------------------------------
// 128 heads: eight waves of up to 256 registers, two per SIMD, in two roles.
//
// Wave w < 4 makes the scores of heads 32 w ..: S^T of a tile (the Q slice, 144 registers, stays in place), the softmax, P to
// LDS.  Wave 4 + w sums value columns 128 w .. of all heads, one tile behind, and issues the transfers.  So one wave's softmax,
// transfers and waits pass under the other's matrix instructions; a wave that did both, alone on its SIMD, left the matrix
// pipe idle for 1700 of the 3900 cycles a tile took.  Splitting the values by columns and not by heads also feeds four products from a
// transposed operand instead of one: 16 such reads a tile and wave instead of 64, for 8 reads of P.  The value sums of four head
// blocks and 128 columns are 256 registers; three of the sixteen 32 x 32 blocks (heads 0 .. 95, the last 32 columns) therefore live
// in the scores' waves, which leaves 208 + 40 there and 144 + 48 + 32 here.  Accumulators and the first half of Q sit in
// accumulation registers, the rest in architectural ones.
// Measured with 8192 queries and 2048 slots, cycles a tile: scores 1350, softmax 630, their share of the values 440; the other
// role transfers 640, products 1900: near 2650 in all, 2176 of them matrix instructions; LDS (77 reads a tile on each SIMD,
// and the arriving tile) is close behind.  Forward 3.70 -> 3.33 ms, with the logits 4.39 -> 3.97; 1500 queries behind
// a long prefix 809 -> 715 us.  Transfers spread over the products instead of first in the step: products
// 2550 cycles (a transfer holds the wave, and the operand reads behind it); wave priorities: no difference.
//
// Set-up: the scores' waves bring the first 5 of 9 column groups of Q by whole lines through LDS, where tiles 1 and 2 and P will be, and
// load the rest in the operands' layout, which takes 32 bytes of each of 32 rows and keeps the address path busy for four times as long a
// byte; meanwhile the other waves make the list of tiles and start tile 0.  With all of Q in the operands' layout and the list made by all
// waves, i.e. behind the issue of those loads, the first scores of a query started 16 800 cycles after it, now 11 600, of 198 000 in all at
// 8192 queries x 2048 slots.  The forward there is held by the power it takes (2.40 ms with zeros for data, at full clock), so that
// cycles saved are time saved in part: 3.41 -> 3.36 ms on one card, 3.51 -> 3.49 on another; 96 queries in ranges 72.3 -> 70.8 us, 1300 x
// 512 with logits 239.0 -> 234.7, 600 x 128 heads 327 -> 323, 600 x 96 heads, whose fourth wave has nothing to load, 319 -> 308.  Output rows
// by whole lines through LDS as well: no difference (one wave of a SIMD rounds 13 of its 16 blocks, which takes as long as the stores did).
// ---------------------------------------------------------------------------------------------
constexpr int WIDE_RING = 3;                 // tiles: the values of n, the scores of n + 1, the transfers of n + 2
constexpr int P_BYTES = 4 * 2 * 1024;        // P of a tile, [32-head block][16 keys][lane] of 16 bytes
constexpr int WIDE_LDS = WIDE_RING * TILE_BYTES + 2 * P_BYTES;
constexpr int Q_ACC = 18;                    // k-steps of the Q slice in accumulation registers
constexpr int Q_GROUPS = 5;                  // 128-byte groups of the rows of Q that pass through LDS, behind tile 0
static_assert(TILE_BYTES + 4 * Q_GROUPS * GRP_BYTES <= WIDE_LDS, "Q lies where tiles 1 and 2 and P will be");

// -> the head blocks to be done again (bit hb) and, where there are any, 16 times the wave's number
template <bool SCORES, bool SPLIT, int POUT>
__device__ __forceinline__ unsigned wide_body(const FwdArgs& a, int qi, int sp, unsigned char* smem) {
  const int lane = threadIdx.x & 63, r = lane & 31, g = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3);
  const int H = a.H, K = a.K;
  const int k0 = sp * a.k_loc;
  const int KL = min(a.k_loc, K - k0), NT = KL / BI;
  unsigned char* const pbuf = smem + WIDE_RING * TILE_BYTES;
  int* idx_s = (int*)(smem + WIDE_LDS);
  unsigned* tmask = (unsigned*)(idx_s + KL);
  int* tlist = (int*)(tmask + NT);
  float* const inv_s = (float*)pbuf;         // after the last tile
  unsigned* const marked_s = (unsigned*)(inv_s + 128);
  unsigned marked = 0;
  auto marked_blocks = [&] {
    return (unsigned)__builtin_amdgcn_readfirstlane(marked_s[0] | (marked_s[1] << 1) | (marked_s[2] << 2) | (marked_s[3] << 3));
  };

  const int* const ids = a.ids + (size_t)qi * K + k0;
  const int h = 32 * w + r;                  // of the scores
  const bool head_ok = h < H;                // the same for all lanes of a wave
  const unsigned row0 = (unsigned)(r * 128 + ((g ^ swz(r)) << 4));       // chunk 2 j + g of a group: row0 ^ 32 j
  bf16x8 qreg[SCORES ? KSTEPS : 1];
  const unsigned q_lds = (unsigned)(uintptr_t)smem + TILE_BYTES + w * Q_GROUPS * GRP_BYTES;
  int first[8];
  if constexpr (SCORES) {
    const unsigned char* const base = (const unsigned char*)uniform_ptr(a.q + ((size_t)qi * H + 32 * w) * DQK);
#pragma unroll
    for (int i = 0; i < 4 && head_ok; i++) { // rows 8 i .. of the wave's heads
      const int row = 8 * i + (lane >> 3);
      const unsigned src = (unsigned)(row * (DQK * 2) + ((lane & 7) ^ swz(row)) * 16);
#pragma unroll
      for (int p = 0; p < Q_GROUPS; p++) dma16(__builtin_amdgcn_readfirstlane(q_lds + p * GRP_BYTES + i * 1024), src + p * 128, base);
    }
  } else {
    request_first_ids(ids, 0, KL, first, threadIdx.x & 255);
    stage_requested(first, ids, KL, a.Skv, a.q_start + qi, idx_s, tmask, threadIdx.x & 255);
  }
  __syncthreads();
  if (!SCORES && w == 0) list_tiles(NT, tmask, tlist, tlist + NT, (int)threadIdx.x);
  __syncthreads();
  const int ntiles = tlist[NT];
  if constexpr (SCORES) {
    if (head_ok) {
      const bf16x8* qp = (const bf16x8*)(a.q + ((size_t)qi * H + h) * DQK) + g;
#pragma unroll
      for (int ks = 4 * Q_GROUPS; ks < KSTEPS; ks++) qreg[ks] = qp[2 * ks];
      __builtin_amdgcn_sched_barrier(0);
      DSA_WAIT_VMCNT(KSTEPS - 4 * Q_GROUPS); // the wave's own rows are in LDS
      asm volatile("" ::: "memory");
#pragma unroll
      for (int ks = 0; ks < 4 * Q_GROUPS; ks++)
        qreg[ks] = *LDS_PTR(const bf16x8, (uintptr_t)(((q_lds + row0) ^ (32 * (ks & 3))) + (ks >> 2) * GRP_BYTES));
    } else {                                 // 96 heads: nothing of this wave's scores is used
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ks++) qreg[ks] = bf16x8{};
    }
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ks++) {
      if (ks < Q_ACC) asm volatile("" : "+a"(qreg[ks]));
      else asm volatile("" : "+v"(qreg[ks]));
    }
  }
  if constexpr (SCORES) {
    const int tile0 = k0 / BI, p_skip = a.p_skip;
    // slots of tiles that are never visited still need their -inf in p_out
    // (p_out holds the slots from p_skip on: its rows are K - p_skip wide)
    if (POUT != 0 && a.p_all && head_ok && ntiles < NT) {
      for (int t = 0; t < NT; t++) {
        if (tmask[t] != 0u || (tile0 + t) * BI < p_skip) continue;
        const size_t pbase = ((size_t)qi * H + h) * (K - p_skip) + (size_t)((tile0 + t) * BI - p_skip) + 16 * g;
        if (POUT == 2) {
          const f32x4 ninf = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
          for (int j = 0; j < 4; j++) *(f32x4*)((float*)a.p_out + pbase + 4 * j) = ninf;
        } else {
          const uint4 ninf = make_uint4(0xff80ff80u, 0xff80ff80u, 0xff80ff80u, 0xff80ff80u);
#pragma unroll
          for (int j = 0; j < 2; j++) *(uint4*)((unsigned short*)a.p_out + pbase + 8 * j) = ninf;
        }
      }
    }
    const float c2 = a.sm_scale * LOG2E;
    float m_ref = -1e30f, l_run = 0.f;
    bool overflow = false;
    f32x16 o[3];                             // value columns 128 w + 96 .. of heads 0 .. 95
#pragma unroll
    for (int hb = 0; hb < 3; hb++) {
#pragma unroll
      for (int e = 0; e < 16; e++) o[hb][e] = 0.f;
      asm volatile("" : "+a"(o[hb]));
    }
    f32x16 s_acc;
    auto chain = [&](unsigned tb) {
      bf16x8 f[4];
      const unsigned tb0 = tb + row0;
      auto row = [&](int ks) { return *LDS_PTR(const bf16x8, (uintptr_t)((tb0 ^ (32 * (ks & 3))) + (ks >> 2) * GRP_BYTES)); };
#pragma unroll
      for (int ks = 0; ks < 4; ks++) f[ks] = row(ks);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ks++) {
        if (ks == 0) mfma_v_va_first(s_acc, f[0], qreg[0]);
        else if (ks < Q_ACC) mfma_v_va(s_acc, f[ks & 3], qreg[ks]);
        else mfma_v_vv(s_acc, f[ks & 3], qreg[ks]);
        if (ks + 4 < KSTEPS) f[ks & 3] = row(ks + 4);
        __builtin_amdgcn_sched_barrier(0);
      }
      mfma_done_v(s_acc);
    };
    auto soft = [&](int n, int tile, unsigned mask) {        // the chain's tile n of the list: p_out, statistics, P to LDS
      // accumulator e of this lane is key 8*(e/4) + 4*g + (e%4) of the tile
      if (mask != 0xffffffffu) {
        const unsigned mg = mask >> (4 * g);
#pragma unroll
        for (int e = 0; e < 16; e++)
          if (!((mg >> (8 * (e >> 2) + (e & 3))) & 1u)) s_acc[e] = -INFINITY;
      }
      if (POUT != 0 && head_ok && (tile0 + tile) * BI >= p_skip) {
        const size_t prow = ((size_t)qi * H + h) * (K - p_skip) + (size_t)((tile0 + tile) * BI - p_skip);
        if (POUT == 2) {
#pragma unroll
          for (int j = 0; j < 4; j++) {
            f32x4 v = {s_acc[4 * j], s_acc[4 * j + 1], s_acc[4 * j + 2], s_acc[4 * j + 3]};
            *(f32x4*)((float*)a.p_out + prow + 4 * g + 8 * j) = v;
          }
        } else {
          // A lane holds keys 8j + 4g .. +3 of its head (j = 0..3): 8-byte pieces.  The two half-waves
          // trade pieces so that each lane ends up with 8 consecutive keys, twice: 16-byte stores.
          uint4 t[2];
          acc_row_to_16B(s_acc, 1.0f, t);
          *(uint4*)((unsigned short*)a.p_out + prow + 8 * g) = t[0];
          *(uint4*)((unsigned short*)a.p_out + prow + 16 + 8 * g) = t[1];
        }
      }
      if (n == 0) m_ref = reference_point(tile_max(s_acc) * c2);
      bf16x8 pb[2];
      const float sum = softmax_numerators(s_acc, c2, m_ref, pb);
      l_run += sum;
      overflow |= sum > REDO_TERM;           // one of the terms, or a few just below
      bf16x8* const p = (bf16x8*)(pbuf + (n & 1) * P_BYTES + w * 2048) + lane;
      p[0] = pb[0];
      p[64] = pb[1];
    };
    unsigned tr0[2];                         // transposed reads of value columns 128 w + 96 .., [t]; 16 keys on: + 2048
    { const LaneOffsets lo = lane_offsets(); tr0[0] = lo.tr_off[0][0][1]; tr0[1] = lo.tr_off[0][1][1]; }
    auto values = [&](int n, int slot) {
      const unsigned char* vb = smem + slot * TILE_BYTES + (2 * w + 1) * GRP_BYTES;
      const bf16x8* const p = (const bf16x8*)(pbuf + (n & 1) * P_BYTES) + lane;
      bf16x8 v[2], pr[2][3];
#pragma unroll
      for (int s = 0; s < 2; s++) {
        v[s] = value_operand(read_tr(vb + tr0[0] + 2048 * s), read_tr(vb + tr0[1] + 2048 * s));
#pragma unroll
        for (int hb = 0; hb < 3; hb++) pr[s][hb] = p[hb * 128 + s * 64];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < 2; s++)
#pragma unroll
        for (int hb = 0; hb < 3; hb++) mfma_a_vv(o[hb], v[s], pr[s][hb]);
    };
    __syncthreads();                         // tile 0 has landed, Q is in registers
    int slot = -1;                           // of tile n
    if (ntiles > 0) {
      int tile_v = tlist[0];
#pragma clang loop unroll(disable)
      for (int n = -1; n < ntiles; n++) {
        asm volatile("" : "+s"(n));          // one copy of the body: a peeled one costs registers
        const int next = slot == WIDE_RING - 1 ? 0 : slot + 1;
        const int tile = tile_v;
        const unsigned mask = tmask[tile_v];
        tile_v = tlist[min(n + 2, ntiles - 1)];
        const unsigned tb = (unsigned)(uintptr_t)smem + next * TILE_BYTES;
        if (n >= 0) values(n, slot);
        if (n + 1 < ntiles) {
          chain(tb);
          soft(n + 1, __builtin_amdgcn_readfirstlane(tile), __builtin_amdgcn_readfirstlane(mask));
        }
        slot = next;
        __syncthreads();
      }
    }
    const float l_tot = l_run + __shfl_xor(l_run, 32, 64);
    const bool again = __ballot(overflow) != 0ull;
    if (SPLIT) {
      if (head_ok && g == 0) {
        float* const part_ml = a.part_ml + (((size_t)qi * a.ksplit + sp) * H + h) * 2;
        part_ml[0] = again ? __builtin_bit_cast(float, REDO_MARK) : m_ref;
        part_ml[1] = l_tot;
      }
    } else {
      const Final fin = finish_head(m_ref, l_tot, a.sink && head_ok ? a.sink + h : nullptr);
      if (head_ok && g == 0 && !again) a.lse[(size_t)qi * H + h] = fin.lse;
      if (g == 0) inv_s[h] = fin.inv;
      if (lane == 0) marked_s[w] = again && head_ok;
    }
    __syncthreads();
    if (!SPLIT) marked = marked_blocks();
#pragma unroll
    for (int hb = 0; hb < 3; hb++) {
      mfma_done_a(o[hb]);
      if (32 * hb < H && !((marked >> hb) & 1)) {
        const int dt = 4 * w + 3;
        if (SPLIT) store_partial(o[hb], a.part_o + ((((size_t)qi * a.ksplit + sp) * (H / 32) + hb) * DTILES + dt) * 256 + lane);
        else store_out(o[hb], inv_s[32 * hb + r], (unsigned short*)a.out + ((size_t)qi * H + 32 * hb + r) * DV + 32 * dt + 8 * g);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
    const LaneOffsets lo = lane_offsets();
    const unsigned lds0 = (unsigned)(uintptr_t)smem;
    const int gkey = (threadIdx.x & 255) >> 3, gsub = lane & 7;
    const unsigned gsl = (unsigned)((gsub ^ swz(gkey)) * 16);
    auto gather = [&](int n, int slot) {     // tile n of the list
      const unsigned goff = (unsigned)max(idx_s[tlist[n] * BI + gkey], 0) * (DQK * 2) + gsl;
      const unsigned lb = lds0 + slot * TILE_BYTES + w * 1024;
#pragma unroll
      for (int grp = 0; grp < 9; grp++) dma16(lb + grp * GRP_BYTES, goff + grp * 128, a.kv);
    };
    f32x16 oa[2][4], ov[4], o3;              // value columns 128 w + 32 i of head block hb: i = 0, 1; i = 2; i = 3, the last block
#pragma unroll
    for (int hb = 0; hb < 4; hb++) {
#pragma unroll
      for (int e = 0; e < 16; e++) oa[0][hb][e] = oa[1][hb][e] = ov[hb][e] = o3[e] = 0.f;
      asm volatile("" : "+a"(oa[0][hb]), "+a"(oa[1][hb]));
      asm volatile("" : "+v"(ov[hb]));
    }
    asm volatile("" : "+v"(o3));
    if (ntiles > 0) gather(0, 0);
    DSA_WAIT_VMCNT(0);
    __syncthreads();
#pragma unroll
    for (int n = 1; n < WIDE_RING; n++)
      if (n < ntiles) gather(n, n);
    if (ntiles > 0) {
      if (ntiles >= 3) { DSA_WAIT_VMCNT(9); }
      else { DSA_WAIT_VMCNT(0); }
      __syncthreads();
      int slot = 0;
#pragma clang loop unroll(disable)
      for (int n = 0; n < ntiles; n++) {
        const int before = slot == 0 ? WIDE_RING - 1 : slot - 1;
        if (n > 0 && n + 2 < ntiles) gather(n + 2, before);
        const unsigned char* vb = smem + slot * TILE_BYTES + 2 * w * GRP_BYTES;
        const bf16x8* const pp = (const bf16x8*)(pbuf + (n & 1) * P_BYTES) + lane;
        auto read_v = [&](int u) {           // unit u = 4 s + i
          const unsigned char* b = vb + ((u & 3) >> 1) * GRP_BYTES;
          return value_operand(read_tr(b + lo.tr_off[u >> 2][0][u & 1]), read_tr(b + lo.tr_off[u >> 2][1][u & 1]));
        };
        bf16x8 p[4], v[2];
#pragma unroll
        for (int hb = 0; hb < 4; hb++) p[hb] = pp[hb * 128];
        v[0] = read_v(0);
        v[1] = read_v(1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 8; u++) {
          const int i = u & 3;
          if (i < 2) {
#pragma unroll
            for (int hb = 0; hb < 4; hb++) mfma_a_vv(oa[i][hb], v[u & 1], p[hb]);
          } else if (i == 2) {
#pragma unroll
            for (int hb = 0; hb < 4; hb++) mfma_v_vv(ov[hb], v[u & 1], p[hb]);
          } else {
            mfma_v_vv(o3, v[u & 1], p[3]);
          }
          if (u + 2 < 8) v[u & 1] = read_v(u + 2);
          if (u == 2) {
#pragma unroll
            for (int hb = 0; hb < 3; hb++) p[hb] = pp[hb * 128 + 64];
          }
          if (u == 3) p[3] = pp[3 * 128 + 64];
          __builtin_amdgcn_sched_barrier(0);
        }
        slot = slot == WIDE_RING - 1 ? 0 : slot + 1;
        DSA_WAIT_VMCNT(0);                   // tile n + 2 has landed
        __syncthreads();
      }
    }
    __syncthreads();                         // the heads' factors
    if (!SPLIT) marked = marked_blocks();
    auto store = [&](const f32x16& t, int hb, int i) {
      if (32 * hb >= H || ((marked >> hb) & 1)) return;
      const int dt = 4 * w + i;
      if (SPLIT) store_partial(t, a.part_o + ((((size_t)qi * a.ksplit + sp) * (H / 32) + hb) * DTILES + dt) * 256 + lane);
      else store_out(t, inv_s[32 * hb + r], (unsigned short*)a.out + ((size_t)qi * H + 32 * hb + r) * DV + 32 * dt + 8 * g);
    };
#pragma unroll
    for (int hb = 0; hb < 4; hb++) {
      mfma_done_a(oa[0][hb]);
      store(oa[0][hb], hb, 0);
      mfma_done_a(oa[1][hb]);
      store(oa[1][hb], hb, 1);
      mfma_done_v(ov[hb]);
      store(ov[hb], hb, 2);
      __builtin_amdgcn_sched_barrier(0);
    }
    mfma_done_v(o3);
    store(o3, 3, 3);
  }
  return marked ? marked | (unsigned)(w + (SCORES ? 0 : 4)) << 4 : 0;
}

template <bool SPLIT, int POUT>
__global__ __launch_bounds__(512, 2) void mla_fwd_wide_kernel(FwdArgs a) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  // Longest prefixes first, but for the first round.  us, in strict order / spread over K / over 4 K queries: with logits 1300 x 512 slots 223 /
  // 199 / 211, 5000 x 1024 in five documents 928 / 893 / 900, 8192 x 2048 4006 / 3949 / 3973; without them the same within 1 %.
  const int u = (int)blockIdx.x;
  const int qi = a.S - 1 - (SPLIT ? u / a.ksplit : spread_start(u, a.S, 256, a.K)), sp = SPLIT ? u % a.ksplit : 0;
  unsigned marked;
  if (threadIdx.x < 256) marked = wide_body<true, SPLIT, POUT>(a, qi, sp, smem);
  else marked = wide_body<false, SPLIT, POUT>(a, qi, sp, smem);
  if (!SPLIT && marked) redo_marked<8>(a, qi, marked & 15, marked >> 4, lane_again());
}

// ---------------------------------------------------------------------------------------------
// 64 or 32 heads and more queries than compute units: four waves of up to 256 registers, two workgroups on a compute unit.
//
// With one workgroup of 512 registers a lane on a compute unit (mode 1) nothing fills what a query spends outside its tiles - Q, ids,
// the hand-over between the streams, the output: 12 us of the 31 that 640 slots took - nor a wave's softmax and transfers.  Here
// wave w has the scores of 16 heads (16x16x32 products: 72 registers of Q) and the value columns 128 w .. of all 64 (128
// accumulation registers), P passes through LDS, and a workgroup takes 79 KB: two tiles, P, and of the slot list only the masks,
// so that the longest one fits; the ids are read again a tile ahead of the transfers.  While one workgroup waits the other one works.
// Cycles a tile, two workgroups at work: transfers 740, scores 1440 (36 row reads of LDS for 576 matrix cycles), softmax
// 360, values 840, waits 330: bound by LDS, 56 reads a wave and tile, and by the gather where the keys lie far apart (65536 keys: no
// gain over mode 1).  3072 queries x 640 slots 372 -> 303 us (with the logits), 2048 x 512 220 -> 175, 3072 x 2048 1005 -> 940.
// 32 heads: a wave has the scores of 16 heads and one half of a tile's keys; 3000 queries x 640 slots 288 -> 216 us, x 2048 747 -> 575,
// 1024 x 256 62 -> 45 (against mode 2).
// ---------------------------------------------------------------------------------------------
constexpr int HALF_P = 4096;                 // P of a tile, [32-head block][16 keys][lane] of 16 bytes
constexpr int HALF_LDS = 2 * TILE_BYTES + HALF_P;
constexpr int HALF_AHEAD = 6;                // row reads in flight
__host__ __device__ inline size_t mask_lds_bytes(int K) { return (size_t)(K / BI) * 8 + 16; }
static_assert(HALF_LDS + 8192 / BI * 8 + 16 <= 80 * 1024, "two workgroups on a compute unit at the longest list");
static_assert(TILE_BYTES + 8192 * 4 + 8192 / BI * 8 + 16 <= HALF_LDS, "a tile and the ids of a block done again");

// The tiles' slot function with bit 0 of the row alone below: 16 rows x 4 chunks (an operand of 16x16x32) and the transposed
// reads of lane_offsets are both free of bank conflicts.
__device__ __forceinline__ int swz16(int r) { return (((r >> 1) & 1) << 2) | (((r >> 2) & 1) << 1) | (r & 1); }

// stage_ids without the ids: the masks and the list of the tiles that have a valid slot
// (v: the first eight loads of a thread, requested ahead of the operands as in request_first_ids: 2077 queries x 512 slots x 64 heads with
// logits 145 -> 142 us)
__device__ __forceinline__ void request_mask_ids(const int* __restrict__ ids, int K, int t0, int (&v)[8]) {
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = ids[min(t0 + i * 256, K - 64) + (int)(threadIdx.x & 63)];    // (under its condition each would be waited for by itself)
}
__device__ __forceinline__ int stage_masks(int (&v)[8], const int* __restrict__ ids, int K, unsigned limit, unsigned* tmask, int* tlist, int* ntile_s) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int NT = K / BI;
  for (int t0 = wave * 64; t0 < K; t0 += 8 * 256) {          // eight loads in flight
    if (t0 >= 8 * 256) request_mask_ids(ids, K, t0, v);
    asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]));
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const unsigned long long b = __ballot((unsigned)v[i] < limit);
      if (lane == 0 && t0 + i * 256 < K) {
        tmask[(t0 + i * 256) / BI] = (unsigned)b;
        tmask[(t0 + i * 256) / BI + 1] = (unsigned)(b >> 32);
      }
    }
  }
  __syncthreads();
  if (wave == 0) list_tiles(NT, tmask, tlist, ntile_s, lane);
  __syncthreads();
  return *ntile_s;
}

template <int HB, int POUT>                // HB 32-head blocks of a workgroup: 2, or 1
__global__ __launch_bounds__(256, 2) void mla_fwd_half_kernel(FwdArgs a) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  constexpr int KS = DQK / 32;               // 18 k-steps of 32
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 15, kg = lane >> 4;   // scores: head m of the wave's 16, keys 4 kg .. + 3 of each half tile
  const int hw = HB == 2 ? w : w & 1;        // its 16 heads; one block: it has half tile w / 2 alone, the other one is in wave w ^ 2
  const int h0 = HB == 2 ? 0 : w >> 1;       // its first half tile
  const int r = lane & 31, g = lane >> 5;    // values: head r of a block of 32
  const int S = a.S, H = a.H, K = a.K, p_skip = a.p_skip;

  int hg;
  const int u = unit_of(a, (int)blockIdx.x, hg);     // longest prefixes first
  if (u >= S) return;
  const int qi = S - 1 - u;
  const int NT = K / BI;
  // valid ids are below: none for a query in front of the keys (a negative bound would be a huge one here), and no sum past INT_MAX
  const int qpos = a.q_start + qi;
  const unsigned limit = qpos < 0 ? 0u : (unsigned)min(a.Skv - 1, qpos) + 1u;

  unsigned char* const pbuf = smem + 2 * TILE_BYTES;
  unsigned* tmask = (unsigned*)(smem + HALF_LDS);
  int* tlist = (int*)(tmask + NT);

  const int h = 32 * HB * hg + 16 * hw + m;  // of the scores
  const bool head_ok = 32 * HB * hg + 16 * hw < H;           // the same for all lanes of a wave
  const int* const row_ids = a.ids + (size_t)qi * K;
  int first[8];
  request_mask_ids(row_ids, K, w * 64, first);
  __builtin_amdgcn_sched_barrier(0);
  bf16x8 qreg[KS];
  {
    const bf16x8* qp = (const bf16x8*)(a.q + ((size_t)qi * H + (head_ok ? h : m)) * DQK) + kg;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) qreg[ks] = qp[4 * ks];
  }
  __builtin_amdgcn_sched_barrier(0);
  const int ntiles = stage_masks(first, row_ids, K, limit, tmask, tlist, tlist + NT);
#pragma unroll
  for (int ks = 0; ks < KS; ks++) asm volatile("" : "+v"(qreg[ks]));

  // slots of tiles that are never visited still need their -inf in p_out
  // (p_out holds the slots from p_skip on: its rows are K - p_skip wide)
  if (POUT != 0 && a.p_all && head_ok && h0 == 0 && ntiles < NT) {
    for (int t = 0; t < NT; t++) {
      if (tmask[t] != 0u || t * BI < p_skip) continue;
      const size_t pbase = ((size_t)qi * H + h) * (K - p_skip) + (size_t)(t * BI - p_skip) + 8 * kg;
      if (POUT == 2) {
        const f32x4 ninf = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
        for (int j = 0; j < 2; j++) *(f32x4*)((float*)a.p_out + pbase + 4 * j) = ninf;
      } else {
        *(uint4*)((unsigned short*)a.p_out + pbase) = make_uint4(0xff80ff80u, 0xff80ff80u, 0xff80ff80u, 0xff80ff80u);
      }
    }
  }

  // ---- transfers: thread (key = tid / 8, sub = tid % 8) moves slot `sub` of each of the 9 groups.  The ids come from memory,
  // a tile ahead of the transfers that need them: beside two tiles LDS has no room for those of a long list ----
  const unsigned lds0 = (unsigned)(uintptr_t)smem;
  const int gkey = tid >> 3;
  const unsigned gsl = (unsigned)(((tid & 7) ^ swz16(gkey)) * 16);
  auto id_of = [&](int n) { return row_ids[tlist[min(n, ntiles - 1)] * BI + gkey]; };
  auto offset_of = [&](int id) { return ((unsigned)id < limit ? (unsigned)id : 0u) * (DQK * 2) + gsl; };
  auto gather = [&](unsigned goff, int slot) {
    const unsigned lb = __builtin_amdgcn_readfirstlane(lds0 + (unsigned)(slot * TILE_BYTES + w * 1024));
#pragma unroll
    for (int grp = 0; grp < 9; grp++) dma16(lb + grp * GRP_BYTES, goff + grp * 128, a.kv);
  };

  // operand A of the scores: key 16 hh + m, chunk 4 (ks % 2) + kg of group ks / 2; hh: + 2048 (the slot function repeats after 8 rows)
  const unsigned row0 = (unsigned)(2048 * h0 + m * 128 + ((kg ^ swz16(m)) << 4));
  // transposed reads of a value tile, as in lane_offsets with this kernel's slots: keys 16 s + 8 t + 4 g .. + 3; s: + 2048, t: + 1024
  unsigned tr0;
  {
    const int blk = lane >> 4, ii = lane & 15;
    const int key = 4 * g + (ii >> 2), cl = 2 * (blk & 1) + ((ii & 3) >> 1);
    tr0 = (unsigned)(key * 128 + ((cl ^ swz16(key)) << 4) + (ii & 1) * 8);             // odd column tile of a group: ^ 64
  }
  const float c2 = a.sm_scale * LOG2E;
  // l_run: sum of the numerators, for lse.  w_run: of the same rounded to bf16, which are what the values are summed with: an output
  // normalised by it keeps of a numerator's rounding only the part along (value - output), 3 - 7 % less error in all.
  float m_ref = -1e30f, l_run = 0.f, w_run = 0.f;
  bool overflow = false;
  f32x16 o[4][HB];                           // value columns 128 w + 32 i of head block hb
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int hb = 0; hb < HB; hb++) {
#pragma unroll
      for (int e = 0; e < 16; e++) o[i][hb][e] = 0.f;
      asm volatile("" : "+a"(o[i][hb]));
    }
  const unsigned p_lds = lds0 + 2 * TILE_BYTES;
  const unsigned p_wr = p_lds + (unsigned)((HB == 2 ? (w >> 1) * 2048 : h0 * 1024) + ((kg & 1) * 32 + 16 * (w & 1) + m) * 16 + (kg >> 1) * 8);
  const unsigned p_rd = p_lds + (unsigned)(lane * 16);

  int id_next = 0;
  if (ntiles > 0) {
    const int id0 = id_of(0);
    id_next = id_of(1);
    gather(offset_of(id0), 0);
  }
  int stores_after = 0;                      // p_out stores a wave issued after the transfers it waits for
#pragma clang loop unroll(disable)
  for (int n = 0; n < ntiles; n++) {
    asm volatile("" : "+s"(n));              // one copy of the body
    if (POUT == 1 && stores_after) { DSA_WAIT_VMCNT(1); }
    else if (POUT == 2 && stores_after) { DSA_WAIT_VMCNT(HB); }
    else { DSA_WAIT_VMCNT(0); }
    __syncthreads();                         // the tile has landed; the other one and P have been read
    if (n + 1 < ntiles) {
      unsigned goff = offset_of(id_next);
      asm volatile("" : "+v"(goff));         // before the next load is on its way: the wait for this one would be for both
      id_next = id_of(n + 2);
      __builtin_amdgcn_sched_barrier(0);
      gather(goff, (n + 1) & 1);
    }
    const unsigned tb = lds0 + (unsigned)((n & 1) * TILE_BYTES);
    const int tile = __builtin_amdgcn_readfirstlane(tlist[n]);
    const unsigned mask = __builtin_amdgcn_readfirstlane(tmask[tile]);

    // ---- S^T of the wave's 16 heads; two chains: the half tiles, or the even and the odd k-steps of one ----
    f32x4 sa[2];
    {
      constexpr int NX = HB * KS;
      const unsigned t0 = tb + row0;
      auto row = [&](int x) {
        const int ks = HB == 2 ? x >> 1 : x, hh = HB == 2 ? x & 1 : 0;
        return *LDS_PTR(const bf16x8, (uintptr_t)((t0 ^ (64 * (ks & 1))) + (ks >> 1) * GRP_BYTES + 2048 * hh));
      };
      bf16x8 f[HALF_AHEAD];
#pragma unroll
      for (int x = 0; x < HALF_AHEAD; x++) f[x] = row(x);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 0; x < NX; x++) {
        mfma16_v(sa[x & 1], f[x % HALF_AHEAD], qreg[HB == 2 ? x >> 1 : x], x < 2);
        if (x + HALF_AHEAD < NX) f[x % HALF_AHEAD] = row(x + HALF_AHEAD);
        __builtin_amdgcn_sched_barrier(0);
      }
      mfma16_done(sa[0], sa[1]);
      if (HB == 1) {
#pragma unroll
        for (int e = 0; e < 4; e++) sa[0][e] += sa[1][e];
      }
    }
    // accumulator e of half hh is key 16 hh + 4 kg + e of the tile
    if (mask != 0xffffffffu) {
      const unsigned mg = mask >> (16 * h0 + 4 * kg);
#pragma unroll
      for (int hh = 0; hh < HB; hh++)
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (!((mg >> (16 * hh + e)) & 1u)) sa[hh][e] = -INFINITY;
    }
    stores_after = 0;
    if (POUT != 0 && head_ok && tile * BI >= p_skip) {
      const size_t prow = ((size_t)qi * H + h) * (K - p_skip) + (size_t)(tile * BI - p_skip);
      if (POUT == 2) {
#pragma unroll
        for (int hh = 0; hh < HB; hh++) *(f32x4*)((float*)a.p_out + prow + 16 * (h0 + hh) + 4 * kg) = sa[hh];
      } else if (HB == 1) {
        typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
        *(u32x2*)((unsigned short*)a.p_out + prow + 16 * h0 + 4 * kg) = u32x2{cvt_pk_bf16(sa[0][0], sa[0][1]), cvt_pk_bf16(sa[0][2], sa[0][3])};
      } else {
        // 8-byte pieces of each half tile; lanes 16 apart trade them, so that a lane stores 8 consecutive keys: those from
        // 0, 16, 8, 24 on for kg = 0 .. 3
        unsigned x0 = cvt_pk_bf16(sa[0][0], sa[0][1]), x1 = cvt_pk_bf16(sa[0][2], sa[0][3]);
        unsigned y0 = cvt_pk_bf16(sa[1][0], sa[1][1]), y1 = cvt_pk_bf16(sa[1][2], sa[1][3]);
        asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3\n\ts_nop 1"
                     : "+v"(x0), "+v"(y0), "+v"(x1), "+v"(y1));
        *(uint4*)((unsigned short*)a.p_out + prow + 16 * (kg & 1) + 8 * (kg >> 1)) = make_uint4(x0, x1, y0, y1);
      }
      stores_after = 1;
    }
    // ---- softmax numerators (base 2); P to LDS ----
    if (n == 0) {
      float mx = sa[0][0];
#pragma unroll
      for (int e = 1; e < 4 * HB; e++) mx = fmaxf(mx, sa[e >> 2][e & 3]);
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      if (HB == 1) {                         // and of the other half tile
        float* const half_s = (float*)(pbuf + 2048);         // [4][16], behind the one block's P
        if (kg == 0) half_s[16 * w + m] = mx;
        __syncthreads();
        mx = fmaxf(mx, half_s[16 * (w ^ 2) + m]);
      }
      m_ref = reference_point(mx * c2);
    }
    float sum = 0.f;
#pragma unroll
    for (int hh = 0; hh < HB; hh++) {
      float p[4];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        p[e] = __builtin_amdgcn_exp2f(fmaf(sa[hh][e], c2, -m_ref));
        sum += p[e];
      }
      typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
      const u32x2 pw = {cvt_pk_bf16(p[0], p[1]), cvt_pk_bf16(p[2], p[3])};
      *LDS_PTR(u32x2, (uintptr_t)(p_wr + 1024 * hh)) = pw;
#pragma unroll
      for (int x = 0; x < 2; x++) w_run += __builtin_bit_cast(float, pw[x] << 16) + __builtin_bit_cast(float, pw[x] & 0xffff0000u);
    }
    l_run += sum;
    overflow |= sum > REDO_TERM;             // one of the terms, or a few just below
    __syncthreads();

    // ---- O^T += V^T . P^T ----
    {
      const unsigned vb = tb + tr0 + (unsigned)(2 * w * GRP_BYTES);
      auto read_v = [&](int x) {             // x = 4 s + i
        const unsigned b = (vb ^ (64 * (x & 1))) + ((x & 3) >> 1) * GRP_BYTES + 2048 * (x >> 2);
        return value_operand(__builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(i16x4, (uintptr_t)b)),
                             __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(i16x4, (uintptr_t)(b + 1024))));
      };
      bf16x8 p[2][HB], v[3];
#pragma unroll
      for (int s = 0; s < 2; s++)
#pragma unroll
        for (int hb = 0; hb < HB; hb++) p[s][hb] = *LDS_PTR(const bf16x8, (uintptr_t)(p_rd + hb * 2048 + s * 1024));
#pragma unroll
      for (int x = 0; x < 3; x++) v[x] = read_v(x);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 0; x < 8; x++) {
#pragma unroll
        for (int hb = 0; hb < HB; hb++) mfma_a_vv(o[x & 3][hb], v[x % 3], p[x >> 2][hb]);
        if (x + 3 < 8) v[x % 3] = read_v(x + 3);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  // ---- epilogue: a mark is of a whole 32-head block, i.e. of two waves, or of all four ----
  float l_tot = l_run + __shfl_xor(l_run, 16, 64);
  l_tot += __shfl_xor(l_tot, 32, 64);
  float w_tot = w_run + __shfl_xor(w_run, 16, 64);
  w_tot += __shfl_xor(w_tot, 32, 64);
  float* const inv_s = (float*)pbuf;         // [64] factors, then [4] marks
  int* const again_s = (int*)(inv_s + 64);
  float* const l_s = inv_s + 128;            // [2][4][16]
  __syncthreads();                           // P has been read
  const bool mine = __ballot(overflow) != 0ull;
  if (lane == 0) again_s[w] = mine;
  if (HB == 1 && kg == 0) { l_s[16 * w + m] = l_tot; l_s[64 + 16 * w + m] = w_tot; }
  __syncthreads();
  const bool lower = __builtin_amdgcn_readfirstlane(again_s[0] | again_s[1]) != 0, upper = __builtin_amdgcn_readfirstlane(again_s[2] | again_s[3]) != 0;
  const bool again[2] = {HB == 2 ? lower : lower || upper, upper};       // of the workgroup's blocks
  if (HB == 1) {
    l_tot = l_s[16 * hw + m] + l_s[16 * hw + 32 + m];
    w_tot = l_s[64 + 16 * hw + m] + l_s[96 + 16 * hw + m];
  }
  const float* const sink = a.sink && head_ok ? a.sink + h : nullptr;
  const Final fin = finish_head(m_ref, l_tot, sink);
  if (kg == 0 && h0 == 0) {
    if (head_ok && !again[HB == 2 ? w >> 1 : 0]) a.lse[(size_t)qi * H + h] = fin.lse;
    inv_s[16 * hw + m] = finish_head(m_ref, w_tot, sink).inv;
  }
  __syncthreads();
#pragma unroll
  for (int hb = 0; hb < HB; hb++) {
    if (32 * (HB * hg + hb) >= H || again[hb]) continue;
    const float inv = inv_s[32 * hb + r];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int dt = 4 * w + i;
      mfma_done_a(o[i][hb]);
      store_out(o[i][hb], inv, (unsigned short*)a.out + ((size_t)qi * H + 32 * (HB * hg + hb) + r) * DV + 32 * dt + 8 * g);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  unsigned marked = 0;
#pragma unroll
  for (int hb = 0; hb < HB; hb++)
    if (32 * (HB * hg + hb) < H && again[hb]) marked |= 1u << (HB * hg + hb);
  if (marked) redo_marked<4>(a, qi, marked, w, lane_again());
}

// Sum of the ksplit partial results of a query, reading the accumulator layout in which they were stored (1 KB per
// instruction).  HBM / L2-bound with many queries (ksplit * H * 2 KB each): one wave per (query, 32-head block, value column
// tile).  A few queries are bound by the chain of round trips to memory and by the compute units at work: SHARED gives the
// tile to the four waves of a workgroup, a quarter of the ranges each, whose sums meet in LDS.
template <bool SHARED>
__global__ __launch_bounds__(256) void mla_fwd_combine_kernel(FwdArgs a) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31;
  const int HB = a.H / 32;
  const int per = SHARED ? DTILES : DTILES / 4;
  const int dt = SHARED ? (int)blockIdx.x % per : ((int)blockIdx.x % per) * 4 + wave;
  const int hb = ((int)blockIdx.x / per) % HB, qi = ((int)blockIdx.x / per) / HB;
  const int ns = a.ksplit, s0 = SHARED ? wave : 0, s_step = SHARED ? 4 : 1;
  const float* ml = a.part_ml + ((size_t)qi * ns * a.H + hb * 32 + r) * 2;
  const f32x4* po = a.part_o + (((size_t)qi * ns * HB + hb) * DTILES + dt) * 256 + lane;
  const size_t o_step = (size_t)HB * DTILES * 256;
  constexpr int AHEAD = SHARED ? 4 : 2;      // ranges requested together; the first ones beside the statistics
  f32x4 v[AHEAD][4];
  auto load = [&](int s) {
#pragma unroll
    for (int i = 0; i < AHEAD; i++)
      if (s + i * s_step < ns) {
#pragma unroll
        for (int j = 0; j < 4; j++) v[i][j] = po[(s + i * s_step) * o_step + j * 64];
      }
  };
  load(s0);
  float m = -1e30f;
  bool again = false;                        // the same for all threads of the workgroup
#pragma unroll 8
  for (int s = 0; s < ns; s++) {
    const float ms = ml[(size_t)s * a.H * 2];
    again |= is_marked(ms);
    m = fmaxf(m, ms);
  }
  float l = 0.f;
  f32x16 acc;
#pragma unroll
  for (int e = 0; e < 16; e++) acc[e] = 0.f;
  if (__ballot(again) != 0ull) {
    redo_block<false>(a, qi, hb, dt, acc, m, l, (int)threadIdx.x);
    if (SHARED && wave != 0) return;         // all waves have the same block
  } else {
    for (int s = s0; s < ns; s += AHEAD * s_step) {
      if (s != s0) load(s);
#pragma unroll
      for (int i = 0; i < AHEAD; i++) {
        const int si = s + i * s_step;
        if (si >= ns) break;
        const float f = __builtin_amdgcn_exp2f(ml[(size_t)si * a.H * 2] - m);
        l = fmaf(ml[(size_t)si * a.H * 2 + 1], f, l);
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
          for (int e = 0; e < 4; e++) acc[4 * j + e] = fmaf(v[i][j][e], f, acc[4 * j + e]);
      }
    }
    if (SHARED) {
      extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
      f32x4* box = (f32x4*)smem + lane;                                  // [wave - 1][4][lane], then the sums l
      float* box_l = (float*)(smem + 3 * 4096) + lane;
      if (wave != 0) {
#pragma unroll
        for (int j = 0; j < 4; j++) box[((wave - 1) * 4 + j) * 64] = f32x4{acc[4 * j], acc[4 * j + 1], acc[4 * j + 2], acc[4 * j + 3]};
        box_l[(wave - 1) * 64] = l;
      }
      __syncthreads();
      if (wave != 0) return;
#pragma unroll
      for (int w = 0; w < 3; w++) {
        l += box_l[w * 64];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const f32x4 o = box[(w * 4 + j) * 64];
#pragma unroll
          for (int e = 0; e < 4; e++) acc[4 * j + e] += o[e];
        }
      }
    }
  }
  write_block(a, qi, hb, dt, acc, m, l, (int)threadIdx.x);
}

// ---------------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------------
struct FwdPlan { int mode, n_hg, ksplit, k_loc; };

int max_slots(int mode) {                    // slots of a range whose id arrays fit LDS beside the tile ring
  if (mode >= 3) return 8192;                // (they read them from memory)
  const int ring = mode == 0 ? WIDE_LDS : 4 * TILE_BYTES;
  return (160 * 1024 - ring - 16) * 16 / 68 / 64 * 64;                  // 4 B per slot + 8 B per tile of 32
}

// The combine kernel shares a tile's ranges among waves for few head blocks (2048 slots, us with it / without: 1 query x 128
// heads 18.4 / 20.2, 1 x 32 17.3 / 18.9, 4 x 128 22.2 / 22.6, 8 x 128 24.6 / 24.6, 16 x 128 32.3 / 30.2).
constexpr int SHARE_RANGES = 4, SHARE_BLOCKS = 16;
bool combine_shares(int S, int H, int ksplit) { return ksplit >= SHARE_RANGES && (long)S * (H / 32) <= SHARE_BLOCKS; }

// Two ranges of modes 1 and 2 meet by themselves: both workgroups write their sums, through to where every XCD sees them, and the one
// that is second puts its own, which it still has, beside the other's.  That is one launch less, and half of the sums are read.  us, with
// mla_fwd_combine_kernel behind / so: 48 queries x 128 heads x 2048 slots 52.5 / 49.4, 61 x 64 x 1024 29.6 / 27.8, 121 x 32 x 1024 28.6 / 26.0, 30 x
// 128 x 1024 28.4 / 27.0.  With fences for the whole device around plain stores and loads 37 for the second of these (each writes back, or
// drops, an XCD's whole L2), with such stores and a fence before plain loads 33.
bool ranges_meet(int mode, int ksplit) { return ksplit == 2 && (mode == 1 || mode == 2); }

// The mode and the number of slot ranges with the least estimated time: rounds of workgroups over the 256 compute
// units (512 places in modes 3 and 4), each a fixed part (Q rows, ids, first tile, epilogue) plus its pairs of tiles, plus the kernel
// that follows.  The constants are measured times in us, random rows.  A round among others, FULL: the rows of all its queries come in
// together, and the gathers of 256 workgroups share the fabric.  A single or last round, LAST: IDLE on an empty chip, and nearly that
// while it is half empty, hence the square.  Modes 3 and 4 by whether workgroups share a compute unit; where few do, what they take
// with keys that lie far apart.  Those of single rounds and of the ranges are fitted to every form and number of ranges timed at 1300
// sizes (1 - 1200 queries, 32 - 128 heads, 192 - 8192 slots, keys of one long sequence and of a sequence per query): the form that
// the estimate picks takes 0.6 % more than the best one in the mean, 10 % at most (1.2 and 23 % with constants from a dozen sizes).  us,
// before and after: 61 queries x 64 heads x 1024 slots 31.4 (one range) and 28.9 (two), 121 x 32 x 1024 42.7 and 37.9, 80 x 128 x 2048 83
// (mode 1) and 73 (mode 0 in two ranges), 40 x 64 x 768 25.5 and 22.3 (three ranges), 250 x 64 x 512 35 (mode 1) and 31 (mode 3).
// 2048 slots, 128 heads: one query 86 us in mode 0 and 15 as 64 workgroups of mode 2 in 16 ranges; 48 queries 90 in mode 0 and
// 47 in mode 1 of two ranges; 128 queries 100 and 82 (mode 1), 160 queries 100 and 148, 600 queries 334 and 392.  64 heads: 256 queries
// 94 us in mode 3 and 83 in mode 1, 300 queries 123 and 140, 3000 817 and 900; 513 - 738 queries, one
// round of mode 3's 512 places and a short second one, are as fast in mode 1 (600 queries 218 and 216, with 65536 keys 243 and 256) and take it.
// Mode 0 in ranges: of up to 2048 slots for some 43 - 101 queries (70 queries 65 us, mode 1 73); lists beyond what
// modes 1 and 2 hold (3840) have it up to some hundred queries: 100 queries x 4096 slots 121 us and 152 in mode 1 of two ranges, x 8192
// 215 and 285 (303 in mode 0 undivided), 300 x 4096 357 and 391 (381).
// 32 heads: 257 queries 78 us in mode 4 and 112 in mode 2, 800 queries 175 and 236.  4000 queries of 128 heads: 256 slots 440 us in
// mode 0 and 390 in mode 3, 640 slots 760 and 800 (150 queries x 256 slots 28.6 and 31.2).
// WHOLE: what modes 0 and 1 take beyond the fit with all slots in one workgroup, more with few pairs (250 queries x 64 heads x 256 slots
// 27.5 us in mode 1 and 23.7 in mode 3, 89 x 128 x 256 22.8 and 21.2; 94 x 128 x 2048 82.6 in mode 1 and 87.6 in two ranges of mode 0).
// MEET_BYTES: what two ranges that meet (modes 1 and 2) take of the time for the sums' bytes, of which half are not read back; the wait of one
// workgroup for the other takes the place of the launch.  251 random sizes of 32 - 128 heads, 1 - 256 queries, 128 - 2048 slots: 0.975 of the time
// with a kernel behind all ranges in the mean, 0.89 to 1.025; with nothing but the bytes for them small calls split where they should not
// (up to 1.27).
// Blocks done again inside them and not by a kernel behind: 168 x 64 x 512 35.2 -> 32.2 us, 108 x 128 x 1024 52.7 -> 50.6.
// One pair of tiles is always mode 3, so that a query has the same bits whatever heads stand beside it: 4000 queries of 128 heads 320 us in
// mode 0 and 278, 1800 of 64 heads 90 and 64, 2 of 32 11.0 and 10.4.
FwdPlan plan_fwd(int S, int H, int K, bool may_split) {
  constexpr float WHOLE = 1.8f, WHOLE_FEW = 4.6f, COMBINE = 2.37f, COMBINE_RANGE = 0.22f, SHARED_RANGE = 0.1f, COMBINE_BYTES_PER_US = 6.2e6f, MEET_BYTES = 0.62f;
  constexpr float FIXED_IDLE[5] = {4.91f, 5.86f, 4.51f, 5.57f, 3.8f}, FIXED_FULL[5] = {14.5f, 10.5f, 6.8f, 9.0f, 8.5f};
  constexpr float PAIR_FULL[5] = {3.36f, 2.1f, 1.8f, 4.05f, 2.8f}, PAIR_IDLE[5] = {2.35f, 1.68f, 1.31f, 2.82f, 1.78f};
  constexpr float PAIR_LAST[3] = {3.65f, 2.24f, 1.75f}, PAIR_SHARED[5] = {0.f, 0.f, 0.f, 3.41f, 1.42f};
  constexpr int HEADS[5] = {128, 64, 32, 64, 32}, SLOTS[5] = {256, 256, 256, 512, 512};
  if (K <= 2 * BI) return {3, (H + HEADS[3] - 1) / HEADS[3], 1, K};
  const int pairs = K / (2 * BI);
  FwdPlan best = {0, 1, 1, K};
  float best_t = 1e30f;
  for (int mode = H > 64 ? 0 : H > 32 ? 1 : 2; mode < 5; mode++) {
    if (mode == (H > 32 ? 4 : 3)) continue;
    // 128 heads: mode 3 up to 256 slots, mode 0 from there on; 96 fill two thirds of mode 3
    if (H > 64 && mode == (H > 96 && K <= 256 ? 0 : 3)) continue;
    const int n_hg = (H + HEADS[mode] - 1) / HEADS[mode];
    for (int want = 1; want <= (may_split && mode < 3 ? 32 : 1) && want <= pairs; want++) {
      const int per = (pairs + want - 1) / want, ksplit = (pairs + per - 1) / per;
      if (ksplit != want || 64 * per > max_slots(mode)) continue;
      const long wgs = (long)S * n_hg * ksplit;
      const long rounds = wgs <= SLOTS[mode] ? 0 : wgs / SLOTS[mode];                  // full ones, with others behind or before
      const float rest = (float)(wgs - rounds * SLOTS[mode]) / (float)SLOTS[mode];
      const float pair = mode < 3      ? PAIR_IDLE[mode] + rest * rest * (PAIR_LAST[mode] - PAIR_IDLE[mode])
                         : rest > 0.5f ? PAIR_SHARED[mode] + 2.0f * (rest - 0.5f) * (PAIR_FULL[mode] - PAIR_SHARED[mode])
                                       : PAIR_IDLE[mode];
      const float fixed = mode >= 3 && rest > 0.5f ? FIXED_FULL[mode] : FIXED_IDLE[mode];
      float t = (float)rounds * (FIXED_FULL[mode] + per * PAIR_FULL[mode]);
      if (rest > 0.0f) t += fixed + per * pair;
      t += ksplit == 1 ? (mode >= 2 ? 0.0f : pairs <= 8 ? WHOLE_FEW : WHOLE)
                       : COMBINE + (combine_shares(S, H, ksplit) ? SHARED_RANGE : COMBINE_RANGE) * ksplit +
                             (ranges_meet(mode, ksplit) ? MEET_BYTES : 1.0f) * (float)S * ksplit * H * (2 * DV * 4) / COMBINE_BYTES_PER_US;
      if (t < best_t) { best_t = t; best = {mode, n_hg, ksplit, 64 * per}; }
      if (wgs >= 4096) break;                // more ranges only add rounds
    }
  }
  return best;
}

// Neighbouring units that share an XCD, as many as leave the XCDs evenly loaded.  The four tokens of each of 50 sequences (2500 keys, 32
// heads, 512 slots): 28.4 us apart and 27.0 together with ids at random, 27.2 and 23.1 where they have four fifths of them in
// common; 150 x 4 75.3 / 71.4 and 72.0 / 56.3; 16 x 4 of 8000 keys, 64 heads, 2048 slots in ranges 44.7 / 42.0 and 42.4 / 38.1.  Queries
// that share nothing: the same within 1 % either way.
int unit_span(const FwdPlan& p, int S) {
  const int units = S * p.ksplit;
  return units >= 128 ? 4 : units >= 64 ? 2 : 1;
}

size_t part_bytes(const FwdPlan& p, int S, int H) {
  if (p.ksplit == 1) return 0;
  return (size_t)S * p.ksplit * H * (DV * 4 + 8) + 256 + (ranges_meet(p.mode, p.ksplit) ? (size_t)S * p.n_hg * 8 : 0);
}

// A number that no other call of the process has, and that what lies in uninitialised memory does not hold but by a chance of 2^-64.
unsigned long long call_number() {
  static std::atomic<unsigned long long> next{(unsigned long long)std::chrono::system_clock::now().time_since_epoch().count() << 20};
  unsigned long long x = next.fetch_add(1, std::memory_order_relaxed);
  x = (x ^ x >> 31) * 0x9e3779b97f4a7c15ull;           // (one to one)
  return x ? x : call_number();
}

template <int MODE, bool SPLIT, int POUT>
constexpr auto fwd_kernel() {
  if constexpr (MODE == 0) return mla_fwd_wide_kernel<SPLIT, POUT>;
  else if constexpr (MODE >= 3) return mla_fwd_half_kernel<MODE == 3 ? 2 : 1, POUT>;
  else return mla_fwd_kernel<MODE, SPLIT, POUT>;
}

template <int MODE, bool SPLIT>
int launch_fwd(const FwdArgs& a, int p_out_f32, bool shared, hipStream_t st) {
  const size_t smem = MODE == 0   ? WIDE_LDS + ids_lds_bytes(a.k_loc)
                      : MODE >= 3 ? HALF_LDS + mask_lds_bytes(a.k_loc)
                                  : 4 * TILE_BYTES + ids_lds_bytes(a.k_loc);
  if (smem > 160 * 1024) return -1;
  const int units = a.S * a.ksplit;
  const dim3 grid(MODE == 0 ? units : dsa_cdiv(units, 8 * a.span) * 8 * a.span * a.n_hg), block(MODE == 0 ? 512 : 256);
#define DSA_FWD_LAUNCH(P) do { \
    auto kern = fwd_kernel<MODE, SPLIT, P>(); \
    if (dsa_reserve_lds((const void*)kern, smem) != hipSuccess) return -2; \
    kern<<<grid, block, smem, st>>>(a); \
  } while (0)
  if (!a.p_out) DSA_FWD_LAUNCH(0);
  else if (!p_out_f32) DSA_FWD_LAUNCH(1);
  else DSA_FWD_LAUNCH(2);
#undef DSA_FWD_LAUNCH
  const size_t tail = (size_t)TILE_BYTES + ids_lds_bytes(a.K);           // one tile and the ids, for blocks done again
  if (a.turn) return 0;
  auto combine = shared ? mla_fwd_combine_kernel<true> : mla_fwd_combine_kernel<false>;
  if (!SPLIT) return 0;
  if (dsa_reserve_lds((const void*)combine, tail) != hipSuccess) return -2;
  combine<<<dim3(a.S * (a.H / 32) * (shared ? DTILES : DTILES / 4)), 256, tail, st>>>(a);
  return 0;
}

// S_all: the queries of the call of which these S are a block (S where it is the whole).  They, not S, choose the form, the ranges
// and the way the ranges' sums are put together, so a query has the same bits in a block of any size.
int fwd_impl(const void* q, const void* kv, const int32_t* ids, int S_all, int S, int H, int Skv, int K, int q_start, float sm_scale,
             int d_v, void* out, float* lse, void* p_out, int p_out_f32, const float* attn_sink, int p_out_skip,
             void* workspace, size_t workspace_bytes, void* stream, bool p_all = true) {
  DSA_REQUIRE(d_v == DV, "dsa_sparse_mla_fwd: only d_v = 512 (d_qk = 576) is supported, got d_v = %d", d_v);
  DSA_REQUIRE(S >= 0 && Skv > 0, "dsa_sparse_mla_fwd: bad sequence sizes S=%d Skv=%d", S, Skv);
  DSA_REQUIRE(S_all >= S, "dsa_sparse_mla_fwd: a block of %d queries of %d", S, S_all);
  DSA_REQUIRE(H > 0 && H <= 128 && H % 32 == 0, "dsa_sparse_mla_fwd: head count must be 32, 64, 96 or 128, got %d", H);
  DSA_REQUIRE(K > 0 && K % 64 == 0, "dsa_sparse_mla_fwd: top-k must be a positive multiple of 64, got %d", K);
  DSA_REQUIRE(p_out_skip >= 0 && p_out_skip < K && p_out_skip % BI == 0,
              "dsa_sparse_mla_fwd: p_out_skip must be a multiple of %d in [0, top-k), got %d", BI, p_out_skip);
  DSA_REQUIRE((size_t)Skv * DQK * 2 <= 0xffffffffull, "dsa_sparse_mla_fwd: kv larger than 4 GiB is not supported");
  DSA_REQUIRE(((uintptr_t)q % 16) == 0 && ((uintptr_t)kv % 16) == 0 && ((uintptr_t)out % 8) == 0 &&
              ((uintptr_t)p_out % 16) == 0 && ((uintptr_t)attn_sink % 4) == 0 && ((uintptr_t)workspace % 16) == 0,
              "dsa_sparse_mla_fwd: misaligned pointer");
  DSA_REQUIRE(K <= 8192, "dsa_sparse_mla_fwd: top-k %d exceeds the supported maximum 8192", K);
  if (S == 0) return DSA_OK;
  hipStream_t st = (hipStream_t)stream;
  FwdPlan p = plan_fwd(S_all, H, K, true);
  if (part_bytes(p, S, H) > workspace_bytes || (p.ksplit > 1 && workspace == nullptr)) p = plan_fwd(S_all, H, K, false);
  FwdArgs a{(const __bf16*)q, (const __bf16*)kv, ids, (__bf16*)out, lse, p_out, S, H, Skv, K, q_start, sm_scale, attn_sink,
            p_out ? p_out_skip : 0, p_all, p.n_hg, p.ksplit, p.k_loc, unit_span(p, S), (f32x4*)workspace,
            (float*)((unsigned char*)workspace + (size_t)S * p.ksplit * H * DV * 4), nullptr, 0};
  if (ranges_meet(p.mode, p.ksplit)) {
    a.turn = (unsigned long long*)((unsigned char*)workspace + (size_t)S * p.ksplit * H * (DV * 4 + 8));
    a.token = call_number();
  }
  int rc;
  const bool split = p.ksplit > 1, shared = combine_shares(S_all, H, p.ksplit);
  if (p.mode == 0) rc = split ? launch_fwd<0, true>(a, p_out_f32, shared, st) : launch_fwd<0, false>(a, p_out_f32, shared, st);
  else if (p.mode == 3) rc = launch_fwd<3, false>(a, p_out_f32, shared, st);
  else if (p.mode == 4) rc = launch_fwd<4, false>(a, p_out_f32, shared, st);
  else if (p.mode == 1) rc = split ? launch_fwd<1, true>(a, p_out_f32, shared, st) : launch_fwd<1, false>(a, p_out_f32, shared, st);
  else rc = split ? launch_fwd<2, true>(a, p_out_f32, shared, st) : launch_fwd<2, false>(a, p_out_f32, shared, st);
  DSA_REQUIRE(rc != -1, "dsa_sparse_mla_fwd: top-k %d does not fit LDS", K);
  if (rc == -2) DSA_FAIL(DSA_ERR_LAUNCH, "dsa_sparse_mla_fwd: cannot reserve LDS");
  DSA_CHECK_LAUNCH("dsa_sparse_mla_fwd");
  return DSA_OK;
}

}  // namespace

extern "C" size_t dsa_sparse_mla_fwd_block_workspace_bytes(int S_all, int S, int H, int Skv, int K) {
  (void)Skv;
  if (S <= 0 || S_all < S || H <= 0 || H % 32 || K <= 0 || K % 64) return 0;
  return part_bytes(plan_fwd(S_all, H, K, true), S, H);
}

extern "C" size_t dsa_sparse_mla_fwd_workspace_bytes(int S, int H, int Skv, int K) {
  return dsa_sparse_mla_fwd_block_workspace_bytes(S, S, H, Skv, K);
}

extern "C" int dsa_sparse_mla_fwd_form(int S, int H, int K, int with_workspace, int* ranges) {
  if (S <= 0 || H <= 0 || H > 128 || H % 32 || K <= 0 || K % 64 || K > 8192) return -1;
  const FwdPlan p = plan_fwd(S, H, K, with_workspace != 0);
  if (ranges) *ranges = p.ksplit;
  return p.mode;
}

extern "C" int dsa_sparse_mla_fwd_block(const void* q, const void* kv, const int32_t* ids, int S_all, int S, int H, int Skv, int K,
                                        int q_start, float sm_scale, int d_v, void* out, float* lse, void* p_out,
                                        int p_out_f32, const float* attn_sink, int p_out_skip, void* workspace,
                                        size_t workspace_bytes, void* stream) {
  return fwd_impl(q, kv, ids, S_all, S, H, Skv, K, q_start, sm_scale, d_v, out, lse, p_out, p_out_f32, attn_sink, p_out_skip,
                  workspace, workspace_bytes, stream);
}

extern "C" int dsa_sparse_mla_fwd_dist(const void* q, const void* kv, const int32_t* ids, int S_all, int S, int H, int Skv, int K,
                                       int q_start, float sm_scale, int d_v, void* out, float* lse, const float* attn_sink,
                                       int dist_heads, float* target, void* logits, void* workspace, size_t workspace_bytes,
                                       void* stream) {
  DSA_REQUIRE(logits != nullptr && target != nullptr && dist_heads > 0 && dist_heads <= H, "dsa_sparse_mla_fwd_dist: bad arguments (%d of %d heads)", dist_heads, H);
  DSA_REQUIRE(K <= 4096, "dsa_sparse_mla_fwd_dist: K=%d exceeds the supported maximum 4096", K);
  // what the reduction does not read, the forward does not write: the tiles of short prefixes behind their last slot
  const bool live = ((uintptr_t)logits % 32) == 0 && ((uintptr_t)ids % 16) == 0 && sm_scale > 0.f;
  const int rc = fwd_impl(q, kv, ids, S_all, S, H, Skv, K, q_start, sm_scale, d_v, out, lse, logits, 0, attn_sink, 0, workspace,
                          workspace_bytes, stream, !live);
  if (rc != DSA_OK || S == 0) return rc;
  if (!live) return dsa_attn_dist(logits, 0, S, dist_heads, K, (int64_t)H * K, K, sm_scale, target, stream);
  DSA_REQUIRE(dsa_attn_dist_live(logits, ids, S, dist_heads, Skv, K, (int64_t)H * K, q_start, sm_scale, target, (hipStream_t)stream) == 0,
              "dsa_sparse_mla_fwd_dist: unsupported K");
  DSA_CHECK_LAUNCH("dsa_sparse_mla_fwd_dist");
  return DSA_OK;
}

extern "C" int dsa_sparse_mla_fwd_ws(const void* q, const void* kv, const int32_t* ids, int S, int H, int Skv, int K,
                                     int q_start, float sm_scale, int d_v, void* out, float* lse, void* p_out,
                                     int p_out_f32, const float* attn_sink, int p_out_skip, void* workspace,
                                     size_t workspace_bytes, void* stream) {
  return fwd_impl(q, kv, ids, S, S, H, Skv, K, q_start, sm_scale, d_v, out, lse, p_out, p_out_f32, attn_sink, p_out_skip,
                  workspace, workspace_bytes, stream);
}

extern "C" int dsa_sparse_mla_fwd_ex(const void* q, const void* kv, const int32_t* ids, int S, int H, int Skv, int K,
                                     int q_start, float sm_scale, int d_v, void* out, float* lse, void* p_out,
                                     int p_out_f32, const float* attn_sink, int p_out_skip, void* stream) {
  return fwd_impl(q, kv, ids, S, S, H, Skv, K, q_start, sm_scale, d_v, out, lse, p_out, p_out_f32, attn_sink, p_out_skip,
                  nullptr, 0, stream);
}

extern "C" int dsa_sparse_mla_fwd(const void* q, const void* kv, const int32_t* ids, int S, int H, int Skv, int K,
                                  int q_start, float sm_scale, int d_v, void* out, float* lse, void* p_out,
                                  int p_out_f32, void* stream) {
  return fwd_impl(q, kv, ids, S, S, H, Skv, K, q_start, sm_scale, d_v, out, lse, p_out, p_out_f32, nullptr, 0, nullptr, 0, stream);
}
