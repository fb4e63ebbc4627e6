// Sparse MQA-MLA attention backward for gfx950, deterministic.
//
// Per (query, selected key) pair the backward needs five products:
//   S  = Q.KV^T (576)   dP = dO.V^T (512)   dQ += dS.KV (576)   dKV[key] += dS^T.Q (576) + P^T.dO (512)
// The operands Q and dO of one query (278 KB in bf16 with 128 heads) plus the fp32 dQ accumulators
// (295 KB) do not fit one compute unit (512 KB of registers, 160 KB of LDS) next to the gathered key
// tiles, and the products over d and over heads need the same operands in two orientations.  The work
// is therefore split into passes:
//   P, dS, rows  (bwd_pds_rows_kernel)  S and dP per 32-key tile -> P and dS; the tile's pair rows dS^T.Q + P^T.dO (sum over all
//                heads) -> one bf16 row of 576 values in a pair buffer, at the position given by a key-sorted order.  Both
//                orientations of Q and dO and P stay on the compute unit; dS goes to HBM as bf16, 2 KB per 32 heads and tile
//   dQ           dQ^T += KV^T.dS^T, both operands by LDS transpose reads
//   dKV          dKV[key] = sum of that key's rows, in ascending query order
// The last two share a launch (bwd_dq_reduce_kernel).
// The key-sorted order comes from a bitmap key x query, its row-wise prefix popcounts and
// an exclusive scan over keys: integer work only, so the order - and with it every fp32 sum - is
// identical from run to run.  No floating-point atomics anywhere.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "mla_tile.h"
#include "order.h"

namespace {
using namespace mla;

// dS of one (query, tile) in memory, P and dS of a tile in LDS: [4 HG chunk groups][32 keys][8 heads] bf16.  HG is the number of 32-head groups the passes are
// compiled for: 1 or 2, or 4 for 96 and 128 heads.
constexpr int pds_kind_bytes(int HG) { return HG * 2048; }
inline int head_groups(int H) { return H <= 32 ? 1 : H <= 64 ? 2 : 4; }
constexpr int ROW_BYTES = DQK * 2;           // one pair row of the dKV buffer
constexpr int EXP_BYTES = 16;                // its exponents where rows may be those of joint units: see below
constexpr int PDS_THREADS = 512;

// Joint units.  With 64 or 32 heads, 2 or 4 consecutive queries may be worked as one query of 128 heads: their rows of Q, dO, O, lse and
// dQ follow one another in memory just like that.  The unit's slots are the union of the queries' keys, ascending; an entry carries
// in bits 24 .. 27 which of the queries have it (UNIT_KEY masks the key), and P and dS are zero for the heads of the others.  One
// pair row then stands for the key's pairs with all of them, and a key tile is gathered once.  order::qmap_unit_kernel decides
// for every group; `units` holds its padded slot count, or 0 where the queries stay by themselves, and the work list (order::WorkList) what there
// is to do.
// Why: the backward of few heads is bound by its pair rows, 1152 bytes written and read whatever the heads, and neighbouring queries share
// keys - a sliding window all but one, a selection of K out of L at least K / L of them.  The matrix work of the heads that have not
// selected a slot is wasted, which the pipes have room for.  Whole backward, us, by themselves / joint / as the rule takes them (u:
// union over sum of the lists): 3072 queries x 640 slots, window and compressed keys, 64 heads (u 0.54) 1138 / 904 / 903, 32 heads (0.27)
// 959 / 519 / 517; 2077 x 512 at random, 64 heads (0.73) 740 / 751 / 736, 32 heads (0.48) 617 / 509 / 519; 4000 x 512, 64 heads (0.83)
// 1482 / 1612 / 1486, 32 heads (0.63) 1229 / 1211 / 1128; 8000 x 256, 64 heads (0.94) 1889 / 2138 / 1831; 3000 x 2048, 32 heads (0.28)
// 2338 / 1167 / 1170.
//
// A unit's row stands for 2 or 4 rows, so it is held in more bits than they: 11 instead of 8 significant ones, fp16 with a power of
// two for every 64 columns (16 of the rotary part), chosen so that the largest of them lies in [2^14, 2^15).  Values down to 2^-29 of that
// one have all 11 bits.  Its fp32 exponent is one of EXP_BYTES bytes per row: groups 0 - 7 the 64-column groups, 8 - 11 the
// rotary ones; 0 marks a bf16 row, one of a query by itself: all of them are 0 before the rows are written, and where a call has no unit
// they are neither cleared nor read (marked row by row instead: scores and rows of 3000 x 2048 of 32768 keys, no units, 2867 -> 3234 us).
// In bf16 the rounding error would be that of the rows it stands for only where those are independent, and grows with what neighbouring
// queries have in common.  Its rms, emulated, over 256 queries x 256 of 288 slots, with rows per query 1, with units in bf16 / fp16: correlation 0
// of Q and dO 1.00 / 0.13; 0.9 1.27 / 0.16 (64 heads), 1.68 / 0.21 (32 heads); 0.99 1.36 / 0.17, 1.88 / 0.24.  What it takes, bf16 / fp16: scores and rows 521 / 562 us at 3072 queries x 640 slots x 64 heads and 276 / 297 at 2077 x 512 (maxima 22
// of the 41, products with the power 10, the exponents' way through LDS 8), dQ and the sums 308 / 314 and 180 / 176.
constexpr int unit_queries(int HG) { return 4 / HG; }
constexpr int UNIT_SLOTS = 3072;             // what the lists in LDS behind the operands of 128 heads have room for
constexpr int UNIT_KEY = 0xffffff;
inline int unit_slots(int HG, int K) { return unit_queries(HG) * K < UNIT_SLOTS ? unit_queries(HG) * K : UNIT_SLOTS; }
// dS of a group of G queries in memory: of the queries by themselves or of their unit
inline size_t group_pds_bytes(int HG, int G, int K) {
  const size_t apart = (size_t)G * (K / BI) * pds_kind_bytes(HG), joint = (size_t)(unit_slots(HG, K) / BI) * pds_kind_bytes(4);
  return G == 1 || apart > joint ? apart : joint;
}
// A unit's list of `n` slots (a multiple of 32) to LDS.  Slots behind the last key repeat the first one, for none of the queries.
__device__ __forceinline__ void stage_unit(const int* __restrict__ list, int n, int* idx_s) {
  const int pad = list[0] & UNIT_KEY;
  for (int t = threadIdx.x; t < n; t += blockDim.x) {
    const int v = list[t];
    idx_s[t] = v < 0 ? pad : v;
  }
  __syncthreads();
}

// ---------------------------------------------------------------------------------------------
// dQ
// ---------------------------------------------------------------------------------------------
// dQ^T[d, head] += KV^T[d, key] . dS^T[key, head] per 32-key tile.  Both operands are LDS transpose
// reads: of the gathered key tile (18 d-tiles) and of the tile's dS block copied verbatim from
// memory.  Twelve waves share the 72 accumulator tiles (18 d-tiles x 4 head groups): wave
// (dg, hp) = (wave % 6, wave / 6) owns d-tiles 3dg .. 3dg+2 for the head groups 2hp, 2hp+1: 6 tiles
// (96 accumulator registers), 12 MFMAs and 20 transposing reads per wave and tile.  A wave issues one
// LDS instruction per 40-odd cycles whatever its width, and a transposing read carries 8 bytes per
// lane: with eight waves (9 tiles, 28 reads each) the reads of a wave took longer than the MFMAs of
// the two waves of a SIMD together (1 200 against 1 152 cycles per tile).  Three waves per SIMD at
// under 168 registers per lane issue them in two thirds of the time, and one wave's transfer issue and
// waits run under the MFMAs of the other two.
// With up to 64 heads a wave owns its 3 d-tiles for head group hp only; with up to 32, for one k-step (16 keys) of the only
// head group, and the two k-steps' sums are added at the end.
constexpr int DQ_THREADS = 768;
// ids, pds, dq: the query's (UNIT: the joint unit's) slots, dS tiles and rows of dQ; qpos: its position; of every `per` heads the first
// `real` have a row in dq
// once: dS is read with the non-temporal hint
template <int STAGES, int HG, bool UNIT>
__device__ __forceinline__ void dq_body(
    const __bf16* __restrict__ kv, const int* __restrict__ ids, const unsigned char* __restrict__ pds,
    __bf16* __restrict__ dq, int H, int per, int real, int Skv, int K, int qpos, const int* __restrict__ dup_flag, bool once,
    unsigned char* smem) {
  constexpr int STAGE_BYTES = TILE_BYTES + pds_kind_bytes(HG);
  constexpr int NJ = HG == 4 ? 2 : 1;          // head groups of a wave
  constexpr int DS_WAVES = 2 * HG;             // waves that move 1 KB of the dS block each
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int dg = wave % 6, hp = wave / 6;
  const int r = lane & 31, g = lane >> 5;
  const int NT = K / BI;
  int* idx_s = (int*)(smem + STAGES * STAGE_BYTES);
  unsigned* tmask = (unsigned*)(idx_s + K);
  int* tlist = (int*)(tmask + NT);
  int* ntile_s = tlist + NT;
  int ntiles = NT;
  // (the helper is written for four waves; the others repeat part of its work with equal results)
  if constexpr (UNIT) stage_unit(ids, K, idx_s);
  else ntiles = stage_ids(ids, 0, K, Skv, qpos, idx_s, tmask, tlist, ntile_s);

  const unsigned lds0 = (unsigned)(uintptr_t)smem;
  // transposed read of the dS block: lane (blk, ii) points at key 16s + 8t + 4g + ii/4 and the 4 heads
  // 16*(blk&1) + 4*(ii&3) .. +3 of a head group.  In HBM the block is [head group][s'][g'][key][8 heads];
  // in LDS the 16-byte pieces of a head group are reordered to [key][s'][g'], so that the 16 pieces a
  // half-wave reads at once (4 keys x 4 head octets) are 256 consecutive bytes: no bank conflicts.
  unsigned ds_off[2][2];
  // transposed read of the key tile for the wave's d-tiles 3dg + i (same formula as LaneOffsets::tr_off,
  // with the parity of the d-tile known only at run time)
  unsigned a_off[3][2][2];
  {
    const int blk = lane >> 4, ii = lane & 15, qq = ii & 3;
    const int cl = 2 * (blk & 1) + ((ii & 3) >> 1), half = ii & 1;
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
      for (int t = 0; t < 2; t++) {
        const int key = 16 * s + 8 * t + 4 * g + (ii >> 2);
        ds_off[s][t] = (unsigned)(TILE_BYTES + key * 64 + (blk & 1) * 32 + (qq & 1) * 16 + (qq >> 1) * 8);
#pragma unroll
        for (int i = 0; i < 3; i++) {
          const int dt = 3 * dg + i;
          a_off[i][s][t] = (unsigned)((dt >> 1) * GRP_BYTES + key * 128 + (((4 * (dt & 1) + cl) ^ swz(key)) << 4) + half * 8);
        }
      }
  }
  // Transfers of a tile: 44 of 1 KB each.  Transfer t < 36 is slot t % 4 (keys 8*slot .. +7, thread (key,
  // sub) moving 16 bytes) of the 128-byte group t / 4 of the key rows; transfer 36 + b is 1 KB of the dS
  // block, piece P of the LDS order coming from piece src_piece(P) of the HBM order.  Wave v takes
  // transfers v, v + 12, v + 24 (groups v/4, v/4 + 3, v/4 + 6 of its slot v % 4) and, for v < 8, 36 + v.
  auto src_piece = [](int P) { return (P >> 7) * 128 + ((P >> 1) & 1) * 64 + (P & 1) * 32 + ((P >> 2) & 31); };
  const unsigned ds_src = (unsigned)src_piece((wave & (DS_WAVES - 1)) * 64 + lane) * 16u;
  const int gkey = 8 * (wave & 3) + (lane >> 3), gsub = lane & 7;
  const unsigned gslot = (unsigned)((gsub ^ swz(gkey)) * 16) + (unsigned)((wave >> 2) * 128);
  unsigned t_goff = 0, t_lb = 0, t_lbd = 0;
  const unsigned char* t_src = nullptr;
  auto issue_prepare = [&](int n) {
    const int tile = UNIT ? n : tlist[n];
    const unsigned sb = lds0 + (unsigned)((n % STAGES) * STAGE_BYTES);
    int kid = idx_s[tile * BI + gkey];
    kid = UNIT ? kid & UNIT_KEY : kid < 0 ? 0 : kid;
    t_goff = (unsigned)kid * (DQK * 2) + gslot;
    t_lb = __builtin_amdgcn_readfirstlane(sb + (unsigned)((wave & 3) * 1024 + (wave >> 2) * GRP_BYTES));
    t_lbd = __builtin_amdgcn_readfirstlane(sb + (unsigned)(TILE_BYTES + (wave & (DS_WAVES - 1)) * 1024));
    t_src = uniform_ptr(pds + (size_t)tile * pds_kind_bytes(HG));     // dS
  };
  // step 0 .. 2: the wave's three groups of the key rows; step 3: its part of the dS block (waves 0 .. DS_WAVES - 1)
  auto issue_step = [&](int j) {
    if (j < 3) dma16(t_lb + 3 * j * GRP_BYTES, t_goff + 3 * j * 128, kv);
    else if (wave < DS_WAVES) {
      if (once) dma16_once(t_lbd, ds_src, t_src);
      else dma16(t_lbd, ds_src, t_src);
    }
  };

  const int hg0 = HG == 4 ? 2 * hp : HG == 2 ? hp : 0;
  const int s0 = HG == 1 ? hp : 0;
  constexpr int NS = HG == 1 ? 1 : 2;          // k-steps of a wave
  f32x16 acc[3 * NJ];      // u = NJ * i + j: d-tile 3dg + i, head group hg0 + j
#pragma unroll
  for (int u = 0; u < 3 * NJ; u++)
#pragma unroll
    for (int e = 0; e < 16; e++) acc[u][e] = 0.f;
  typedef short i16x8 __attribute__((ext_vector_type(8)));
  auto tr_pair = [&](const unsigned char* p0, const unsigned char* p1) {
    const i16x4 x0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(i16x4, p0));
    const i16x4 x1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(i16x4, p1));
    return __builtin_bit_cast(bf16x8, (i16x8)__builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  for (int n = 0; n < STAGES - 1 && n < ntiles; n++) {
    issue_prepare(n);
#pragma unroll
    for (int j = 0; j < 4; j++) issue_step(j);
  }
  for (int n = 0; n < ntiles; n++) {
    static_assert(STAGES == 3, "one tile of transfers in flight behind the awaited one");
    // transfers per wave and tile: 4 for waves 0 .. DS_WAVES - 1, 3 for the others
    if (n + 1 < ntiles) { if (wave < DS_WAVES) { DSA_WAIT_VMCNT(4); } else { DSA_WAIT_VMCNT(3); } } else { DSA_WAIT_VMCNT(0); }
    __syncthreads();
    const bool more = n + STAGES - 1 < ntiles;
    if (more) { issue_prepare(n + STAGES - 1); issue_step(3); }
    const unsigned char* tb = smem + (n % STAGES) * STAGE_BYTES;
    // key-tile operands one d-tile ahead, the dS operands of the wave's head groups: [head group][k-step]
    bf16x8 a[2][NS], bds[NJ][NS];
    auto key_operand = [&](int i, int s) {
      return HG == 1 ? tr_pair(tb + (hp ? a_off[i][1][0] : a_off[i][0][0]), tb + (hp ? a_off[i][1][1] : a_off[i][0][1]))
                     : tr_pair(tb + a_off[i][s][0], tb + a_off[i][s][1]);
    };
#pragma unroll
    for (int s = 0; s < NS; s++) a[0][s] = key_operand(0, s);
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
      for (int s = 0; s < NS; s++) {
        const unsigned o0 = HG == 1 ? (s0 ? ds_off[1][0] : ds_off[0][0]) : ds_off[s][0];
        const unsigned o1 = HG == 1 ? (s0 ? ds_off[1][1] : ds_off[0][1]) : ds_off[s][1];
        bds[j][s] = tr_pair(tb + (hg0 + j) * 2048 + o0, tb + (hg0 + j) * 2048 + o1);
      }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 3; i++) {
      if (i + 1 < 3) {
#pragma unroll
        for (int s = 0; s < NS; s++) a[(i + 1) & 1][s] = key_operand(i + 1, s);
      }
#pragma unroll
      for (int s = 0; s < NS; s++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
          acc[NJ * i + j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i & 1][s], bds[j][s], acc[NJ * i + j], 0, 0, 0);
      if (more) issue_step(i);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if constexpr (HG == 1) {       // the second k-step's sums join the first one's
    __syncthreads();
    f32x4* box = (f32x4*)smem + (size_t)(dg * 12) * 64 + lane;
    if (hp == 1) {
#pragma unroll
      for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) box[(4 * i + j) * 64] = f32x4{acc[i][4 * j], acc[i][4 * j + 1], acc[i][4 * j + 2], acc[i][4 * j + 3]};
    }
    __syncthreads();
    if (hp == 1) return;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const f32x4 v = box[(4 * i + j) * 64];
#pragma unroll
        for (int e = 0; e < 4; e++) acc[i][4 * j + e] += v[e];
      }
  }
  // ---- write dQ: accumulator e of a lane is d = 32*dt + 8*(e/4) + 4*g + (e%4), head = 32*hg + r ----
  const bool poison = *dup_flag != 0;          // a query row with a repeated id: NaN instead of a sum that misses a term
#pragma unroll
  for (int u = 0; u < 3 * NJ; u++) {
    const int dt = 3 * dg + u / NJ;
    const int h = (hg0 + u % NJ) * 32 + r;
    if (h < H) {                               // the same for all lanes of a wave (H is a multiple of 32)
      const int query = UNIT ? h / per : 0, own = UNIT ? h % per : h;
      unsigned short* op = (unsigned short*)dq + (size_t)(query * real + own) * DQK + 32 * dt + 8 * g;
      uint4 o[2];
      acc_row_to_16B(acc[u], 1.0f, o);
      if (poison) o[0] = o[1] = make_uint4(0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u);
      if (own < real) {
        *(uint4*)op = o[0];
        *(uint4*)(op + 16) = o[1];
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// P, dS and the rows of the pairs, for 32 and 64 heads
// ---------------------------------------------------------------------------------------------
// Q and dO of 64 heads fit the registers of a compute unit in both orientations: 136 per lane for the products over d (wave
// (hw, hh) = (wave % 4, wave / 4): 16 heads, the 16 keys of half tile hh) and 64 for those over the heads (wave w: the columns
// 64 w .. 64 w + 63 of both; 16 columns of the rotary part come from LDS).  So P never leaves the compute unit, dS is written for
// the dQ products only, and a pair costs 1152 + 128 bytes of writes where two kernels with P and dS in memory between them wrote
// 1152 + 256 and read 256.
// Between two barriers a wave works on S, dP of tile n and on the rows of tile n - 1, whose P and dS all waves have put into
// LDS (two buffers) before the barrier; waves 0-3 take them in this order, waves 4-7 in the other one, so that the two waves
// of a SIMD issue stores and exponentials under each other's MFMAs.  The transfers of tile n + 2 come first in a step: between
// the MFMAs behind the row stores of a step they held waves 4-7 for 2600 cycles per tile instead of 1100.
// Bound by the row writes: a step of 5000 cycles writes 41 KB per compute unit, 4.7 TB/s, and the set-up of a query (208 KB
// read, 31 000 cycles) does not overlap it.  3072 queries x 128 + 512 slots of compressed keys: 0.68 ms against 0.41 + 0.51; 2077 x 512: 0.35 against 0.23 + 0.26.
// 32 heads have the same rows to write; four waves then have no scores to make.  The whole backward of 3072 queries x 640 slots 1501 ->
// 1108 us against two passes with P and dS in memory, 3000 x 2048 3172 -> 2474, 1024 x 256 254 -> 204.
constexpr int FUSED_STAGES = 3;
constexpr int FUSED_XCH = 2 * pds_kind_bytes(2);      // P and dS of a tile
constexpr int FUSED_ROT = 16384;                      // every wave's operands of the rotary columns
static_assert(64 * (DQK + DV) * 2 <= FUSED_STAGES * TILE_BYTES + 2 * FUSED_XCH + FUSED_ROT, "Q and dO of a query pass through this part of LDS");
__host__ __device__ inline size_t fused_lds_bytes(int K) {
  return (size_t)FUSED_STAGES * TILE_BYTES + 2 * FUSED_XCH + FUSED_ROT + ids_lds_bytes(K) + 512 + (size_t)K * 4;
}
template <int hh, int HG>                    // HG: groups of 32 heads, 2 or 1
__device__ __forceinline__ void pds_rows_body(
    const __bf16* __restrict__ q, const __bf16* __restrict__ kv, const int* __restrict__ ids,
    const __bf16* __restrict__ out, const __bf16* __restrict__ dout, const float* __restrict__ lse,
    unsigned char* __restrict__ pds, const int* __restrict__ dst, unsigned char* __restrict__ rows,
    int q0, int ql, int Skv, int K, int q_start, float sm_scale, int dummy_row, unsigned char* smem) {
  constexpr int H = 32 * HG, KS = DQK / 32, VS = DV / 32, STAGES = FUSED_STAGES;
  constexpr int DO_ACC = 12;                   // steps of dO in accumulation registers, beside all of Q: 120
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 15, kg = lane >> 4, g = lane >> 5;
  // One group: two waves of each half have S and dP, on SIMDs 0, 1 and 2, 3; the other four the rows alone.
  const int hw = HG == 2 ? wave & 3 : wave & 1;
  const bool scores = HG == 2 || (wave & 3) >> 1 == hh;
  const int qi = q0 + ql;
  const int NT = K / BI;
  // [ring][P and dS, two buffers][rotary operands], all of it Q and dO of the query at first | ids arrays | statistics | dst rows [K]
  unsigned char* xch = smem + STAGES * TILE_BYTES;
  bf16x8* xr_s = (bf16x8*)(xch + 2 * FUSED_XCH) + wave * 128 + lane;
  int* idx_s = (int*)(xch + 2 * FUSED_XCH + FUSED_ROT);
  unsigned* tmask = (unsigned*)(idx_s + K);
  int* tlist = (int*)(tmask + NT);
  int* ntile_s = tlist + NT;
  float* stat_s = (float*)(ntile_s + 4);       // [2][64]: lse * log2(e), delta
  int* dst_s = (int*)(stat_s + 128);
  const unsigned lds0 = (unsigned)(uintptr_t)smem;

  int slot_id[4], slot_row[4];
  request_ids(ids, ql, K, slot_id);
  request_ids(dst, ql, K, slot_row);
  __builtin_amdgcn_sched_barrier(0);
  // Q and dO travel to LDS as they are, in groups of 128 bytes of all 64 rows (Q: 9, dO: 8), chunk c of row r in slot c ^ (r & 7):
  // both orientations are read from there.  Wave w moves rows 8 w .. 8 w + 7.
  if (8 * wave < H) {
    const __bf16* q_rows = uniform_ptr(q + (size_t)qi * H * DQK);
    const __bf16* do_rows = uniform_ptr(dout + (size_t)qi * H * DV);
    const unsigned lb = __builtin_amdgcn_readfirstlane(lds0 + (unsigned)wave * 1024u);
    const unsigned row = (unsigned)(8 * wave + (lane >> 3)), col = (unsigned)(((lane & 7) ^ (lane >> 3)) * 16);
#pragma unroll
    for (int k = 0; k < 9; k++) dma16_once(lb + k * 8192, row * (DQK * 2) + col + k * 128, q_rows);
#pragma unroll
    for (int k = 0; k < 8; k++) dma16_once(lb + (9 + k) * 8192, row * (DV * 2) + col + k * 128, do_rows);
  }
  const int h = hw * 16 + m;
  const size_t hrow = (size_t)qi * H + h;
  bf16x8 qreg[KS], doreg[VS], oreg[VS];
  if (scores) {
    const bf16x8* op = (const bf16x8*)(out + hrow * DV) + kg;
#pragma unroll
    for (int ks = 0; ks < VS; ks++) oreg[ks] = op[4 * ks];
  }
  const float lse_h = lse[hrow];
  __builtin_amdgcn_sched_barrier(0);
  const int ntiles = stage_requested_ids(slot_id, K, Skv, q_start + qi, idx_s, tmask, tlist, ntile_s);
#pragma unroll
  for (int i = 0; i < 4; i++)                  // invalid slots land in a scratch row: the store count stays fixed
    if (tid + 512 * i < K) dst_s[tid + 512 * i] = slot_row[i] >= 0 ? slot_row[i] : dummy_row;
  DSA_WAIT_VMCNT(0);
  if (ntiles == 0) return;
  __syncthreads();
  if (scores) {
    const unsigned char* rb = smem + h * 128;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      qreg[ks] = *(const bf16x8*)(rb + (ks >> 1) * 8192 + (((4 * (ks & 1) + kg) ^ (h & 7)) << 4));
      asm volatile("" : "+a"(qreg[ks]));
    }
    float part = 0.f;                          // delta = rowsum(O . dO)
#pragma unroll
    for (int ks = 0; ks < VS; ks++) {
      doreg[ks] = *(const bf16x8*)(rb + (9 + (ks >> 1)) * 8192 + (((4 * (ks & 1) + kg) ^ (h & 7)) << 4));
#pragma unroll
      for (int e = 0; e < 8; e++) part = fmaf((float)oreg[ks][e], (float)doreg[ks][e], part);
      if (ks < DO_ACC) asm volatile("" : "+a"(doreg[ks]));
      else asm volatile("" : "+v"(doreg[ks]));
    }
    part += __shfl_xor(part, 16, 64);
    part += __shfl_xor(part, 32, 64);
    if (kg == 0) {
      stat_s[h] = lse_h * LOG2E;
      stat_s[64 + h] = part;
    }
  }
  // ---- operands of the rows: 16 columns by k-step ks of 32 heads, in the chunk order of P and dS ----
  typedef short i16x8 __attribute__((ext_vector_type(8)));
  auto tr_pair = [&](const unsigned char* p0, const unsigned char* p1) {
    const i16x4 x0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(i16x4, p0));
    const i16x4 x1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(i16x4, p1));
    return __builtin_bit_cast(bf16x8, (i16x8)__builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  // Row 4 j + e of the operand is column {0, 8, 4, 12}[j] + e of the 16, so that lanes 32 apart end up with neighbouring columns.
  // The heads of lane chunk kg are 32 ks + 16 (kg / 2) + 4 (kg % 2) + {0 .. 3, 8 .. 11}.
  bf16x8 xq[4][HG], xo[4][HG];
  {
    const int ii = lane & 15, jj = ((ii & 1) << 1) | ((ii >> 1) & 1);
    const int hd = 16 * (kg >> 1) + 4 * (kg & 1) + (ii >> 2);
    auto column_operand = [&](int group, int c, int ks) {
      const unsigned char* p = smem + group * 8192 + (32 * ks + hd) * 128 + (((2 * c + (jj >> 1)) ^ (hd & 7)) << 4) + (jj & 1) * 8;
      return tr_pair(p, p + 8 * 128);
    };
    bf16x8 xr[HG];
#pragma unroll
    for (int ks = 0; ks < HG; ks++) {
#pragma unroll
      for (int c = 0; c < 4; c++) {
        xq[c][ks] = column_operand(wave, c, ks);
        xo[c][ks] = column_operand(9 + wave, c, ks);
      }
      xr[ks] = column_operand(8, wave & 3, ks);      // rotary columns 16 (wave % 4) ..
    }
#pragma unroll
    for (int ks = 0; ks < HG; ks++) {
      asm volatile("" : "+v"(xq[0][ks]), "+v"(xq[1][ks]), "+v"(xq[2][ks]), "+v"(xq[3][ks]), "+v"(xr[ks]));
      asm volatile("" : "+v"(xo[0][ks]), "+v"(xo[1][ks]), "+v"(xo[2][ks]), "+v"(xo[3][ks]));
    }
    __syncthreads();                           // every wave has its operands: the space is the ring's from here on
#pragma unroll
    for (int ks = 0; ks < HG; ks++) xr_s[64 * ks] = xr[ks];
  }

  // transfers of a tile: waves 0-3 take groups 0-4, waves 4-7 groups 5-8
  const int gkey = (tid & 255) >> 3, gsub = tid & 7;
  const int grp0 = hh * 5;
  const unsigned gslot = (unsigned)((gsub ^ (gkey & 7)) * 16) + (unsigned)(grp0 * 128);
  auto issue = [&](int n) {
    int kid = idx_s[tlist[n] * BI + gkey];
    kid = kid < 0 ? 0 : kid;
    const unsigned goff = __umul24((unsigned)kid, DQK * 2) + gslot;       // (fewer than 2^24 rows: kv is at most 4 GiB)
    const unsigned lb = __builtin_amdgcn_readfirstlane(lds0 + (unsigned)((n % STAGES) * TILE_BYTES + (wave & 3) * 1024 + grp0 * GRP_BYTES));
#pragma unroll
    for (int i = 0; i < 5 - hh; i++) dma16(lb + i * GRP_BYTES, goff + i * 128, kv);
  };
  for (int n = 0; n < STAGES - 1 && n < ntiles; n++) issue(n);

  // accumulator i of a lane is head 16 hw + 4 kg + i, for key 16 hh + m
  const float* stat = stat_s + hw * 16 + 4 * kg;
  const int krow = 16 * hh + m;
  unsigned boff[2];
#pragma unroll
  for (int par = 0; par < 2; par++) boff[par] = (unsigned)(krow * 128 + (((4 * par + kg) ^ (krow & 7)) << 4));
  const unsigned half_chunk = (unsigned)((2 * hw + (kg & 1)) * 512 + krow * 16 + (kg >> 1) * 8);   // of the lane's key and 4 heads
  const unsigned coff = (unsigned)(kg * 512 + m * 16);                 // coefficients of k-step ks (32 heads) and half tile kt: + 2048 ks + 256 kt
  // the lane's 16 bytes of a row for a pair of column tiles: the lower half-wave has the first one's, lanes kg + 2 and kg trade
  const unsigned coloff = (unsigned)(wave * 128 + g * 32 + (kg & 1) * 16);
  const unsigned rotoff = (unsigned)(DV * 2 + (wave & 3) * 32 + ((kg & 1) * 2 + (kg >> 1)) * 8);
  const float c2 = sm_scale * LOG2E;

  // S, dP -> P, dS of tile n
  auto phase_pds = [&](int n) {
    const int tile = __builtin_amdgcn_readfirstlane(tlist[n]);
    const unsigned mask = __builtin_amdgcn_readfirstlane(tmask[tile]);
    const unsigned char* tb = smem + (n % STAGES) * TILE_BYTES;
    f32x4 sacc, dpacc;
    constexpr int FD = 3;                      // operand reads in flight
    bf16x8 f[FD];
    auto operand = [&](int ks) { return *(const bf16x8*)(tb + (ks >> 1) * GRP_BYTES + boff[ks & 1]); };
#pragma unroll
    for (int j = 0; j < FD; j++) f[j] = operand(j);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      mfma16_a(sacc, qreg[ks], f[ks % FD], ks == 0);
      if (ks < DO_ACC) mfma16_a(dpacc, doreg[ks], f[ks % FD], ks == 0);
      else if (ks < VS) mfma16_v(dpacc, doreg[ks], f[ks % FD], false);
      if (ks + FD < KS) f[ks % FD] = operand(ks + FD);
      __builtin_amdgcn_sched_barrier(0);
    }
    mfma16_done(sacc, dpacc);
    const f32x4 lse2 = *(const f32x4*)stat, delta = *(const f32x4*)(stat + 64);
    const bool valid = (mask >> krow) & 1u;
    float pf[4], df[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      pf[i] = valid ? __builtin_amdgcn_exp2f(fmaf(sacc[i], c2, -lse2[i])) : 0.f;
      df[i] = pf[i] * (dpacc[i] - delta[i]) * sm_scale;
    }
    const uint2 pw = make_uint2(cvt_pk_bf16(pf[0], pf[1]), cvt_pk_bf16(pf[2], pf[3]));
    const uint2 dw = make_uint2(cvt_pk_bf16(df[0], df[1]), cvt_pk_bf16(df[2], df[3]));
    unsigned char* xb = xch + (n & 1) * FUSED_XCH + half_chunk;
    *(uint2*)xb = dw;
    *(uint2*)(xb + pds_kind_bytes(2)) = pw;
    *(uint2*)(pds + (size_t)tile * pds_kind_bytes(HG) + half_chunk) = dw;
    __builtin_amdgcn_sched_barrier(0);
  };
  // the rows of tile n
  auto phase_rows = [&](int n) {
    const unsigned char* xb = xch + (n & 1) * FUSED_XCH;
    const int* drow = dst_s + tlist[n] * BI;
#pragma unroll
    for (int kt = 0; kt < 2; kt++) {
      bf16x8 cs[HG], cp[HG];
#pragma unroll
      for (int ks = 0; ks < HG; ks++) {
        cs[ks] = *(const bf16x8*)(xb + ks * 2048 + coff + kt * 256);
        cp[ks] = *(const bf16x8*)(xb + pds_kind_bytes(2) + ks * 2048 + coff + kt * 256);
      }
      unsigned char* row = rows + (size_t)drow[16 * kt + m] * ROW_BYTES;
#pragma unroll
      for (int cp2 = 0; cp2 < 2; cp2++) {
        f32x4 acc[2];
#pragma unroll
        for (int ks = 0; ks < HG; ks++)
#pragma unroll
          for (int i = 0; i < 2; i++) mfma16_v(acc[i], xq[2 * cp2 + i][ks], cs[ks], ks == 0);
#pragma unroll
        for (int ks = 0; ks < HG; ks++)
#pragma unroll
          for (int i = 0; i < 2; i++) mfma16_v(acc[i], xo[2 * cp2 + i][ks], cp[ks], false);
        mfma16_done(acc[0], acc[1]);
        unsigned w0[2], w1[2];
#pragma unroll
        for (int e = 0; e < 2; e++) {
          w0[e] = cvt_pk_bf16(acc[0][2 * e], acc[0][2 * e + 1]);
          w1[e] = cvt_pk_bf16(acc[1][2 * e], acc[1][2 * e + 1]);
          swap_halves(w0[e], w1[e]);
        }
        *(uint4*)(row + cp2 * 64 + coloff) = make_uint4(w0[0], w0[1], w1[0], w1[1]);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (kt == hh) {
        f32x4 acc;
#pragma unroll
        for (int ks = 0; ks < HG; ks++) mfma16_v(acc, xr_s[64 * ks], cs[ks], ks == 0);
        mfma16_done(acc);
        *(uint2*)(row + rotoff) = make_uint2(cvt_pk_bf16(acc[0], acc[1]), cvt_pk_bf16(acc[2], acc[3]));
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };

#pragma clang loop unroll(disable)
  for (int n = 0; n <= ntiles; n++) {
    asm volatile("" : "+s"(n));                // one copy of the loop: peeled ones cost registers
    // A wave's operations behind the transfer of tile n, which went out two steps ago.  A step is 5 transfers (4 of waves 4-7), the
    // dS store (not of every wave with one group) and 5 row stores.  The first tiles and the last one, behind which there are fewer,
    // wait for all.
    if (n < ntiles) {
      if (n >= 3 && n + 1 < ntiles) {
        if (HG == 2) { if (hh == 0) { DSA_WAIT_VMCNT(17); } else { DSA_WAIT_VMCNT(16); } }
        else { if (hh == 0) { DSA_WAIT_VMCNT(15); } else { DSA_WAIT_VMCNT(14); } }
      }
      else { DSA_WAIT_VMCNT(0); }
    }
    __syncthreads();
    if (n + STAGES - 1 < ntiles) issue(n + STAGES - 1);       // ahead of the step's stores, which the transfers would queue behind
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (hh == 0) {
      if (n < ntiles && scores) phase_pds(n);
      if (n > 0) phase_rows(n - 1);
    } else {
      if (n > 0) phase_rows(n - 1);
      if (n < ntiles && scores) phase_pds(n);
    }
  }
}

// ---------------------------------------------------------------------------------------------
// P, dS and the rows of the pairs, for 96 and 128 heads
// ---------------------------------------------------------------------------------------------
// Both orientations of 128 heads are 557 KB; registers (512 KB) and LDS (160 KB) hold them together with the tile because what
// lies in LDS serves either orientation: row reads for the products over d, transposing reads for those over the heads.  In LDS:
// the first 32 of every 64 columns of dO (64 KB) and the rotary columns of Q (16 KB).  In registers (192 per lane): Q and the
// other columns of dO by rows (wave w: heads 16 w ..) and by columns (wave w: columns 64 w ..).
// That leaves room for one tile and one buffer of P and dS, so a step has two halves with a barrier each: S, dP -> P, dS of the
// tile; then the transfer of the next tile starts and the rows are multiplied and stored under it.
// The set-up of a query is one round trip to memory: ids, Q, dO and O are requested together (410 KB), dO goes on to LDS from the
// registers that its sums with O had it in, and the first tile travels meanwhile.  (ids behind the operands, dO read twice and the first tile
// behind all that were four: 12000 queries of three documents x 256 slots 2692 us and 2455 now, 5000 x 1024 1898 and 1816, 5000 of
// window and compressed keys 1786 and 1743, 2077 x 512 x 64 heads 291 and 286, 8192 x 2048 8.89 ms and 8.81.  The first 32 of every
// 64 columns read again from the L2 instead of kept, which saves 32 registers on the way: 1 - 5 % slower.)
// 7700 cycles a step at 8192 queries x 2048 slots x 128 heads, 4352 of them in the matrix pipe (46 % busy): the 816 LDS reads,
// 36 KB of transfers and 37 KB of stores of a step share the way between the registers and LDS or cache, and hold each other up: LDS reads slow down by half while a tile arrives.  8.7 ms where
// the two passes took 4.15 + 5.55, with 8 KB less to write and 16 KB less to read per tile.  Slower than this form, though each
// has fewer LDS reads: 32x32x16 products for the rows (644, stores of 32 bytes in 32 rows), all column tiles at once (704, the
// stores of a step together at its end), and waves 0-3 for P, dS beside waves 4-7 for the rows, with the next tile's first groups
// ahead (640): 8 - 12 % each.
constexpr int WIDE_ROT = 65536;                        // behind dO's columns [4 pairs of 64][128 heads][2 x 32 columns]
constexpr int WIDE_TILE = WIDE_ROT + 16384;
constexpr int WIDE_XCH = WIDE_TILE + TILE_BYTES;
constexpr int WIDE_LISTS = 128 * DQK * 2;              // Q of the query fits in front of the lists before the rest is there
static_assert(WIDE_XCH + 2 * pds_kind_bytes(4) <= WIDE_LISTS && WIDE_TILE + 65536 <= WIDE_LISTS, "the lists lie behind everything else");
inline size_t wide_lds_bytes(int K) { return (size_t)WIDE_LISTS + ids_lds_bytes(K) + 1024 + 2048; }
__host__ __device__ constexpr size_t unit_lds_bytes(int slots) { return (size_t)WIDE_LISTS + (size_t)slots * 4 + 1024 + 2048 + BI * EXP_BYTES; }
static_assert(unit_lds_bytes(UNIT_SLOTS) <= 160 * 1024, "the list of a joint unit");

// Largest magnitude over the values of every lane with the same lane % 16, as bits, and at least 2^-112 (below that the scale stays as it
// is).  Values that are not finite do not count: they are what they are in fp16.
template <int N>
__device__ __forceinline__ unsigned group_max(const f32x4 (&x)[N]) {
  constexpr float LEAST = 0x1p-112f;
  float most = LEAST;
#pragma unroll
  for (int i = 0; i < N; i++)
#pragma unroll
    for (int e = 0; e < 4; e += 2) asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(most) : "v"(x[i][e]), "v"(x[i][e + 1]));      // (passes over NaN)
  if (__any(most == INFINITY)) {
    most = LEAST;
#pragma unroll
    for (int i = 0; i < N; i++)
#pragma unroll
      for (int e = 0; e < 4; e++) most = fabsf(x[i][e]) < INFINITY ? fmaxf(most, fabsf(x[i][e])) : most;
  }
  float other = most;
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1\n\tv_max_f32 %0, %0, %1\n\tv_mov_b32 %1, %0\n\ts_nop 1\n\t"
               "v_permlane16_swap_b32 %0, %1\n\ts_nop 1\n\tv_max_f32 %0, %0, %1" : "+v"(most), "+v"(other));
  return __builtin_bit_cast(unsigned, most);
}
// 2^(14 - k) for a largest magnitude of 2^k .. 2^(k + 1), whose exponent bits are kept with the row
__device__ __forceinline__ float group_scale(unsigned most) { return __builtin_bit_cast(float, (268u << 23) - (most & 0x7f800000u)); }
// (a scale, b scale) in fp16.  (v_fma_mixlo_f16 / mixhi, a product and its rounding in one, are no faster than these three: scores and rows
// of 3072 queries x 640 slots 566 and 562 us.)
__device__ __forceinline__ unsigned scaled_pk_f16(float a, float b, float scale) {
  const f32x2_t v = {a * scale, b * scale};
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v, f16x2_t));
}

// Zero where a bf16 value is not finite (exponent all ones), in 16 bytes of LDS
__device__ __forceinline__ void drop_nonfinite(unsigned char* p) {
  uint4 v = *(uint4*)p;
  unsigned* w = (unsigned*)&v;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    if ((w[i] & 0x7f80u) == 0x7f80u) w[i] &= 0xffff0000u;
    if ((w[i] & 0x7f800000u) == 0x7f800000u) w[i] &= 0xffffu;
  }
  *(uint4*)p = v;
}

// All arrays from the query's first head on.  G > 1: a joint unit of G queries with 128 / G heads each (H = 128, K its slots).  The
// products over the heads then meet heads whose query has not selected the key: their P and dS are zero, and what is not finite in
// their rows of Q and dO would still make the pair row NaN.  Such values become zero in LDS, where the column operands are read; the
// query's own pairs are NaN all the same, through lse (NaN for a head with such a value in Q) or delta (not finite with one in dO).
template <int hh, int G>
__device__ __forceinline__ void pds_rows_wide_body(
    const __bf16* __restrict__ q, const __bf16* __restrict__ kv, const int* __restrict__ ids,
    const __bf16* __restrict__ out, const __bf16* __restrict__ dout, const float* __restrict__ lse,
    unsigned char* __restrict__ pds, const int* __restrict__ dst, unsigned char* __restrict__ rows, unsigned char* __restrict__ exps,
    int H, int Skv, int K, int qpos, float sm_scale, int dummy_row, unsigned char* smem) {
  constexpr int VS = DV / 32;
  constexpr int XQ_ACC = 7;                    // column operands of Q in accumulation registers, beside all row operands: 124
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int NT = K / BI;
  unsigned char* xch = smem + WIDE_XCH;
  int* idx_s = (int*)(smem + WIDE_LISTS);
  unsigned* tmask = (unsigned*)(idx_s + K);    // (no masks and list of tiles in a joint unit: its slots are dense)
  int* tlist = (int*)(tmask + NT);
  int* ntile_s = tlist + NT;
  float* stat_s = G > 1 ? (float*)(idx_s + K) : (float*)(ntile_s + 4);       // [2][128]: lse * log2(e), delta
  int* dst_s = (int*)(stat_s + 256);           // [2][256]: destination rows from the tile's first slot on
  unsigned char* exp_s = (unsigned char*)(dst_s + 512);                      // G > 1: [32][EXP_BYTES], exponents of the tile's rows
  const unsigned lds0 = (unsigned)(uintptr_t)smem;
  // Registers are short: what depends on the lane is worked out anew for every part.
  auto fresh_lane = []() {
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
  };

  // Rows of Q and dO travel to LDS in groups of 128 bytes of all 128 rows, chunk c of row r in slot c ^ (r & 7).  Wave w moves rows
  // 8 w .. 8 w + 7 and 64 + 8 w ..; heads beyond H repeat the last one (their P and dS are zero).
  const unsigned char* q_rows = (const unsigned char*)uniform_ptr(q);
  const unsigned lb = __builtin_amdgcn_readfirstlane(lds0 + (unsigned)wave * 1024u);
  // The ids are requested first, then Q, O and dO: one round trip to memory.
  constexpr int NV = G > 1 ? UNIT_SLOTS / PDS_THREADS : 4;
  int v[NV], pad = 0;
  if constexpr (G > 1) {
    pad = ids[0];
#pragma unroll
    for (int i = 0; i < NV; i++) v[i] = ids[min(tid + PDS_THREADS * i, K - 1)];
  } else {
    request_ids(ids, 0, K, v);
  }
  __builtin_amdgcn_sched_barrier(0);
  auto group_base = [](int p) { return p < 4 ? p * 16384 : p < 8 ? WIDE_TILE + (p - 4) * 16384 : WIDE_ROT; };
  {
    const int l = fresh_lane();
#pragma unroll
    for (int rb = 0; rb < 2; rb++) {
      const unsigned src = (unsigned)min(64 * rb + 8 * wave + (l >> 3), H - 1) * (DQK * 2) + ((l & 7) ^ (l >> 3)) * 16;
#pragma unroll
      for (int p = 0; p < 9; p++) dma16_once(lb + rb * 8192 + group_base(p), src + p * 128, q_rows);
    }
  }
  const int m = lane & 15, kg = lane >> 4;
  const int h = wave * 16 + m;
  const bool head_ok = h < H;
  const size_t hrow = min(h, H - 1);
  int ntiles = NT;
  bf16x8 dkeep[VS / 2], doreg[VS / 2];         // dO, the even and the odd 32 columns
  unsigned bad_do = 0;                         // G > 1: which of the wave's heads have values in dO that are not finite
  auto of_heads = [](unsigned long long b) { return (unsigned)((b | b >> 16 | b >> 32 | b >> 48) & 0xffffu); };   // lanes (m, kg) -> heads m
  {
    const bf16x8* op = (const bf16x8*)(out + hrow * DV) + kg;
    const bf16x8* dp = (const bf16x8*)(dout + hrow * DV) + kg;
    bf16x8 o[VS], d[VS];
#pragma unroll
    for (int ks = 0; ks < VS; ks++) { d[ks] = dp[4 * ks]; o[ks] = op[4 * ks]; }
    const float lse_h = lse[hrow];
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (G > 1) {
      // slots behind the last key repeat the first one, for none of the queries
#pragma unroll
      for (int i = 0; i < NV; i++) {
        const int t = tid + PDS_THREADS * i;
        if (t < K) idx_s[t] = v[i] < 0 ? pad & UNIT_KEY : v[i];
      }
    } else {
      ntiles = stage_requested_ids(v, K, Skv, qpos, idx_s, tmask, tlist, ntile_s);
    }
    float part = 0.f;                          // delta = rowsum(O . dO)
#pragma unroll
    for (int ks = 0; ks < VS; ks++) {
#pragma unroll
      for (int e = 0; e < 8; e++) part = fmaf((float)o[ks][e], (float)d[ks][e], part);
      if (ks & 1) {
        doreg[ks >> 1] = d[ks];
        asm volatile("" : "+a"(doreg[ks >> 1]));
      } else {
        dkeep[ks >> 1] = d[ks];
      }
    }
    part += __shfl_xor(part, 16, 64);
    part += __shfl_xor(part, 32, 64);
    if (G > 1 ? fresh_lane() < 16 : kg == 0) {
      stat_s[h] = head_ok ? lse_h * LOG2E : INFINITY;
      stat_s[128 + h] = head_ok ? part : 0.f;
    }
    if (G > 1) bad_do = of_heads(__ballot(!(fabsf(part) < INFINITY)));
  }
  DSA_WAIT_VMCNT(0);
  if (ntiles == 0) return;
  __syncthreads();

  // ---- resident operands: rows of Q (32 columns each) and of dO (the columns that are not in LDS), columns of both ----
  typedef short i16x8 __attribute__((ext_vector_type(8)));
  auto tr_pair = [&](const unsigned char* p) {             // 16 columns by the heads of chunk kg: 8 rows apart
    const i16x4 x0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(i16x4, p));
    const i16x4 x1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(i16x4, p + 8 * 128));
    return __builtin_bit_cast(bf16x8, (i16x8)__builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  // Operand rows as in the body for 64 heads: row 4 j + e is column {0, 8, 4, 12}[j] + e of 16, chunk kg of k-step ks holds heads
  // 32 ks + 16 (kg / 2) + 4 (kg % 2) + {0 .. 3, 8 .. 11}
  auto tr_off = [](int l, int chunk) {
    const int ii = l & 15, jj = ((ii & 1) << 1) | ((ii >> 1) & 1), hd = 16 * (l >> 5) + 4 * ((l >> 4) & 1) + (ii >> 2);
    return (unsigned)(hd * 128 + (((chunk + (jj >> 1)) ^ (hd & 7)) << 4) + (jj & 1) * 8);
  };
  auto row_off = [](int l, int par) {          // row l % 16 of 16, an even or odd 32 columns of a group
    return (unsigned)((l & 15) * 128 + (((4 * par + (l >> 4)) ^ (l & 7)) << 4));
  };
  bf16x8 qreg[VS], xq[4][4], xo[2][4];
  {
    const int l = fresh_lane();
    const unsigned off[2] = {2048 * wave + row_off(l, 0), 2048 * wave + row_off(l, 1)};
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    u16x2 most = {0, 0};                       // largest magnitude, as bits
    auto look = [&](const bf16x8& x) {
      const uint4 v = __builtin_bit_cast(uint4, x);
      const unsigned wd[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int i = 0; i < 4; i++) most = __builtin_elementwise_max(most, __builtin_bit_cast(u16x2, wd[i] & 0x7fff7fffu));
    };
#pragma unroll
    for (int ks = 0; ks < VS; ks++) {
      qreg[ks] = *(const bf16x8*)(smem + group_base(ks >> 1) + off[ks & 1]);
      if (G > 1) look(qreg[ks]);
      asm volatile("" : "+a"(qreg[ks]));
    }
    if constexpr (G > 1) {
#pragma unroll
      for (int par = 0; par < 2; par++) look(*(const bf16x8*)(smem + WIDE_ROT + off[par]));
      const unsigned bad = of_heads(__ballot(most[0] >= 0x7f80 || most[1] >= 0x7f80));
      if (bad) {                               // the wave's own rows, all columns
        if (l < 16 && (bad >> l & 1u)) stat_s[16 * wave + l] = NAN;
#pragma unroll 1
        for (int p = 0; p < 9; p++)
#pragma unroll 1
          for (int c = l; c < 128; c += 64) drop_nonfinite(smem + group_base(p) + 2048 * wave + c * 16);
      }
      __syncthreads();
    }
  }
  {
    const int l = fresh_lane();
    const unsigned char* xg = smem + (wave < 4 ? wave * 16384 : WIDE_TILE + (wave - 4) * 16384);
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
      for (int ks = 0; ks < 4; ks++) {
        xq[c][ks] = tr_pair(xg + ks * 4096 + tr_off(l, 2 * c));
        if (4 * c + ks < XQ_ACC) asm volatile("" : "+a"(xq[c][ks]));
        else asm volatile("" : "+v"(xq[c][ks]));
      }
  }
  __syncthreads();                             // Q is in registers: its place is free for the first tile and for dO
  // transfers of a tile: waves 0-3 take groups 0-4, waves 4-7 groups 5-8; wave 7 the tile's destination rows
  const int grp0 = hh * 5;
  const unsigned tile_lb = __builtin_amdgcn_readfirstlane(lds0 + (unsigned)(WIDE_TILE + (wave & 3) * 1024 + grp0 * GRP_BYTES));
  auto issue = [&](int n) {
    const int tile = G > 1 ? n : __builtin_amdgcn_readfirstlane(tlist[n]), l = fresh_lane();
    int kid = idx_s[tile * BI + 8 * (wave & 3) + (l >> 3)];
    kid = G > 1 ? kid & UNIT_KEY : kid < 0 ? 0 : kid;
    const unsigned goff = __umul24((unsigned)kid, DQK * 2) + (unsigned)(((l & 7) ^ (l >> 3)) * 16 + grp0 * 128);       // (fewer than 2^24 rows: kv is at most 4 GiB)
#pragma unroll
    for (int i = 0; i < 5 - hh; i++) dma16(tile_lb + i * GRP_BYTES, goff + i * 128, kv);
    // 1 KB from the tile's first slot on (behind the last query's slots the workspace goes on with the sorted list)
    if (wave == 7) dma16(lds0 + (unsigned)((unsigned char*)dst_s - smem) + (n & 1) * 1024, (unsigned)l * 16, dst + tile * BI);
  };
  issue(0);
  // dO from the registers: of every 64 columns first the second 32, for the column operands, then the first 32, to stay.  Chunk c of a row
  // of group j (columns 128 j + 64 (c / 4) + 8 (c % 4) .., of the first or second 32) lies in slot c ^ (row & 7).
  auto put_do = [&](const bf16x8 (&x)[VS / 2]) {
    const int l = fresh_lane();
    unsigned char* row = smem + (wave * 16 + (l & 15)) * 128;
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int half = 0; half < 2; half++) *(bf16x8*)(row + j * 16384 + (((4 * half + (l >> 4)) ^ (l & 7)) << 4)) = x[2 * j + half];
    if constexpr (G > 1) {
      if (bad_do) {                            // the wave's own rows
#pragma unroll 1
        for (int j = 0; j < 4; j++)
#pragma unroll 1
          for (int c = l; c < 128; c += 64) drop_nonfinite(smem + j * 16384 + 2048 * wave + c * 16);
      }
    }
  };
  put_do(doreg);
  __syncthreads();
  {
    const int l = fresh_lane();
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
      for (int ks = 0; ks < 4; ks++) {
        xo[c][ks] = tr_pair(smem + (wave >> 1) * 16384 + ks * 4096 + tr_off(l, 4 * (wave & 1) + 2 * c));
        asm volatile("" : "+v"(xo[c][ks]));
      }
  }
  __syncthreads();
  put_do(dkeep);

  const int ln = fresh_lane();
  const int lm = ln & 15, lk = ln >> 4, lg = ln >> 5;

  // accumulator i of a lane is head 16 wave + 4 lk + i, for key 16 kt + lm
  unsigned boff[2], loff[2];                   // row operands of even and odd 32 columns: of a key, of the lane's head
#pragma unroll
  for (int par = 0; par < 2; par++) {
    boff[par] = (unsigned)WIDE_TILE + row_off(ln, par);
    loff[par] = (unsigned)(2048 * wave) + row_off(ln, par);
  }
  const unsigned chunk = (unsigned)((2 * wave + (lk & 1)) * 512 + (16 * lg + lm) * 16);  // after the trade: 8 heads of key 16 lg + lm
  const unsigned coff = (unsigned)(lk * 512 + lm * 16);                // coefficients of k-step ks and half tile kt: + 2048 ks + 256 kt
  const unsigned coloff = (unsigned)(wave * 128 + lg * 32 + (lk & 1) * 16);
  const unsigned rotoff = (unsigned)(DV * 2 + (wave & 3) * 32 + ((lk & 1) * 2 + (lk >> 1)) * 8);
  // column operands: dO of the first column tile (the second one's: ^ 32), rotary columns
  const unsigned tr_do = (unsigned)((wave >> 1) * 16384) + tr_off(ln, 4 * (wave & 1)), tr_rot = (unsigned)WIDE_ROT + tr_off(ln, 2 * (wave & 3));
  const float c2 = sm_scale * LOG2E;

  // S, dP -> P, dS of tile n
  auto phase_pds = [&](int n) {
    const int tile = G > 1 ? n : __builtin_amdgcn_readfirstlane(tlist[n]);
    const unsigned mask = G > 1 ? 0u : __builtin_amdgcn_readfirstlane(tmask[tile]);
    f32x4 sacc[2], dpacc[2];
    constexpr int NJ = 2 * (DQK / 32), FD = 3;
    bf16x8 f[FD], x;                           // key rows of step j = 2 ks + kt; row operand from LDS: dO of even ks, Q of the rotary ks
    auto operand = [&](int j) { return *(const bf16x8*)(smem + (j >> 2) * GRP_BYTES + (j & 1) * 2048 + boff[(j >> 1) & 1]); };
    x = *(const bf16x8*)(smem + loff[0]);
#pragma unroll
    for (int j = 0; j < FD; j++) f[j] = operand(j);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NJ; j++) {
      const int ks = j >> 1, kt = j & 1;
      if (ks < VS) {
        mfma16_a(sacc[kt], qreg[ks < VS ? ks : 0], f[j % FD], ks == 0);
        if (ks & 1) mfma16_a(dpacc[kt], doreg[ks < VS ? ks >> 1 : 0], f[j % FD], false);
        else mfma16_v(dpacc[kt], x, f[j % FD], ks == 0);
      } else {
        mfma16_v(sacc[kt], x, f[j % FD], false);
      }
      if (j + FD < NJ) f[j % FD] = operand(j + FD);
      if (kt == 1 && ks < VS - 2 && (ks & 1) == 0) x = *(const bf16x8*)(smem + ((ks + 2) >> 2) * 16384 + loff[((ks + 2) >> 1) & 1]);
      if (kt == 1 && (ks == VS - 2 || ks == VS)) x = *(const bf16x8*)(smem + WIDE_ROT + loff[ks == VS]);
      __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("s_nop 15\n\ts_nop 3" : "+v"(sacc[0]), "+v"(sacc[1]), "+v"(dpacc[0]), "+v"(dpacc[1]));
    const f32x4 lse2 = *(const f32x4*)(stat_s + wave * 16 + 4 * lk), delta = *(const f32x4*)(stat_s + 128 + wave * 16 + 4 * lk);
    unsigned pw[2][2], dw[2][2];
#pragma unroll
    for (int kt = 0; kt < 2; kt++) {
      // (G > 1: the query of the wave's heads is wave * G / 8)
      const bool valid = G > 1 ? (idx_s[n * BI + 16 * kt + (fresh_lane() & 15)] >> (24 + wave * G / 8)) & 1 : (mask >> (16 * kt + lm)) & 1u;
      float pf[4], df[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        pf[i] = valid ? __builtin_amdgcn_exp2f(fmaf(sacc[kt][i], c2, -lse2[i])) : 0.f;
        df[i] = G > 1 && !valid ? 0.f : pf[i] * (dpacc[kt][i] - delta[i]) * sm_scale;
      }
      pw[kt][0] = cvt_pk_bf16(pf[0], pf[1]); pw[kt][1] = cvt_pk_bf16(pf[2], pf[3]);
      dw[kt][0] = cvt_pk_bf16(df[0], df[1]); dw[kt][1] = cvt_pk_bf16(df[2], df[3]);
    }
    // lanes 32 apart trade half tiles: 16 bytes of a key's heads for a lane
#pragma unroll
    for (int r2 = 0; r2 < 2; r2++) {
      swap_halves(pw[0][r2], pw[1][r2]);
      swap_halves(dw[0][r2], dw[1][r2]);
    }
    const uint4 d16 = make_uint4(dw[0][0], dw[0][1], dw[1][0], dw[1][1]);
    *(uint4*)(xch + chunk) = d16;
    *(uint4*)(xch + pds_kind_bytes(4) + chunk) = make_uint4(pw[0][0], pw[0][1], pw[1][0], pw[1][1]);
    i32x4* const d_out = (i32x4*)(pds + (size_t)tile * pds_kind_bytes(4) + chunk);
    if constexpr (G == 1) __builtin_nontemporal_store(__builtin_bit_cast(i32x4, d16), d_out);
    else *d_out = __builtin_bit_cast(i32x4, d16);
    __builtin_amdgcn_sched_barrier(0);
  };
  // the rows of tile n
  auto put_exponent = [&](unsigned most, int row, int group) { exp_s[(row + (fresh_lane() & 15)) * EXP_BYTES + group] = (unsigned char)(most >> 23); };
  auto phase_rows = [&](int n) {
#pragma unroll
    for (int kt = 0; kt < 2; kt++) {
      const int drow = dst_s[(n & 1) * 256 + 16 * kt + (G > 1 ? fresh_lane() & 15 : lm)];
      f32x4 acc[4], rot;
      bf16x8 cf[2], x[2];                      // coefficients of step k = 0 .. 3: dS . Q, 4 .. 7: P . dO; column operands from LDS
      auto coef = [&](int k) { return *(const bf16x8*)(xch + k * 2048 + kt * 256 + coff); };
      cf[0] = coef(0);
      if (kt == hh) x[0] = tr_pair(smem + tr_rot);
#pragma unroll
      for (int k = 0; k < 8; k++) {
        if (k < 7) cf[(k + 1) & 1] = coef(k + 1);
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int c = (i + 2) & 3;           // dO of column tiles 0 and 1 comes from LDS: those last
          if (k >= 4) mfma16_v(acc[c], c < 2 ? x[c & 1] : xo[c & 1][k & 3], cf[k & 1], false);
          else if (4 * c + k < XQ_ACC) mfma16_a(acc[c], xq[c][k & 3], cf[k & 1], k == 0);
          else mfma16_v(acc[c], xq[c][k & 3], cf[k & 1], k == 0);
          if (k >= 4 && k < 7 && c < 2) x[c & 1] = tr_pair(smem + (k - 3) * 4096 + (tr_do ^ (32u * c)));
        }
        if (kt == hh && k < 4) {
          mfma16_v(rot, x[k & 1], cf[k & 1], k == 0);
          if (k < 3) x[(k + 1) & 1] = tr_pair(smem + tr_rot + (k + 1) * 4096);
        }
        if (k == 3) {
          x[0] = tr_pair(smem + tr_do);
          x[1] = tr_pair(smem + (tr_do ^ 32u));
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      asm volatile("s_nop 15\n\ts_nop 3" : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]));
      unsigned char* row = rows + (size_t)(drow >= 0 ? drow : dummy_row) * ROW_BYTES;       // invalid slots: a scratch row
      float scale = 1.f;
      auto pack = [&](float a, float b) { return G > 1 ? scaled_pk_f16(a, b, scale) : cvt_pk_bf16(a, b); };
      if constexpr (G > 1) {
        const unsigned most = group_max(acc);
        scale = group_scale(most);
        put_exponent(most, 16 * kt, wave);
      }
#pragma unroll
      for (int pr = 0; pr < 2; pr++) {
        unsigned w0[2], w1[2];
#pragma unroll
        for (int e = 0; e < 2; e++) {
          w0[e] = pack(acc[2 * pr][2 * e], acc[2 * pr][2 * e + 1]);
          w1[e] = pack(acc[2 * pr + 1][2 * e], acc[2 * pr + 1][2 * e + 1]);
          swap_halves(w0[e], w1[e]);
        }
        *(uint4*)(row + pr * 64 + coloff) = make_uint4(w0[0], w0[1], w1[0], w1[1]);
      }
      if (kt == hh) {
        mfma16_done(rot);
        if constexpr (G > 1) {
          const f32x4 r1[1] = {rot};
          const unsigned most = group_max(r1);
          scale = group_scale(most);
          put_exponent(most, 16 * kt, 8 + (wave & 3));
        }
        *(uint2*)(row + rotoff) = make_uint2(pack(rot[0], rot[1]), pack(rot[2], rot[3]));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // exponents of the rows of tile n: 512 bytes by one wave, ahead of the next transfers (that tile's destination rows are in LDS until then)
  auto put_exponents = [&](int n) {
    const int l = fresh_lane();
    if (wave == 7 && l < BI) {
      const int drow = dst_s[(n & 1) * 256 + l];
      *(uint4*)(exps + (size_t)(drow >= 0 ? drow : dummy_row) * EXP_BYTES) = *(const uint4*)(exp_s + l * EXP_BYTES);
    }
    __builtin_amdgcn_sched_barrier(0);
  };

#pragma clang loop unroll(disable)
  for (int n = 0; n < ntiles; n++) {
    asm volatile("" : "+s"(n));                // one copy of the loop: peeled ones cost registers
    // behind the tile's transfers: the five row stores of the tile before
    if (n > 0) { DSA_WAIT_VMCNT(5); } else { DSA_WAIT_VMCNT(0); }
    __syncthreads();
    if (G > 1 && n > 0) put_exponents(n - 1);
    phase_pds(n);
    __syncthreads();
    if (n + 1 < ntiles) issue(n + 1);
    __builtin_amdgcn_sched_barrier(0);
    phase_rows(n);
  }
  if (G > 1) {
    __syncthreads();
    put_exponents(ntiles - 1);
  }
}

// ---------------------------------------------------------------------------------------------
// dKV[key] = sum of that key's rows, ascending query order
// ---------------------------------------------------------------------------------------------
// One key per workgroup (504 of its threads): 72 column chunks of 8 elements x 7 row groups (row r of the
// segment goes to group r % 7); the seven partial sums are combined in a fixed order, so the result
// depends only on the segment, never on scheduling.  Pure streaming reads of 1152-byte rows, RED_FLIGHT to
// twice that of them in flight per thread: a batch is loaded while the one before is summed, over the borders of keys, and
// always as a whole.  (One batch of 16 at a time, with a key's last rows loaded one by one, each behind the sum of the one
// before: with the dQ role beside it 1024 queries x 256 slots of 16 heads 60 us and 52 in batches of 8, 2077 x 512 of 64 heads 205 and
// 181, 3072 x 640 341 and 309; 8192 x 2048 of 128 heads, where the rows of a key fill many batches and the caches' gathers bound the
// launch, 4.50 ms either way.)
// The rows are read once: a non-temporal load keeps them from displacing other lines in the caches
// (a streaming read of this size runs at 6.8 TB/s with it against 6.1 TB/s without).
typedef unsigned u32x4_nt __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint4 row_load16(const void* p) {
  const u32x4_nt v = __builtin_nontemporal_load((const u32x4_nt*)p);
  return make_uint4(v.x, v.y, v.z, v.w);
}
constexpr int RED_GROUPS = 7;
// Row pieces a thread loads at a time; it sums one such batch while the next is on its way.  A batch never holds rows of two keys, so what a key
// lacks of it is loaded in vain: batches of 2 where there are few rows per key.  Whole backward, us, batches of 2 / 4 / 8 / one of 16 at a
// time and single loads: 2000 queries x 512 slots of 131072 keys (8 rows per key) 128 heads 1865 / 1962 / 2257 / 2049, 64 heads
// 1704 / 1805 / 2101 / 1772; 8000 x 256 of 131072 (16) x 64 heads 3269 / 3273 / 3608 / 3339, of 32768 (62) 2247 / 2247 / 2281 / 2484, of
// 8000 (256) 2025 / 1988 / 2020 / 1938; with 128 heads 2568 / 2559 / 2577 / 2765.
constexpr int RED_FLIGHT = 4, RED_FLIGHT_FEW = 2, RED_FEW_ROWS = 24;
constexpr int RED_KEYS = 4;                  // consecutive keys per workgroup
// A workgroup sums RED_KEYS consecutive keys (their rows follow one another in the buffer): every thread walks its
// share of the first key's rows, then of the next one's, without a barrier in between; one barrier, then the seven partial sums of each key are
// combined.  (One key per workgroup left the per-key latencies - segment bounds, first loads, barrier, combine -
// exposed once a key has few rows per launch: with the queries of 32768 tokens walked in four chunks the launch
// took 27.1 ms against 18.9 ms for one sweep; per key the sums and their order are the same as before.)
// SCALED: rows may be those of joint units; a chunk's exponent is loaded beside it.
template <bool SCALED, int RED_FLIGHT>
__device__ __forceinline__ void reduce_body(const unsigned char* __restrict__ rows, const unsigned char* __restrict__ exps, const int* __restrict__ start,
                                            float* __restrict__ dkv_acc, unsigned short* __restrict__ dkv, int key0, int n_keys,
                                            int accumulate, const int* __restrict__ dup_flag, unsigned char* smem) {
  constexpr int RED_BATCH = RED_FLIGHT * RED_GROUPS;
  float* part = (float*)smem;                  // [RED_KEYS][RED_GROUPS][DQK]
  const int tid = threadIdx.x;
  const int ch = tid % 72, grp = tid / 72;
  const int nk = min(RED_KEYS, n_keys - key0);
  const int bounds = start[min(key0 + min(tid & 63, RED_KEYS), n_keys)];        // lane k: the first row of key k
  const int bounds_end = __builtin_amdgcn_readlane(bounds, nk);
  if (grp < RED_GROUPS) {
    // A place in the workgroup's rows: batch [b, b + RED_BATCH) of key k, whose rows end at s1; k == nk: behind the last one.
    struct Place { int k, b, s1; };
    auto settle = [&](Place p) {                              // to the next key that has rows, if this one has none left
      while (p.k < nk && p.b >= p.s1) {
        p.k++;
        p.b = p.s1;
        p.s1 = __builtin_amdgcn_readlane(bounds, min(p.k + 1, RED_KEYS));
      }
      return p;
    };
    auto behind = [&](Place p) {
      p.b = min(p.b + RED_BATCH, p.s1);
      return settle(p);
    };
    // Always RED_FLIGHT loads, whatever is left (behind the rows the last one again, which `add` leaves out): only so can the
    // waits for one batch leave the next one's loads in flight.
    const unsigned lane_off = (unsigned)(grp * ROW_BYTES + ch * 16);
    const unsigned lane_exp = (unsigned)(grp * EXP_BYTES + (ch < DV / 8 ? ch >> 3 : 8 + ((ch - DV / 8) >> 1)));
    struct Batch { uint4 v[RED_FLIGHT]; unsigned e[RED_FLIGHT]; };
    auto load = [&](Batch& t, const Place& p) {
      const int b = p.k < nk ? p.b : bounds_end - 1, n = (p.k < nk ? p.s1 : bounds_end) - b;
      const unsigned last = (unsigned)((n - 1) * ROW_BYTES + ch * 16);
      const unsigned char* base = rows + (size_t)b * ROW_BYTES;
#pragma unroll
      for (int u = 0; u < RED_FLIGHT; u++) t.v[u] = row_load16(base + min((unsigned)(u * RED_GROUPS * ROW_BYTES) + lane_off, last));
      if constexpr (SCALED) {
        const unsigned end = (unsigned)((n - 1) * EXP_BYTES) + lane_exp % EXP_BYTES;
        const unsigned char* base_e = exps + (size_t)b * EXP_BYTES;
#pragma unroll
        for (int u = 0; u < RED_FLIGHT; u++) t.e[u] = base_e[min((unsigned)(u * RED_GROUPS * EXP_BYTES) + lane_exp, end)];
      }
    };
    float acc[8] = {};
    // FORM 0: bf16 rows; 1: fp16 with a power of two; 2: either
    auto add1 = [&](const uint4& x, unsigned exponent, auto form) {
      constexpr int FORM = decltype(form)::value;
      const unsigned w[4] = {x.x, x.y, x.z, x.w};
      const bool half = FORM == 1 || (FORM == 2 && exponent != 0u);
      const float scale = half ? __builtin_bit_cast(float, (exponent - 14u) << 23) : 1.f;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const float b0 = __builtin_bit_cast(float, w[e] << 16), b1 = __builtin_bit_cast(float, w[e] & 0xffff0000u);
        if constexpr (FORM == 0) {
          acc[2 * e] += b0;
          acc[2 * e + 1] += b1;
        } else {
          const f16x2_t h = __builtin_bit_cast(f16x2_t, w[e]);
          acc[2 * e] = fmaf(half ? (float)h[0] : b0, scale, acc[2 * e]);
          acc[2 * e + 1] = fmaf(half ? (float)h[1] : b1, scale, acc[2 * e + 1]);
        }
      }
    };
    auto add_as = [&](const Batch& t, const Place& p, auto form) {
      const int n = p.s1 - p.b;
      if (n >= RED_BATCH) {
#pragma unroll
        for (int u = 0; u < RED_FLIGHT; u++) add1(t.v[u], t.e[u], form);
      } else {
#pragma unroll
        for (int u = 0; u < RED_FLIGHT; u++)
          if (u * RED_GROUPS + grp < n) add1(t.v[u], t.e[u], form);
      }
    };
    auto add = [&](const Batch& t, const Place& p) {
      if constexpr (SCALED) {
        unsigned least = t.e[0];
#pragma unroll
        for (int u = 1; u < RED_FLIGHT; u++) least = min(least, t.e[u]);
        if (__any(least == 0u)) add_as(t, p, std::integral_constant<int, 2>{});
        else add_as(t, p, std::integral_constant<int, 1>{});
      } else {
        add_as(t, p, std::integral_constant<int, 0>{});
      }
    };
    auto put = [&](int k, int k_end) {                         // the sums of key k, and of keys without rows behind it
      for (; k < k_end; k++) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
          part[(k * RED_GROUPS + grp) * DQK + ch * 8 + e] = acc[e];
          acc[e] = 0.f;
        }
      }
    };
    Batch va, vb;
    Place p = settle({0, __builtin_amdgcn_readlane(bounds, 0), __builtin_amdgcn_readlane(bounds, 1)});
    put(0, p.k);
    if (p.k < nk) load(va, p);
    while (p.k < nk) {
      const Place n = behind(p);
      load(vb, n);
      add(va, p);
      put(p.k, n.k);
      if (n.k >= nk) break;
      p = behind(n);
      load(va, p);
      add(vb, n);
      put(n.k, p.k);
    }
  }
  __syncthreads();
  for (int o = tid; o < nk * DQK; o += (int)blockDim.x) {
    const int k = o / DQK, d = o % DQK;
    float sum = part[k * RED_GROUPS * DQK + d];
#pragma unroll
    for (int gq = 1; gq < RED_GROUPS; gq++) sum += part[(k * RED_GROUPS + gq) * DQK + d];
    if (dkv) {       // one sweep over all queries: the sum is complete (NaN everywhere when a query row held a repeated id)
      dkv[(size_t)(key0 + k) * DQK + d] = *dup_flag ? (unsigned short)0x7fc0 : f32_to_bf16_bits(sum);
    } else {
      float* p = dkv_acc + (size_t)(key0 + k) * DQK + d;
      *p = accumulate ? *p + sum : sum;
    }
  }
}

// ---------------------------------------------------------------------------------------------
// kernels: two roles each, chosen per workgroup
// ---------------------------------------------------------------------------------------------
// The dQ products are bound by LDS reads and leave HBM nearly idle; the sums are a pure stream of HBM reads and
// leave everything else idle; each occupies a whole compute unit (140 KB of LDS, or all its
// memory-level parallelism).  One launch carries the workgroups of both, spread evenly over the
// dispatch order, so that both kinds of work are in flight from the first workgroup to the last:
//   bwd_dq_reduce_kernel   dQ of all queries | dKV of all keys      (4.5 ms against 2.6 + 2.75)
// Within a role, the longest work (latest query, earliest key) comes first.
struct RoleSlot { bool first; int i; };
// nX workgroups of the first role and nY of the second, spread evenly over the launch: workgroup b belongs to the
// second role when the count floor(b * nY / (nX + nY)) steps up after it.
__device__ __forceinline__ RoleSlot role_slot(int b, int nX, int nY) {
  const long long tot = (long long)nX + nY;
  const int y0 = (int)((long long)b * nY / tot), y1 = (int)((long long)(b + 1) * nY / tot);
  if (y1 > y0) return {false, y0};
  return {true, b - y0};
}

// What workgroup i does: a query, and the tiles of its unit if it is the first one of a unit; query -1: nothing.  From the last query on, but for the
// first 256 workgroups if RAMP > 0, which spread over the last RAMP * K.  Where some queries are worked jointly they follow the
// work list, so that what has nothing to do comes at the end: a workgroup goes to the XCD, and there to the shader engine, that its number
// says, and waits for a place there.  (With one workgroup per query, those of a unit's other queries returning at once and eight in a row,
// G - 1 of G engines were idle: scores and rows of 4001 x 32 heads of window and compressed keys 1290 us instead of 410.)  The list has units and
// queries by themselves apart: 3000 x 512 of 2000 keys x 32 heads, a third of the groups units, whole backward 1217 us with both kinds mixed,
// 1158 in turns over the groups' queries, 1033 as it is; 1069 all joint, 989 all by themselves.
// RAMP: scores and rows read 410 KB per query or unit in front of 8 to 64 tiles of matrix work.  us, in strict order / first round spread over
// K / over 4 K queries: 5000 x 128 heads, window and compressed keys 1932 / 1922 / 1770, 3072 x 64 heads of these 590 / 591 / 556, 2077 x
// 512 x 64 heads 304 / 302 / 291, 1300 x 512 x 128 432 / 389 / 415, 8192 x 2048 x 128 8967 / 8906 / 8865, long documents of few slots
// and 9000 x 2048 x 64 the same; two rounds spread 6 % slower than one.  dQ, whose set-up is small, does not gain.
constexpr int PDS_RAMP = 4;
struct Work { int query, tiles; };
template <int G, int RAMP>
__device__ __forceinline__ Work work_of(int i, int cnt, int K, const int* __restrict__ work, bool joint) {
  if (G == 1 || !joint) return {cnt - 1 - (RAMP > 0 ? spread_start(i, cnt, 256, RAMP * K) : i), 0};
  const int n = __builtin_amdgcn_readfirstlane(work[0]), first = __builtin_amdgcn_readfirstlane(work[1]);
  if (i >= n) return {-1, 0};
  const int place = RAMP == 0 ? i : i < first ? spread_start(i, first, 256, RAMP * K / G) : first + spread_start(i - first, n - first, 256, RAMP * K / G);
  const int item = __builtin_amdgcn_readfirstlane(work[2 + place]);
  return {item >> 8, item & 255};
}

// G: queries of a group that may be a joint unit (4 / HG), or 1
template <int HG, int G>
__global__ __launch_bounds__(PDS_THREADS, 1) void bwd_pds_rows_kernel(
    const __bf16* __restrict__ q, const __bf16* __restrict__ kv, const int* __restrict__ ids,
    const __bf16* __restrict__ out, const __bf16* __restrict__ dout, const float* __restrict__ lse,
    unsigned char* __restrict__ pds, const int* __restrict__ dst, unsigned char* __restrict__ rows, unsigned char* __restrict__ exps,
    const int* __restrict__ work, const int* __restrict__ flags, size_t group_pds, int q0, int cnt, int H, int Skv, int K, int q_start,
    float sm_scale, int dummy_row) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const Work w = work_of<G, PDS_RAMP>((int)blockIdx.x, cnt, K, work, G > 1 && flags[1]);
  const int ql = w.query;
  if (G > 1 && ql < 0) return;
  // (two copies of every body: each copy meets the same barriers)
  if constexpr (HG == 4 || G > 1) {            // 128 heads: of the query or of a unit
    const int slots = G > 1 ? 32 * w.tiles : K;
    if (slots > 0) {
      const size_t hrow = (size_t)(q0 + ql) * H;
      unsigned char* unit = pds + (size_t)(ql / G) * group_pds;
      const __bf16 *q_rows = q + hrow * DQK, *out_rows = out + hrow * DV, *do_rows = dout + hrow * DV;
      const int *list = ids + (size_t)ql * K, *drow = dst + (size_t)ql * K;
      if (threadIdx.x < 256) pds_rows_wide_body<0, G>(q_rows, kv, list, out_rows, do_rows, lse + hrow, unit, drow, rows, exps, G > 1 ? 128 : H, Skv, slots, q_start + q0 + ql, sm_scale, dummy_row, smem);
      else pds_rows_wide_body<1, G>(q_rows, kv, list, out_rows, do_rows, lse + hrow, unit, drow, rows, exps, G > 1 ? 128 : H, Skv, slots, q_start + q0 + ql, sm_scale, dummy_row, smem);
      return;
    }
  }
  if constexpr (HG <= 2) {
    unsigned char* own = pds + (size_t)(ql / G) * group_pds + (size_t)(ql % G) * (K / BI) * pds_kind_bytes(HG);
    if (threadIdx.x < 256) pds_rows_body<0, HG>(q, kv, ids, out, dout, lse, own, dst, rows, q0, ql, Skv, K, q_start, sm_scale, dummy_row, smem);
    else pds_rows_body<1, HG>(q, kv, ids, out, dout, lse, own, dst, rows, q0, ql, Skv, K, q_start, sm_scale, dummy_row, smem);
  }
}

template <int HG, int G>
__global__ __launch_bounds__(DQ_THREADS, 1) void bwd_dq_reduce_kernel(
    const __bf16* __restrict__ kv, const int* __restrict__ ids, const unsigned char* __restrict__ pds,
    __bf16* __restrict__ dq, const int* __restrict__ work, size_t group_pds, int ds_once, int q0, int cnt, int H, int real, int Skv, int K, int q_start,
    const int* __restrict__ dup_flag, const unsigned char* __restrict__ rows, const unsigned char* __restrict__ exps, const int* __restrict__ start,
    float* __restrict__ dkv_acc, unsigned short* __restrict__ dkv, int n_keys, int accumulate) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const RoleSlot rs = role_slot((int)blockIdx.x, cnt, (n_keys + RED_KEYS - 1) / RED_KEYS);
  if (rs.first) {
    const Work w = work_of<G, 0>(rs.i, cnt, K, work, G > 1 && dup_flag[1]);
    const int ql = w.query;
    if (G > 1 && ql < 0) return;
    const int* list = ids + (size_t)ql * K;
    __bf16* dq_rows = dq + (size_t)(q0 + ql) * real * DQK;
    const unsigned char* own = pds + (size_t)(ql / G) * group_pds;
    if constexpr (G > 1) {
      if (w.tiles > 0) {
        dq_body<3, 4, true>(kv, list, own, dq_rows, 128, 128 / G, real, Skv, 32 * w.tiles, 0, dup_flag, ds_once, smem);
        return;
      }
      own += (size_t)(ql % G) * (K / BI) * pds_kind_bytes(HG);
    }
    dq_body<3, HG, false>(kv, list, own, dq_rows, H, H, real, Skv, K, q_start + q0 + ql, dup_flag, HG == 4 || ds_once, smem);
  } else {
    // longest work first: from the first key on where the first half of the keys has most of the rows (causal windows), else
    // from the last key (compressed keys behind a sliding window)
    const int groups = (n_keys + RED_KEYS - 1) / RED_KEYS;
    const bool forward = 2 * (long long)start[n_keys / 2] >= start[n_keys];
    const int key0 = (forward ? rs.i : groups - 1 - rs.i) * RED_KEYS;
    const bool few = start[n_keys] < RED_FEW_ROWS * (long long)n_keys;
    if (G > 1 && dup_flag[1]) {
      if (few) reduce_body<true, RED_FLIGHT_FEW>(rows, exps, start, dkv_acc, dkv, key0, n_keys, accumulate, dup_flag, smem);
      else reduce_body<true, RED_FLIGHT>(rows, exps, start, dkv_acc, dkv, key0, n_keys, accumulate, dup_flag, smem);
    } else {
      if (few) reduce_body<false, RED_FLIGHT_FEW>(rows, exps, start, dkv_acc, dkv, key0, n_keys, accumulate, dup_flag, smem);
      else reduce_body<false, RED_FLIGHT>(rows, exps, start, dkv_acc, dkv, key0, n_keys, accumulate, dup_flag, smem);
    }
  }
}

// fp32 accumulator -> bf16 dKV; NaN everywhere when a query row held a repeated id
__global__ void cast_bf16_kernel(const float* __restrict__ src, unsigned short* __restrict__ dstp, size_t n,
                                 const int* __restrict__ dup_flag) {
  const bool poison = *dup_flag != 0;
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x)
    dstp[e] = poison ? (unsigned short)0x7fc0 : f32_to_bf16_bits(src[e]);
}

// dQ of the chunks that ran before the flag was raised still holds sums: NaN everywhere in that case
__global__ void poison_bf16_kernel(unsigned short* __restrict__ p, size_t n, const int* __restrict__ dup_flag) {
  if (*dup_flag == 0) return;
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x)
    p[e] = (unsigned short)0x7fc0;
}

// ---------------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------------
// Units pay from 192 groups on, where their lists fit.  Below, too many of the 256 compute units are left without one: 150 pairs of queries
// 82 us by themselves and 85 joint, 75 groups of four 72 and 82.  Looking for them where there are none costs the difference of
// qmap_unit_kernel and qmap_kernel and the look at the keys: 6 + 5 us at 8000 queries x 256 slots of 8000 keys (whole backward 1990), 4 + 8 at
// 3000 x 2048 of 32768 (4950), -4 + 23 at 2000 x 512 of 131072 (1580).
bool use_units(int HG, int S, int Skv, int K) {
  return HG < 4 && S >= 192 * unit_queries(HG) && order::unit_lists_lds(unit_queries(HG), Skv, K) <= (size_t)150 * 1024;
}

struct BwdPlan {
  int chunk;            // queries per pass over the buffers, a multiple of G
  int G;                // queries of a group that may be a unit, or 1: from the whole call, so that a query's dQ does not depend on the chunks
  int W;                // bitmap words per key
  size_t off_bitmap, off_prefix, off_count, off_start, off_flag, off_units, off_work, off_bad, off_dst, off_sorted, off_pds, off_rows, off_exps, off_acc, total;
};

size_t align_up(size_t x) { return (x + 255) & ~(size_t)255; }

int group_queries(int S, int H, int Skv, int K) {
  const int HG = head_groups(H);
  return use_units(HG, S, Skv, K) ? unit_queries(HG) : 1;
}

// For S queries in groups of G, `chunk` of them at a time
BwdPlan layout_plan(int S, int G, int chunk, int H, int Skv, int K) {
  BwdPlan p;
  const int HG = head_groups(H);
  p.G = G;
  chunk = (chunk + G - 1) / G * G;
  p.chunk = chunk;
  p.W = (chunk + 31) / 32;
  size_t o = 0;
  p.off_bitmap = o; o = align_up(o + (size_t)Skv * p.W * 4);
  p.off_prefix = o; o = align_up(o + order::prefix_words(chunk, Skv) * 4);
  p.off_count = o; o = align_up(o + (size_t)(Skv + 1) * 4);
  p.off_start = o; o = align_up(o + (size_t)(Skv + 1) * 4);
  p.off_flag = o; o = align_up(o + 8);
  p.off_units = o; o = align_up(o + (G > 1 ? (size_t)((S + G - 1) / G) * 4 : 0));
  p.off_work = o; o = align_up(o + (G > 1 ? ((size_t)chunk + 2) * 4 : 0));
  p.off_bad = o; o = align_up(o + (size_t)((Skv + 31) / 32) * 4);
  p.off_dst = o; o = align_up(o + (size_t)chunk * K * 4);
  p.off_sorted = o; o = align_up(o + (size_t)chunk * K * 4);
  p.off_pds = o; o = align_up(o + (size_t)(chunk / G) * group_pds_bytes(HG, G, K));
  p.off_rows = o; o = align_up(o + ((size_t)chunk * K + 1) * ROW_BYTES);
  p.off_exps = o; o = align_up(o + (G > 1 ? ((size_t)chunk * K + 1) * EXP_BYTES : 0));
  p.off_acc = o; o = align_up(o + (size_t)Skv * DQK * 4);
  p.total = o;
  return p;
}

// Largest chunk of queries (all of them if possible, else repeated halving, at least 64) whose
// buffers fit the budget; without units if those of the smallest chunk do not.
BwdPlan make_plan(int S, int H, int Skv, int K, size_t budget) {
  BwdPlan p;
  for (int G = group_queries(S, H, Skv, K);; G = 1) {
    int chunk = S;
    p = layout_plan(S, G, chunk, H, Skv, K);
    while (p.total > budget && chunk > 64) {
      chunk = (chunk + 1) / 2;
      p = layout_plan(S, G, chunk, H, Skv, K);
    }
    if (p.total <= budget || G == 1) return p;
  }
}

// What a unit and a query by itself take of a compute unit (scores and rows, dQ and its share of the sums), tenths of us, and, where the units
// are up to three rounds of 256, how much more because the last round is not full: a part of what it lacks, spread over all (in more
// rounds, queries of other lengths fill it).  Fitted to whole backward passes of 800 - 8000 queries of one length x 64 - 2048 slots with
// unions of 1.0 - 3.9 lists, all joint and all by themselves (331 pairs of times): what the prices pick takes 0.2 (64 heads) and 0.1 % more
// than the better one in the mean, 6 and 9 % at most.  us, joint / by themselves, 64 heads: 1100 x 512 547 / 489 (union 24 tiles), 461 / 571 (16),
// 2077 x 512 962 / 918 (24), 801 / 1031 (16); 32 heads: 1100 x 512 533 / 392 (44), 318 / 426 (23), 3072 x 512 1073 / 1024 (44), 807 / 1076 (28),
// 8000 x 256 1770 / 1612 (26).  Near the border the two cost the same, and calls of both kinds a few per cent more.
order::UnitCost unit_cost(int HG, int S) {       // (HG 1 or 2)
  const float rounds = (float)S / (256 * unit_queries(HG)), part = rounds < 3.f ? (HG == 2 ? 0.3f : 0.4f) : 0.f;
  auto waste = [part](float n) { return n < 1.f ? 1.f / n : 1.f + part * (std::ceil(n) - n) / n; };
  const float unit = waste(rounds), apart = waste((float)S / 256);
  return {(int)((HG == 2 ? 310.f : 420.f) * unit), (int)((HG == 2 ? 70.f : 78.f) * unit), (int)((HG == 2 ? 200.f : 180.f) * apart),
          (int)((HG == 2 ? 50.f : 48.f) * apart)};
}

constexpr size_t DEFAULT_BUDGET = (size_t)160 << 30;
// What is read or written once passes by the L2, whose key rows the workgroups of an XCD share: Q (with up to 64 heads dO too: the other
// loads of the set-up take lines by parts) and, with 128 heads, dS both ways.  Up to 64 heads dS is read so up to this size (of queries by
// themselves).  Whole backward, us, dS read plain / so: 64 heads 262 MB (2000 x 1024 slots) 1451 / 1424, 367 MB (1400 x 2048, 2800 x 1024, 5600 x 512)
// 1901 / 1860, 1926 / 1896, 2081 / 2051, above the line 445 MB (1700 x 2048, 3400 x 1024, 6800 x 512) 2286 / 2255, 2230 / 2202, 2523 / 2500, 655 MB
// (2500 x 2048, 5000 x 1024, 10000 x 512) 2938 / 2914, 3041 / 3048, 3790 / 3771, 1049 MB (4000 x 2048) 5214 / 5254; 32 heads 393 MB (3000 x 2048,
// 6000 x 1024, 12000 x 512) 1147 / 1140, 2832 / 2869, 3747 / 3717, 590 MB (4500 x 2048, 9000 x 1024) 2975 / 3012, 4970 / 5020.  So the bytes alone do not
// tell: the line costs 1.3 % at one of the sizes below it and leaves up to 1.4 % of 64 heads above it.  Q and dO: 64 heads 10000 x 512
// 4021 -> 3864, 1000 x 2048 1479 -> 1473, 2077 x 512 741 -> 726, 32 heads 6000 x 1024 2902 -> 2863.  128 heads, plain / Q / dS written so / read
// so: 8192 x 2048 12 968 / 12 883 / 12 835 / 13 002 against 13 028, 400 x 2048 833 / 828 / 822 / 809, 1500 x 1024 1501 / 1490 / 1491 / 1465; units
// write dS as before (1024 x 256 x 32 heads 175 and 180).
constexpr size_t DS_ONCE_BYTES = (size_t)384 << 20;

}  // namespace

extern "C" size_t dsa_sparse_mla_bwd_workspace_bytes(int S, int H, int Skv, int K) {
  if (S <= 0 || Skv <= 0 || K <= 0) return 0;
  return make_plan(S, H, Skv, K, DEFAULT_BUDGET).total;
}

extern "C" size_t dsa_sparse_mla_bwd_workspace_bytes_min(int S, int H, int Skv, int K) {
  if (S <= 0 || Skv <= 0 || K <= 0) return 0;
  return layout_plan(S, group_queries(S, H, Skv, K), S < 64 ? S : 64, H, Skv, K).total;
}

extern "C" int dsa_sparse_mla_bwd_groups(int S, int H, int Skv, int K, size_t workspace_bytes, size_t* units_offset) {
  if (S <= 0 || Skv <= 0 || Skv > order::MAX_KEYS || H <= 0 || H > 128 || H % 32 || K <= 0 || K % 64 || K > 2048) return -1;
  const BwdPlan p = make_plan(S, H, Skv, K, workspace_bytes);
  if (p.total > workspace_bytes) return -1;
  if (units_offset) *units_offset = p.off_units;
  return p.G;
}

static int bwd_impl(const void* q, const void* kv, const void* out, const void* dout, const int32_t* ids,
                    const float* lse, int S, int H, int dq_heads, int Skv, int K, int q_start, float sm_scale, int d_v,
                    void* dq, void* dkv, void* workspace, size_t workspace_bytes, void* stream, float* pass_ms) {
  DSA_REQUIRE(d_v == DV, "dsa_sparse_mla_bwd: only d_v = 512 (d_qk = 576) is supported, got d_v = %d", d_v);
  DSA_REQUIRE(S >= 0 && Skv > 0, "dsa_sparse_mla_bwd: bad sequence sizes S=%d Skv=%d", S, Skv);
  DSA_REQUIRE(H > 0 && H <= 128 && H % 32 == 0, "dsa_sparse_mla_bwd: head count must be 32, 64, 96 or 128, got %d", H);
  DSA_REQUIRE(dq_heads > 0 && dq_heads <= H, "dsa_sparse_mla_bwd: gradients of %d heads of %d", dq_heads, H);
  DSA_REQUIRE(K > 0 && K % 64 == 0 && K <= 2048, "dsa_sparse_mla_bwd: top-k must be a multiple of 64 up to 2048, got %d", K);
  DSA_REQUIRE((size_t)Skv * DQK * 2 <= 0xffffffffull, "dsa_sparse_mla_bwd: kv larger than 4 GiB is not supported");
  DSA_REQUIRE(Skv <= order::MAX_KEYS, "dsa_sparse_mla_bwd: at most %d keys are supported, got %d", order::MAX_KEYS, Skv);
  DSA_REQUIRE(((uintptr_t)q % 16) == 0 && ((uintptr_t)kv % 16) == 0 && ((uintptr_t)out % 16) == 0 &&
              ((uintptr_t)dout % 16) == 0 && ((uintptr_t)dq % 16) == 0 && ((uintptr_t)workspace % 256) == 0,
              "dsa_sparse_mla_bwd: misaligned pointer");
  hipStream_t st = (hipStream_t)stream;
  // choose the largest chunk the given workspace allows
  BwdPlan p = make_plan(S > 0 ? S : 1, H, Skv, K, workspace_bytes);
  if (p.total > workspace_bytes || workspace == nullptr)
    DSA_FAIL(DSA_ERR_WORKSPACE, "dsa_sparse_mla_bwd: workspace of %zu bytes is too small (need at least %zu)",
             workspace_bytes, layout_plan(S, 1, S < 64 ? S : 64, H, Skv, K).total);
  unsigned char* ws = (unsigned char*)workspace;
  unsigned* bitmap = (unsigned*)(ws + p.off_bitmap);
  unsigned* prefix = (unsigned*)(ws + p.off_prefix);
  int* count = (int*)(ws + p.off_count);
  int* start = (int*)(ws + p.off_start);
  int* dup_flag = (int*)(ws + p.off_flag);     // [2]: a query has a repeated id; some queries are worked as one
  int* dstp = (int*)(ws + p.off_dst);
  int* sorted = (int*)(ws + p.off_sorted);
  unsigned char* pds = ws + p.off_pds;
  unsigned char* rows = ws + p.off_rows;
  unsigned char* exps = ws + p.off_exps;       // (units)
  float* acc = (float*)(ws + p.off_acc);
  const order::Room room{pds, p.off_exps - p.off_pds};       // (the sweep before has read them when the next order is made)

  const int HG = head_groups(H);
  // The passes are free to choose their slot order (P, dS and the dKV rows never leave the workspace): they walk each query's valid
  // ids in ascending key order, so that the queries in flight on an XCD gather neighbouring latent rows at the same time, and
  // may work several queries as one.  (The lists are put together in LDS next to a bitmap over all keys; with more keys than
  // fit there the passes walk the caller's slot order instead.)
  const bool sort_ids = order::sorted_list_fits(Skv, K);
  const int G = p.G;
  const size_t group_pds = group_pds_bytes(HG, G, K);
  int* units = (int*)(ws + p.off_units);
  int* work = (int*)(ws + p.off_work);
  unsigned* bad = (unsigned*)(ws + p.off_bad);
  const size_t reduce_lds = (size_t)RED_KEYS * RED_GROUPS * DQK * 4;
  size_t smem_dq = (size_t)3 * (TILE_BYTES + pds_kind_bytes(HG)) + ids_lds_bytes(K);
  if (smem_dq < reduce_lds) smem_dq = reduce_lds;
  if (G > 1) smem_dq = std::max(smem_dq, (size_t)3 * (TILE_BYTES + pds_kind_bytes(4)) + (size_t)unit_slots(HG, K) * 4);
  auto dq_reduce_kernel = HG == 4   ? bwd_dq_reduce_kernel<4, 1>
                          : HG == 2 ? (G > 1 ? bwd_dq_reduce_kernel<2, 2> : bwd_dq_reduce_kernel<2, 1>)
                                    : (G > 1 ? bwd_dq_reduce_kernel<1, 4> : bwd_dq_reduce_kernel<1, 1>);
  auto pds_rows_kernel = HG == 4   ? bwd_pds_rows_kernel<4, 1>
                         : HG == 2 ? (G > 1 ? bwd_pds_rows_kernel<2, 2> : bwd_pds_rows_kernel<2, 1>)
                                   : (G > 1 ? bwd_pds_rows_kernel<1, 4> : bwd_pds_rows_kernel<1, 1>);
  size_t smem_rows = HG <= 2 ? fused_lds_bytes(K) : wide_lds_bytes(K);
  if (G > 1) smem_rows = std::max(smem_rows, unit_lds_bytes(unit_slots(HG, K)));
  if (dsa_reserve_lds((const void*)pds_rows_kernel, smem_rows) != hipSuccess ||
      dsa_reserve_lds((const void*)dq_reduce_kernel, smem_dq) != hipSuccess)
    DSA_FAIL(DSA_ERR_LAUNCH, "dsa_sparse_mla_bwd: cannot reserve LDS");

  // optional timing (profiling entry point only): events between the launch groups
  hipEvent_t ev[4];
  if (pass_ms) {
    for (int i = 0; i < 3; i++) pass_ms[i] = 0.f;
    int made = 0;
    for (; made < 4; made++) if (hipEventCreate(&ev[made]) != hipSuccess) break;
    if (made < 4) {
      for (int i = 0; i < made; i++) hipEventDestroy(ev[i]);
      DSA_FAIL(DSA_ERR_LAUNCH, "dsa_sparse_mla_bwd_profile: cannot create events");
    }
  }
#define DSA_MARK(i) do { if (pass_ms) hipEventRecord(ev[i], st); } while (0)
  bool first = true;
  if (G > 1) order::kv_check_kernel<<<dim3((Skv + 31) / 32), dim3(256), 0, st>>>((const uint4*)kv, Skv, DQK * 2 / 16, bad, dup_flag);
  else order::clear_flag(dup_flag, st);
  for (int q0 = 0; q0 < S; q0 += p.chunk) {
    const int cnt = S - q0 < p.chunk ? S - q0 : p.chunk;
    DSA_MARK(0);
    if (G > 1) order::build_units(ids, q0, cnt, K, Skv, q_start, bitmap, prefix, count, start, dstp, p.W, room, st, dup_flag, sorted, G, bad, units + q0 / G, unit_slots(HG, K), unit_cost(HG, S), (uint4*)exps, work);
    else order::build(ids, q0, cnt, K, Skv, q_start, bitmap, prefix, count, start, dstp, p.W, room, st, dup_flag, sort_ids ? sorted : nullptr);
    DSA_CHECK_LAUNCH("dsa_sparse_mla_bwd(order)");
    const int* sids = sort_ids ? sorted : ids + (size_t)q0 * K;      // row ql belongs to query q0 + ql
    DSA_MARK(1);
    pds_rows_kernel<<<dim3(cnt), dim3(PDS_THREADS), smem_rows, st>>>(
        (const __bf16*)q, (const __bf16*)kv, sids, (const __bf16*)out, (const __bf16*)dout, lse, pds, dstp, rows, exps, work, dup_flag, group_pds, q0, cnt, H, Skv,
        K, q_start, sm_scale, p.chunk * K);
    DSA_CHECK_LAUNCH("dsa_sparse_mla_bwd(P, dS, dKV rows)");
    DSA_MARK(2);
    // dQ of every query beside the sums of every key.
    const int ds_once = (size_t)cnt * (K / BI) * pds_kind_bytes(HG) <= DS_ONCE_BYTES;
    dq_reduce_kernel<<<dim3(cnt + (Skv + RED_KEYS - 1) / RED_KEYS), dim3(DQ_THREADS), smem_dq, st>>>((const __bf16*)kv, sids, pds, (__bf16*)dq, work, group_pds, ds_once, q0, cnt, H, dq_heads, Skv,
                                                                   K, q_start, dup_flag, rows, exps, start, acc,
                                                                   S <= p.chunk ? (unsigned short*)dkv : nullptr, Skv, first ? 0 : 1);
    DSA_CHECK_LAUNCH("dsa_sparse_mla_bwd(dQ | dKV reduce)");
    DSA_MARK(3);
    if (pass_ms) {
      hipEventSynchronize(ev[3]);
      for (int i = 0; i < 3; i++) { float ms = 0.f; hipEventElapsedTime(&ms, ev[i], ev[i + 1]); pass_ms[i] += ms; }
    }
    first = false;
  }
  if (S == 0) {
    order::zero_u32_kernel<<<dim3(256), dim3(256), 0, st>>>((unsigned*)acc, (size_t)Skv * DQK);
  }
  if (S == 0 || S > p.chunk) cast_bf16_kernel<<<dim3(2048), dim3(256), 0, st>>>(acc, (unsigned short*)dkv, (size_t)Skv * DQK, dup_flag);
  if (S > p.chunk)      // more than one chunk: the flag may have come up after earlier chunks wrote their dQ
    poison_bf16_kernel<<<dim3(2048), dim3(256), 0, st>>>((unsigned short*)dq, (size_t)S * dq_heads * DQK, dup_flag);
  DSA_CHECK_LAUNCH("dsa_sparse_mla_bwd(cast)");
  if (pass_ms) for (int i = 0; i < 4; i++) hipEventDestroy(ev[i]);
#undef DSA_MARK
  return DSA_OK;
}

extern "C" int dsa_sparse_mla_bwd(const void* q, const void* kv, const void* out, const void* dout, const int32_t* ids,
                                  const float* lse, int S, int H, int Skv, int K, int q_start, float sm_scale, int d_v,
                                  void* dq, void* dkv, void* workspace, size_t workspace_bytes, void* stream) {
  return bwd_impl(q, kv, out, dout, ids, lse, S, H, H, Skv, K, q_start, sm_scale, d_v, dq, dkv, workspace, workspace_bytes,
                  stream, nullptr);
}

extern "C" int dsa_sparse_mla_bwd_heads(const void* q, const void* kv, const void* out, const void* dout, const int32_t* ids,
                                        const float* lse, int S, int H, int dq_heads, int Skv, int K, int q_start, float sm_scale, int d_v,
                                        void* dq, void* dkv, void* workspace, size_t workspace_bytes, void* stream) {
  return bwd_impl(q, kv, out, dout, ids, lse, S, H, dq_heads, Skv, K, q_start, sm_scale, d_v, dq, dkv, workspace, workspace_bytes,
                  stream, nullptr);
}

#ifdef DSA_BENCH_BUILD     // the benchmark library compiles this file a second time, with the timed entry point
extern "C" int dsa_sparse_mla_bwd_profile(const void* q, const void* kv, const void* out, const void* dout,
                                          const int32_t* ids, const float* lse, int S, int H, int Skv, int K, int q_start,
                                          float sm_scale, int d_v, void* dq, void* dkv, void* workspace,
                                          size_t workspace_bytes, void* stream, float* pass_ms) {
  DSA_REQUIRE(pass_ms != nullptr, "dsa_sparse_mla_bwd_profile: pass_ms must point at 3 floats");
  return bwd_impl(q, kv, out, dout, ids, lse, S, H, H, Skv, K, q_start, sm_scale, d_v, dq, dkv, workspace, workspace_bytes,
                  stream, pass_ms);
}
#endif
