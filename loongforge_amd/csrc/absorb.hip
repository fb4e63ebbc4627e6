// MLA weight absorption around the sparse attention kernels, for gfx950: per-head projections
//
//     C[s, h, n] = sum_k A[s, h, k] * W[h, n, k]            (bf16 in, fp32 accumulate, bf16 out)
//
// read and written in place inside larger tensors, so that no permute / split / concatenate copy
// surrounds them:
//   * query side   A = the no-position part of the up-projected query, [S, H, 128] inside [S, H, 192];
//                  W = W_UK^T [H, 512, 128]; C = the latent part of the attention query,
//                  [S, H, 512] inside [S, H, 576]; the rotary part of the same rows (64 elements of
//                  a row, pairs adjacent in the source) can be rotated into place by the same kernel
//   * output side  A = the attention output [S, H, 512]; W = W_UV [H, 128, 512];
//                  C = [S, H * 128], the input of the output projection
// HBM-bound at both ends: few rows read the weights (16.8 MB at 128 heads) once, many rows move their
// own 1.3 KB per (token, head).
//
// Many rows (absorb_kernel): one workgroup holds a head's 128 KB weight matrix in LDS for many row
// blocks; a wave computes C^T[n, s] = W[n, :] . A[s, :]^T for 32 rows s at a time, the weights as the
// MFMA A operand (LDS row reads), the activation rows as the B operand straight from global memory (16
// bytes per lane, next block requested before this block's MFMAs).  With C^T in the accumulators a lane
// owns one output row; four column tiles go through an 8 KB strip per wave, so that a store instruction
// writes four 256-byte row segments instead of 32 of 32 bytes.
// Few rows (absorb_few_kernel): one wave per (head, 64 columns) on the query side, two per (head, 32
// columns) on the output side read their weight rows straight into registers and walk the row blocks:
// more waves, no trip of the weights through LDS.
#include <algorithm>

#include "mla_tile.h"
#include "rope_quad.h"

namespace {

constexpr int EMB = 64;                   // rotary elements of a row

struct AbsorbArgs {
  const __bf16* a; long a_tok, a_head;
  const __bf16* w;
  __bf16* c; long c_tok, c_head;
  int S, H;
  // rotary part (pe_src == nullptr: none): same strides as a and c; position of a token: positions[s] or s / batch
  const unsigned short* pe_src; unsigned short* pe_dst;
  const void* cos; const void* sin; int cs_f32;
  const int* positions; int batch; int out_pairing;
};

__device__ __forceinline__ long position_of(const AbsorbArgs& p, int s) { return p.positions ? p.positions[s] : s / p.batch; }
__device__ __forceinline__ rope::QuadTables tables_of(const AbsorbArgs& p, long pos, int q) {
  return p.out_pairing == rope::ADJ ? rope::load_tables<rope::ADJ>(p.cos, p.sin, p.cs_f32, pos, q, EMB)
                                    : rope::load_tables<rope::SPLIT>(p.cos, p.sin, p.cs_f32, pos, q, EMB);
}
__device__ __forceinline__ void store_rotated(const AbsorbArgs& p, const rope::Quad& x, const rope::QuadTables& t, int s, int h, int q) {
  unsigned short* dst = p.pe_dst + (size_t)s * p.c_tok + (size_t)h * p.c_head;
  if (p.out_pairing == rope::ADJ) rope::store_quad<rope::ADJ>(rope::rotate<false>(x, t), dst, q, EMB);
  else rope::store_quad<rope::SPLIT>(rope::rotate<false>(x, t), dst, q, EMB);
}

// WAVES * 32 rows per step.  ROPE: the rotary part of the same rows, read one step ahead like the rows themselves.
template <int K, int N, int WAVES, bool ROPE>
__global__ __launch_bounds__(64 * WAVES, 1) void absorb_kernel(AbsorbArgs p, int splits) {
  // W[h] in LDS as K / 64 column groups of [N rows][128 bytes]; inside a group the 16-byte chunk c of row n sits in slot
  // (c & 7) ^ swz(n): the layout of the attention kernels' key tiles, whose 128-bit row reads are bank-conflict free
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  constexpr int KS = K / 16, NT = N / 32, CH = K / 8;                          // k-steps, output tiles, chunks per row
  constexpr int ROWS = 32 * WAVES;
  constexpr int ST = 16 / WAVES, SB = 64 * ST, SC = 4 * ST;                    // tiles, bytes and chunks of a strip row: 32 KB in all
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = blockIdx.x / splits, part = blockIdx.x % splits;
  unsigned char* strip = smem + (size_t)N * K * 2 + wave * (32 * SB);          // [32 rows][SB], chunks XORed with the row

  // ---- the head's weights into LDS -------------------------------------------------------
  {
    const uint4* src = (const uint4*)(p.w + (size_t)h * N * K);
#pragma unroll 8
    for (int e = tid; e < N * CH; e += 64 * WAVES) {
      const int n = e / CH, ch = e % CH;
      *(uint4*)(smem + (size_t)(ch >> 3) * (N * 128) + n * 128 + (((ch & 7) ^ mla::swz(n & 31)) << 4)) = src[e];
    }
  }
  __syncthreads();

  const int nblk = (p.S + ROWS - 1) / ROWS;
  const int b_lo = (int)((long)nblk * part / splits), b_hi = (int)((long)nblk * (part + 1) / splits);
  auto load_rows = [&](int blk, bf16x8 (&t)[KS]) {
    const int s = min(blk * ROWS + wave * 32 + r, p.S - 1);
    const bf16x8* src = (const bf16x8*)(p.a + (size_t)s * p.a_tok + (size_t)h * p.a_head) + g;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) t[ks] = src[2 * ks];
  };
  // rotary quad of (row 8 i + lane / 8 of the wave's 32, quad lane % 8)
  const int qd = lane & 7;
  auto pe_row = [&](int blk, int i) { return min(blk * ROWS + wave * 32 + 8 * i + (lane >> 3), p.S - 1); };
  auto load_pe = [&](int blk, uint4 (&t)[4]) {
#pragma unroll
    for (int i = 0; i < 4; i++)
      t[i] = *(const uint4*)(p.pe_src + (size_t)pe_row(blk, i) * p.a_tok + (size_t)h * p.a_head + 8 * qd);
  };
  bf16x8 cur[KS], nxt[KS];
  uint4 pe[4], pe_nxt[4];
  if (b_lo < b_hi) {
    load_rows(b_lo, cur);
    if (ROPE) load_pe(b_lo, pe);
  }
  for (int blk = b_lo; blk < b_hi; blk++) {
    const int s0 = blk * ROWS + wave * 32;
    if (ROPE) {                              // the tables' rows first: they are waited for with the next rows still on their way
      rope::QuadTables tb[4];
#pragma unroll
      for (int i = 0; i < 4; i++) tb[i] = tables_of(p, position_of(p, pe_row(blk, i)), qd);
      if (blk + 1 < b_hi) { load_rows(blk + 1, nxt); load_pe(blk + 1, pe_nxt); }
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (s0 + 8 * i + (lane >> 3) < p.S)
          store_rotated(p, rope::adjacent_pairs(pe[i]), tb[i], s0 + 8 * i + (lane >> 3), h, qd);
    } else if (blk + 1 < b_hi) {
      load_rows(blk + 1, nxt);
    }
#pragma unroll 1
    for (int nq = 0; nq < NT / ST; nq++) {
#pragma unroll
      for (int ni = 0; ni < ST; ni++) {
        f32x16 acc;
#pragma unroll
        for (int e = 0; e < 16; e++) acc[e] = 0.f;
        const unsigned char* wrow = smem + (32 * (ST * nq + ni) + r) * 128;
        const int sw = mla::swz(r);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
          const bf16x8 wv = *(const bf16x8*)(wrow + (ks >> 2) * (N * 128) + ((((2 * ks + g) & 7) ^ sw) << 4));
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv, cur[ks], acc, 0, 0, 0);
        }
        uint4 o[2];
        acc_row_to_16B(acc, 1.0f, o);
        *(uint4*)(strip + r * SB + (((4 * ni + g) ^ (r & (SC - 1))) << 4)) = o[0];
        *(uint4*)(strip + r * SB + (((4 * ni + 2 + g) ^ (r & (SC - 1))) << 4)) = o[1];
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < SC / 2; i++) {
        const int row = (64 / SC) * i + lane / SC, ch = lane % SC;
        const uint4 v = *(const uint4*)(strip + row * SB + ((ch ^ (row & (SC - 1))) << 4));
        if (s0 + row < p.S)
          *(uint4*)((unsigned short*)p.c + (size_t)(s0 + row) * p.c_tok + (size_t)h * p.c_head + 32 * ST * nq + 8 * ch) = v;
      }
      __builtin_amdgcn_wave_barrier();
    }
    if (blk + 1 < b_hi) {
#pragma unroll
      for (int ks = 0; ks < KS; ks++) cur[ks] = nxt[ks];
      if (ROPE) {
#pragma unroll
        for (int i = 0; i < 4; i++) pe[i] = pe_nxt[i];
      }
    }
  }
}

// The rotary part of the 32 rows of a block, by one wave.  The loads of all rows are in flight before the first is used, and no
// branch lies between them: eight rows after the other, each behind its position and a choice of table type, this wave took
// longer than those with the products (33 rows x 32 heads, cold caches, between events: 11.2 -> 7.6 us; 200 x 32 15.6 -> 12.2;
// 48 x 128 17.5 -> 15.1).
template <int PAIRING, int F32>
__device__ __forceinline__ void rotate_block(const AbsorbArgs& p, int blk, int h) {
  const int lane = threadIdx.x & 63, q = lane & 7;
  int s[4];
  long pos[4];
#pragma unroll
  for (int i = 0; i < 4; i++) s[i] = min(32 * blk + 8 * i + (lane >> 3), p.S - 1);
  if (p.positions) {
#pragma unroll
    for (int i = 0; i < 4; i++) pos[i] = p.positions[s[i]];
  } else {
#pragma unroll
    for (int i = 0; i < 4; i++) pos[i] = (unsigned)s[i] / (unsigned)p.batch;
  }
  rope::Quad x[4];
  rope::QuadTables t[4];
#pragma unroll
  for (int i = 0; i < 4; i++) x[i] = rope::load_quad<rope::ADJ>(p.pe_src + (size_t)s[i] * p.a_tok + (size_t)h * p.a_head, q, EMB);
#pragma unroll
  for (int i = 0; i < 4; i++) t[i] = rope::load_tables<PAIRING>(p.cos, p.sin, F32, pos[i], q, EMB);
#pragma unroll
  for (int i = 0; i < 4; i++)
    if (32 * blk + 8 * i + (lane >> 3) < p.S)
      rope::store_quad<PAIRING>(rope::rotate<false>(x[i], t[i]), p.pe_dst + (size_t)s[i] * p.c_tok + (size_t)h * p.c_head, q, EMB);
}

// One workgroup per (head, column tiles) and range of row blocks, plus one per head for the rotary part.  Query side: one wave
// and two 32-column tiles, so that it fills whole 128-byte lines of the output (us, one / two / four tiles: 48 rows x 128 heads
// 13.1 / 11.1 / 11.6; waves in workgroups of their own: 1 row 4.8, in pairs 5.5, in fours 7.1).  Output side (K = 512): two
// waves share a tile, half of the sum each: half the registers (the next rows are requested before these rows' products) and
// twice the waves; the halves meet in LDS, the two waves storing every other block.
template <int K> constexpr int FEW_SHARE = K == 512 ? 2 : 1;
template <int K> constexpr int FEW_COLS = K == 512 ? 1 : 2;
template <int K, int N>
__global__ __launch_bounds__(64 * FEW_SHARE<K>, 2) void absorb_few_kernel(AbsorbArgs p) {
  constexpr int SHARE = FEW_SHARE<K>, KS = K / 16 / SHARE, COLS = FEW_COLS<K>, NT = N / (32 * COLS);
  __shared__ f32x4 box[SHARE == 1 ? 1 : 2 * 4 * 64];         // [block % 2][4][lane]
  const int lane = threadIdx.x & 63, r = lane & 31, g = lane >> 5;
  const int part = SHARE == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int per = p.pe_src ? NT + 1 : NT;
  const int h = (int)blockIdx.x / per, nt = (int)blockIdx.x % per;
  const int nblk = (p.S + 31) / 32;
  const int b_lo = (int)((long)nblk * blockIdx.y / gridDim.y), b_hi = (int)((long)nblk * (blockIdx.y + 1) / gridDim.y);
  if (nt == NT) {
    for (int blk = b_lo; blk < b_hi; blk++) {
      if (p.out_pairing == rope::ADJ) {
        if (p.cs_f32) rotate_block<rope::ADJ, 1>(p, blk, h); else rotate_block<rope::ADJ, 0>(p, blk, h);
      } else {
        if (p.cs_f32) rotate_block<rope::SPLIT, 1>(p, blk, h); else rotate_block<rope::SPLIT, 0>(p, blk, h);
      }
    }
    return;
  }
  bf16x8 wv[COLS][KS], cur[KS], nxt[KS];
#pragma unroll
  for (int c = 0; c < COLS; c++) {
    const bf16x8* wp = (const bf16x8*)(p.w + ((size_t)h * N + 32 * (COLS * nt + c) + r) * K) + 2 * KS * part + g;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) wv[c][ks] = wp[2 * ks];
  }
  auto load_rows = [&](int blk, bf16x8 (&t)[KS]) {
    const bf16x8* ap = (const bf16x8*)(p.a + (size_t)min(32 * blk + r, p.S - 1) * p.a_tok + (size_t)h * p.a_head) + 2 * KS * part + g;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) t[ks] = ap[2 * ks];
  };
  load_rows(b_lo, cur);
#pragma unroll 1
  for (int blk = b_lo; blk < b_hi; blk++) {
    if (blk + 1 < b_hi) load_rows(blk + 1, nxt);
    __builtin_amdgcn_sched_barrier(0);       // all loads in flight before the first product
#pragma unroll
    for (int c = 0; c < COLS; c++) {
      f32x16 acc;
#pragma unroll
      for (int e = 0; e < 16; e++) acc[e] = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ks++) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv[c][ks], cur[ks], acc, 0, 0, 0);
      bool mine = true;
      if (SHARE == 2) {
        // one barrier per block: a box is written again two blocks on, behind the barrier that follows its reading
        f32x4* b = box + (blk & 1) * 256 + lane;
        mine = part == (blk & 1);
        if (!mine) {
#pragma unroll
          for (int j = 0; j < 4; j++) b[j * 64] = f32x4{acc[4 * j], acc[4 * j + 1], acc[4 * j + 2], acc[4 * j + 3]};
        }
        __syncthreads();
        if (mine) {
#pragma unroll
          for (int j = 0; j < 4; j++) {
            const f32x4 o = b[j * 64];
#pragma unroll
            for (int e = 0; e < 4; e++) acc[4 * j + e] += o[e];
          }
        }
      }
      if (mine) {
        uint4 o[2];
        acc_row_to_16B(acc, 1.0f, o);        // every lane takes part; rows past the end are not stored
        const int s = 32 * blk + r;
        if (s < p.S) {
          unsigned short* out = (unsigned short*)p.c + (size_t)s * p.c_tok + (size_t)h * p.c_head + 32 * (COLS * nt + c) + 8 * g;
          *(uint4*)out = o[0];
          *(uint4*)(out + 16) = o[1];
        }
      }
    }
#pragma unroll
    for (int ks = 0; ks < KS; ks++) cur[ks] = nxt[ks];
  }
}

// Up to this many (row, head) pairs the weights are better re-read by the waves than brought through LDS once per head: there the
// other kernel is one workgroup per head that mostly waits for its weights.  us, this kernel against the other, query side with
// rotary part / output side: 128 heads x 1 row 4.8 / 4.9 against 12.5 / 9.5, x 64 rows 12.5 / 10.7 against 15.8 / 11.3, x 100
// 17.0 / 14.2 against 17.1 / 12.1; 64 heads x 100 11.0 / 8.1 against 14.0 / 10.4, x 200 16.6 / 13.3 against 16.6 / 12.6;
// 32 heads x 200 10.2 / 8.6 against 15.4 / 10.9, x 300 13.1 / 11.2 against 17.1 / 11.0.
template <int K> constexpr int FEW_ROW_HEADS = K == 512 ? 8192 : 12288;
// Row ranges until there are so many workgroups.  The query side's share of the weights is read in one round trip, so every
// row block has its own waves; the output side's is not (48 rows x 128 heads 11.4 us with the weights read by both blocks'
// waves, 9.0 in one range).
template <int K> constexpr int FEW_GROUPS = K == 512 ? 512 : 1 << 16;

template <int K, int N>
int launch(const AbsorbArgs& p, hipStream_t st) {
  if ((long)p.S * p.H <= FEW_ROW_HEADS<K>) {
    const int groups = p.H * (N / (32 * FEW_COLS<K>) + (p.pe_src ? 1 : 0));
    const int ranges = std::max(1, std::min(FEW_GROUPS<K> / groups, (p.S + 31) / 32));
    absorb_few_kernel<K, N><<<dim3(groups, ranges), dim3(64 * FEW_SHARE<K>), 0, st>>>(p);
    return 0;
  }
  constexpr int WAVES = K == 128 ? 8 : 4;    // rows of 1 KB in registers twice: four waves
  const int nblk = (p.S + 32 * WAVES - 1) / (32 * WAVES);
  int splits = (256 + p.H - 1) / p.H;        // one workgroup per compute unit: its LDS holds one weight matrix
  if (splits > nblk) splits = nblk;
  const size_t smem = (size_t)K * N * 2 + 32768;
  auto kern = K == 128 && p.pe_src ? absorb_kernel<K, N, WAVES, K == 128> : absorb_kernel<K, N, WAVES, false>;
  if (dsa_reserve_lds((const void*)kern, smem) != hipSuccess) return -2;
  kern<<<dim3((unsigned)(p.H * splits)), dim3(64 * WAVES), smem, st>>>(p, splits);
  return 0;
}

int absorb(const AbsorbArgs& p, int k_dim, int n_dim, const char* who, hipStream_t st) {
  DSA_REQUIRE(p.S >= 0 && p.H > 0, "%s: bad sizes S=%d H=%d", who, p.S, p.H);
  DSA_REQUIRE((k_dim == 128 && n_dim == 512) || (k_dim == 512 && n_dim == 128),
              "%s: (k, n) must be (128, 512) (query side) or (512, 128) (output side), got (%d, %d)", who, k_dim, n_dim);
  DSA_REQUIRE(p.a_tok % 8 == 0 && p.a_head % 8 == 0 && p.c_tok % 8 == 0 && p.c_head % 8 == 0,
              "%s: row strides must be multiples of 8 elements", who);
  DSA_REQUIRE(((uintptr_t)p.a % 16) == 0 && ((uintptr_t)p.w % 16) == 0 && ((uintptr_t)p.c % 16) == 0, "%s: misaligned pointer", who);
  if (p.S == 0) return DSA_OK;
  const int rc = k_dim == 128 ? launch<128, 512>(p, st) : launch<512, 128>(p, st);
  if (rc == -2) DSA_FAIL(DSA_ERR_LAUNCH, "%s: cannot reserve LDS", who);
  DSA_CHECK_LAUNCH(who);
  return DSA_OK;
}

}  // namespace

extern "C" int dsa_mla_absorb(const void* a, int64_t a_tok, int64_t a_head, const void* w, void* c, int64_t c_tok,
                              int64_t c_head, int S, int H, int k_dim, int n_dim, void* stream) {
  const AbsorbArgs p{(const __bf16*)a, (long)a_tok, (long)a_head, (const __bf16*)w, (__bf16*)c, (long)c_tok, (long)c_head, S, H,
                     nullptr, nullptr, nullptr, nullptr, 0, nullptr, 1, 0};
  return absorb(p, k_dim, n_dim, "dsa_mla_absorb", (hipStream_t)stream);
}

extern "C" int dsa_absorb_rope_query(const void* q_up, int64_t up_tok, int64_t up_head, const void* w, void* query,
                                     int64_t q_tok, int64_t q_head, const void* cos, const void* sin, int cos_sin_f32,
                                     const int32_t* positions, int batch, int S, int H, int out_pairing, void* stream) {
  DSA_REQUIRE(q_up && query && cos && sin, "dsa_absorb_rope_query: null pointer");
  DSA_REQUIRE(positions != nullptr || batch > 0, "dsa_absorb_rope_query: batch must be positive when no positions are given");
  DSA_REQUIRE(out_pairing == 0 || out_pairing == 1, "dsa_absorb_rope_query: pairing must be 0 (adjacent) or 1 (split)");
  DSA_REQUIRE(((uintptr_t)cos % 16) == 0 && ((uintptr_t)sin % 16) == 0, "dsa_absorb_rope_query: misaligned pointer");
  const AbsorbArgs p{(const __bf16*)q_up, (long)up_tok, (long)up_head, (const __bf16*)w, (__bf16*)query, (long)q_tok, (long)q_head, S, H,
                     (const unsigned short*)q_up + 128, (unsigned short*)query + 512, cos, sin, cos_sin_f32, positions, batch, out_pairing};
  return absorb(p, 128, 512, "dsa_absorb_rope_query", (hipStream_t)stream);
}
