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
// Few rows (absorb_few_kernel): one wave per (head, 64 columns) on the query side, two or four per (head,
// 32 or 64 columns) on the output side read their weight rows straight into registers and walk the row
// blocks: more waves, no trip of the weights through LDS.
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

// Bytes of a side's rows, read and written, from which the latter are stored with the non-temporal hint (whole 128-byte lines each): 8192
// tokens x 128 heads 340 -> 326 us on the query side, 256 -> 236 on the output side.  Below, the attention behind it finds rows in the
// memory-side cache: 1500 x 128 73 -> 62 us for the kernel and 1067 -> 1075 with all that follows up to the output's projection, 900 x 128
// 706 -> 717.  A prompt with all that follows, us, neither side / both sides so stored, in MB the query side and the output side: 4000 x 64
// (393, 328) 874 / 875, 5000 x 64 (492, 410) 1041 / 1030, 2600 x 128 (511, 426) 1225 / 1230, 2800 x 128 (551, 459) 1263 / 1249, 3000 x 128 (590, 492) 1315 / 1314,
// 6000 x 64 (590, 492) 1217 / 1195, 3400 x 128 (668, 557) 1718 / 1702, 6800 x 64 (668, 557) 1382 / 1359, 8192 x 128 (1611, 1342) 2574 / 2504.  The line
// is where it began to pay with 128 heads; with 64 it would from 490 MB on, and the output side of the sizes in between stays plain.
constexpr long STREAMED_BYTES = 512l << 20;
// WAVES * 32 rows per step.  ROPE: the rotary part of the same rows, read one step ahead like the rows themselves.
template <int K, int N, int WAVES, bool ROPE, bool STREAMED>
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
        if (s0 + row < p.S) {
          i32x4* dst = (i32x4*)((unsigned short*)p.c + (size_t)(s0 + row) * p.c_tok + (size_t)h * p.c_head + 32 * ST * nq + 8 * ch);
          if constexpr (STREAMED) __builtin_nontemporal_store(__builtin_bit_cast(i32x4, v), dst);
          else *dst = __builtin_bit_cast(i32x4, v);
        }
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

// One workgroup per (head, COLS * 32 columns) and range of row blocks, plus one per head for the rotary part.  SHARE waves share the
// sum over k (K = 512), each a part of it: fewer registers (the next rows are requested before these rows' products) and more
// waves; the parts meet in LDS, every wave adding up and storing its share of the block.
// 16x16x32 products: four lanes read 64 consecutive bytes of a row, and with the weight rows of a tile in the order 8 kg + i,
// 8 kg + 4 + i a lane owns eight consecutive columns of two tiles and four lanes store 64 consecutive bytes (32x32x16: 32 bytes
// either way).  The workgroups of a head sit on one XCD (where the heads divide evenly), so that its L2 fetches the head's rows and
// weights once.  Bound by what the caches deliver and by the round trips of a launch.  us, 32x32x16 products of two tiles and heads
// over all XCDs before / now, cold caches, query side: 48 rows x 128 heads 10.5 / 9.2, 200 x 32 9.5 / 8.5, 61 x 64 7.0 / 6.7, 90 x 128
// 16.0 / 13.2; output side: 48 x 128 9.8 / 8.6, 200 x 32 8.9 / 8.3, 61 x 64 7.0 / 6.3, 120 x 64 9.7 / 8.5.
template <int K, int N, int SHARE, int COLS>
__global__ __launch_bounds__(64 * SHARE, 2) void absorb_few_kernel(AbsorbArgs p) {
  constexpr int KS = K / 32 / SHARE, NT = N / (32 * COLS), MINE = 2 * COLS / SHARE;        // k-steps; column groups; a wave's units of
  static_assert(SHARE == 1 || MINE == 1);                                                   // (16 rows, 32 columns) to store: all, or one
  __shared__ f32x4 box[SHARE == 1 ? 1 : 2 * SHARE * (SHARE - 1) * 2 * 64];                  // [block % 2][unit][other waves][2][lane]
  const int lane = threadIdx.x & 63, m = lane & 15, kg = lane >> 4;
  const int part = SHARE == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int per = p.pe_src ? NT + 1 : NT, bx = (int)blockIdx.x;
  const bool xcd = p.H % 8 == 0;
  const int h = xcd ? 8 * ((bx >> 3) / per) + (bx & 7) : bx / per, nt = (xcd ? bx >> 3 : bx) % per;
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
  bf16x8 wv[2 * COLS][KS], cur[2][KS], nxt[2][KS];
#pragma unroll
  for (int c = 0; c < 2 * COLS; c++) {
    const int n = 32 * (COLS * nt + (c >> 1)) + 8 * (m >> 2) + 4 * (c & 1) + (m & 3);
    const bf16x8* wp = (const bf16x8*)(p.w + ((size_t)h * N + n) * K) + 4 * KS * part + kg;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) wv[c][ks] = wp[4 * ks];
  }
  auto load_rows = [&](int blk, bf16x8 (&t)[2][KS]) {
#pragma unroll
    for (int rt = 0; rt < 2; rt++) {
      const bf16x8* ap = (const bf16x8*)(p.a + (size_t)min(32 * blk + 16 * rt + m, p.S - 1) * p.a_tok + (size_t)h * p.a_head) + 4 * KS * part + kg;
#pragma unroll
      for (int ks = 0; ks < KS; ks++) t[rt][ks] = ap[4 * ks];
    }
  };
  load_rows(b_lo, cur);
#pragma unroll 1
  for (int blk = b_lo; blk < b_hi; blk++) {
    if (blk + 1 < b_hi) load_rows(blk + 1, nxt);
    __builtin_amdgcn_sched_barrier(0);       // all loads in flight before the first product
    f32x4 acc[2][2 * COLS];
#pragma unroll
    for (int rt = 0; rt < 2; rt++)
#pragma unroll
      for (int c = 0; c < 2 * COLS; c++) acc[rt][c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
#pragma unroll
      for (int c = 0; c < 2 * COLS; c++)
#pragma unroll
        for (int rt = 0; rt < 2; rt++) acc[rt][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[c][ks], cur[rt][ks], acc[rt][c], 0, 0, 0);
    if (SHARE > 1) {
      // one barrier per block: a box is written again two blocks on, behind the barrier that follows its reading
      f32x4* b = box + (blk & 1) * (SHARE * (SHARE - 1) * 2 * 64) + lane;
#pragma unroll
      for (int u = 0; u < SHARE; u++)
        if (u != part) {
#pragma unroll
          for (int x = 0; x < 2; x++) b[((u * (SHARE - 1) + (part < u ? part : part - 1)) * 2 + x) * 64] = acc[u / COLS][2 * (u % COLS) + x];
        }
      __syncthreads();
#pragma unroll
      for (int u = 0; u < SHARE; u++)
        if (u == part) {
#pragma unroll
          for (int o = 0; o < SHARE - 1; o++)
#pragma unroll
            for (int x = 0; x < 2; x++) acc[u / COLS][2 * (u % COLS) + x] += b[((u * (SHARE - 1) + o) * 2 + x) * 64];
        }
    }
#pragma unroll
    for (int u = 0; u < 2 * COLS; u++) {
      if (SHARE > 1 && u != part) continue;
      const int rt = u / COLS, c = 2 * (u % COLS), s = 32 * blk + 16 * rt + m;
      const f32x4 lo = acc[rt][c], hi = acc[rt][c + 1];
      if (s < p.S)
        *(uint4*)((unsigned short*)p.c + (size_t)s * p.c_tok + (size_t)h * p.c_head + 32 * COLS * nt + 16 * c + 8 * kg) =
            make_uint4(cvt_pk_bf16(lo[0], lo[1]), cvt_pk_bf16(lo[2], lo[3]), cvt_pk_bf16(hi[0], hi[1]), cvt_pk_bf16(hi[2], hi[3]));
    }
#pragma unroll
    for (int rt = 0; rt < 2; rt++)
#pragma unroll
      for (int ks = 0; ks < KS; ks++) cur[rt][ks] = nxt[rt][ks];
  }
}

// Row ranges: `full` workgroups, or twice as many with more than three row blocks for every two of them; more read the weights too often.
// us, output side with 256 / 512 workgroups: 200 rows x 32 heads 7.6 / 8.6, 48 x 128 8.2 / 9.0, 400 x 32 11.1 / 10.8; query side with up to
// 1200 / 2400: 200 x 32 8.5 / 9.2, 250 x 64 15.9 / 15.2.
template <int K, int N, int SHARE, int COLS>
void launch_few(const AbsorbArgs& p, int full, hipStream_t st) {
  const int groups = p.H * (N / (32 * COLS) + (p.pe_src ? 1 : 0)), nblk = (p.S + 31) / 32, many = 2 * full / groups;
  const int ranges = 2 * nblk > 3 * many ? many : std::min(full / groups, nblk);
  absorb_few_kernel<K, N, SHARE, COLS><<<dim3(groups, std::max(1, ranges)), dim3(64 * SHARE), 0, st>>>(p);
}

// Up to `few` (row, head) pairs the weights are better re-read by the waves than brought through LDS once per head: there the other
// kernel is one workgroup per head that mostly waits for its weights.  us, cold caches, this kernel against the other, query side with
// rotary part / output side: 128 heads x 1 row 5.7 / 5.7 against 14.3 / 11.1, x 100 14.2 / 11.6 against 17.9 / 13.3, x 160 18.7 / 14.4
// against 20.7 / 16.2, x 200 22.3 / 16.9 against 21.3 / 16.4; 64 heads x 250 15.1 / 11.5 against 20.8 / 13.0, x 400 21.0 / 16.4 against
// 20.8 / 16.4; 32 heads x 640 17.8 / 14.9 against 20.6 / 14.1.  The other kernel's workgroups walk whole steps: two of them
// are worse than half as many row blocks here (output side, 128 heads x 300 20.6 against 25.5, 32 heads x 1400 21.7 against 26.1).
// Output side: four waves and 64 columns a workgroup where those fill the chip (61 rows x 64 heads 6.0 and 6.8 as two waves and 32
// columns), two and 32 where they do not (16 x 64 5.5 and 4.7, 33 x 32 6.0 and 4.8).
template <int K, int N>
int launch(const AbsorbArgs& p, hipStream_t st) {
  constexpr int WAVES = K == 128 ? 8 : 4;    // rows of 1 KB in registers twice: four waves
  const int nblk = (p.S + 32 * WAVES - 1) / (32 * WAVES);
  const int splits = std::min((256 + p.H - 1) / p.H, nblk);        // one workgroup per compute unit: its LDS holds one weight matrix
  const long few = K == 128 ? 22528 : nblk <= splits ? 18432 : 49152;
  if ((long)p.S * p.H <= few) {
    if constexpr (K == 128) launch_few<K, N, 1, 2>(p, 1200, st);
    else if (p.H * (N / 64) * ((p.S + 31) / 32) >= 240) launch_few<K, N, 4, 2>(p, 256, st);
    else launch_few<K, N, 2, 1>(p, 512, st);
    return 0;
  }
  const size_t smem = (size_t)K * N * 2 + 32768;
  const bool rope = K == 128 && p.pe_src, streamed = (long)p.S * p.H * 2 * (K + N + (rope ? 2 * EMB : 0)) > STREAMED_BYTES;
  auto kern = rope ? (streamed ? absorb_kernel<K, N, WAVES, K == 128, true> : absorb_kernel<K, N, WAVES, K == 128, false>)
                   : (streamed ? absorb_kernel<K, N, WAVES, false, true> : absorb_kernel<K, N, WAVES, false, false>);
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
