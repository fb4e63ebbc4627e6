// Lightning-indexer logits for gfx950: fp8-e4m3 MFMA GEMM with the ReLU, the head-weight
// reduction and the per-key scale fused into the epilogue.
//
//   logits[i, j] = k_scale[j] * sum_h q_w[i,h] * relu(q8[i,h,:] . k8[j,:])      ks[i] <= j < ke[i]
//
// One workgroup owns 8 consecutive queries, one per wave (512 threads; at 128 registers per lane
// four waves share a SIMD), and streams the keys its queries can see through LDS in tiles of 128
// rows (global_load_lds, double buffered, 16-byte slots XOR-swizzled per row).  For every 32-key
// sub-tile a wave issues, per group of 32 heads, two v_mfma_f32_32x32x64_f8f6f4 (A = the query's fp8
// rows, held in registers for the whole sweep; B = key rows from LDS).  The accumulator layout puts
// one key per lane and 16 heads per register file column, so the weighted ReLU-sum over heads is 2
// VALU ops per element inside a lane plus one exchange between the two half-waves.  Per sub-tile
// that is 4 MFMAs of 64 cycles against about 77 VALU issues of 4 cycles: the VALU port is the busier
// of the two, and the matrix pipe of one wave overlaps the epilogue of the others, not its own -
// hence the small register footprint and the high occupancy.  HBM is far from binding (q8 / k8 are
// read once, logits written once).
#include "dsa_common.h"

namespace {

constexpr int D = 128;          // indexer head dim (bytes per fp8 row)
constexpr int BK = 128;         // keys per LDS tile
constexpr int TILE_BYTES = BK * D;
constexpr int QB = 8;           // queries per workgroup

__device__ __forceinline__ int swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

__device__ __forceinline__ void dma16(unsigned lds_base, unsigned goff, const void* gbase) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :: "s"(lds_base), "v"(goff), "s"(gbase) : "memory");
}
__device__ __forceinline__ void dma4(unsigned lds_base, unsigned goff, const void* gbase) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
               :: "s"(lds_base), "v"(goff), "s"(gbase) : "memory");
}

// max(x, 0) as one instruction, on the bit pattern (a negative float is a negative integer):
// fmaxf would first quiet a possible signalling NaN with a second v_max, which doubles the cost
// of the epilogue.
__device__ __forceinline__ float relu1(float x) {
  return __builtin_bit_cast(float, max(__builtin_bit_cast(int, x), 0));
}

__global__ void fill_neg_inf_kernel(float* __restrict__ p, long rows, long ld, int width) {
  const long n = rows * (long)width;
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x)
    p[(e / width) * ld + (e % width)] = -INFINITY;
}

// sum of x over the two half-waves (lanes l and l ^ 32), in every lane.  v_permlane32_swap
// exchanges the upper half of its first operand with the lower half of its second: afterwards one
// register holds the lower-half values in both halves and the other the upper-half values.  (Written
// as inline assembly: given the same value for both operands the compiler's builtin is folded as if
// both results were equal.)
__device__ __forceinline__ float add_halves(float x) {
  float a = x, b = x;
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
  return a + b;
}

// 32 heads x 32 keys of fp8 products into the weighted ReLU-sum of a lane's key
__device__ __forceinline__ float head_sum(const i32x8 (&aq)[2], const i32x8 (&bk)[2], const float (&wq)[16], float sum) {
  f32x16 acc;
#pragma unroll
  for (int e = 0; e < 16; e++) acc[e] = 0.f;
  acc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(aq[0], bk[0], acc, 0, 0, 0, 127, 0, 127);
  acc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(aq[1], bk[1], acc, 0, 0, 0, 127, 0, 127);
#pragma unroll
  for (int e = 0; e < 16; e++) sum = fmaf(wq[e], relu1(acc[e]), sum);
  return sum;
}

// a query's fp8 rows as the A operand, and the weights of the 16 heads a lane sees per head group
template <int NHT>
__device__ __forceinline__ void load_query(const unsigned char* __restrict__ q8, const float* __restrict__ q_w, int i, int r, int g,
                                           i32x8 (&aq)[NHT][2], float (&wq)[NHT][16]) {
#pragma unroll
  for (int t = 0; t < NHT; t++) {
    const unsigned char* row = q8 + ((size_t)i * NHT * 32 + 32 * t + r) * D + 32 * g;
#pragma unroll
    for (int s = 0; s < 2; s++) {
      const i32x4 lo = *(const i32x4*)(row + 64 * s);
      const i32x4 hi = *(const i32x4*)(row + 64 * s + 16);
      aq[t][s] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    }
    const float* wrow = q_w + (size_t)i * NHT * 32 + 32 * t + 4 * g;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const f32x4 w4 = *(const f32x4*)(wrow + 8 * j);
#pragma unroll
      for (int e = 0; e < 4; e++) wq[t][4 * j + e] = w4[e];
    }
  }
}

template <int NHT, bool RELATIVE>   // groups of 32 heads; columns counted from the start of the window
__global__ __launch_bounds__(64 * QB, NHT == 1 ? 6 : 4) void indexer_logits_kernel(
    const unsigned char* __restrict__ q8, const float* __restrict__ q_w, const unsigned char* __restrict__ k8,
    const float* __restrict__ k_scale, const int* __restrict__ ks, const int* __restrict__ ke,
    int S, int Sk, int width, float* __restrict__ logits, long ld, int q_begin, int q_count, int parts) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[2 * TILE_BYTES + 2 * BK * 4];
  constexpr int NWAVE = QB;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // scalar: window tests below become scalar branches
  const int r = lane & 31, g = lane >> 5;
  const int nblk = (q_count + QB - 1) / QB;
  const int blk = nblk - 1 - (int)blockIdx.x / parts, part = (int)blockIdx.x % parts;            // longest windows first
  const int qb0 = q_begin + blk * QB;
  const int q_end = q_begin + q_count;
  // end of the window that starts at lo: no key has a column beyond the row's (absolute columns: Sk is at most the width)
  auto window_end = [&](int i, int lo) {
    const int hi = min(ke[i], Sk);
    return RELATIVE && hi - lo > width ? lo + width : hi;
  };

  // window union of the block
  int jlo = 0x7fffffff, jhi = 0, total = 0;
  for (int t = 0; t < QB; t++) {
    const int i = qb0 + t;
    if (i < q_end) {
      const int lo = max(ks[i], 0), hi = window_end(i, lo);
      jlo = min(jlo, ks[i]);
      jhi = max(jhi, hi);
      total += (max(hi - lo, 0) + 31) / 32;
    }
  }
  jlo = max(jlo, 0);

  if (2 * total < 3 * ((jhi - jlo + 31) / 32)) {
    // Unrelated windows (the sequences of a batch, or a single query): a key tile in LDS would serve one wave.  The
    // block's 32-key sub-tiles are numbered through and every wave of its workgroups takes an equal run of them,
    // whatever the lengths of the windows, with the key operand straight from global memory one sub-tile ahead.
    const int my = part * NWAVE + wave;
    const int a = (int)((long)total * my / (parts * NWAVE)), b = (int)((long)total * (my + 1) / (parts * NWAVE));
    int before = 0;
#pragma unroll 1
    for (int i = qb0; i < min(qb0 + QB, q_end); i++) {
      const int w_lo = max(ks[i], 0), w_hi = window_end(i, w_lo), n = (max(w_hi - w_lo, 0) + 31) / 32;
      const int u_lo = max(a - before, 0), u_hi = min(b - before, n);
      before += n;
      if (u_lo >= u_hi) continue;
      auto load_keys = [&](int u, i32x4 (&kk)[4], float& sc) {
        const size_t j = (size_t)min(w_lo + 32 * u + r, Sk - 1);
#pragma unroll
        for (int x = 0; x < 4; x++) kk[x] = *(const i32x4*)(k8 + j * D + 32 * g + 64 * (x >> 1) + 16 * (x & 1));
        sc = k_scale[j];
      };
      i32x4 kn[4];
      float scn;
      load_keys(u_lo, kn, scn);
      i32x8 aq[NHT][2];
      float wq[NHT][16];
      load_query(q8, q_w, i, r, g, aq, wq);
      float* lrow = logits + (size_t)(i - q_begin) * ld - (RELATIVE ? w_lo : 0);
#pragma unroll 1
      for (int u = u_lo; u < u_hi; u++) {
        i32x8 bk[2];
#pragma unroll
        for (int s = 0; s < 2; s++) bk[s] = __builtin_shufflevector(kn[2 * s], kn[2 * s + 1], 0, 1, 2, 3, 4, 5, 6, 7);
        const float ksc = scn;
        if (u + 1 < u_hi) load_keys(u + 1, kn, scn);
        float sum = 0.f;
#pragma unroll
        for (int h = 0; h < NHT; h++) sum = head_sum(aq[h], bk, wq[h], sum);
        sum = add_halves(sum) * ksc;
        const int j = w_lo + 32 * u + r;
        if (g == 0 && j < w_hi) lrow[j] = sum;
      }
    }
    return;
  }

  // this wave's query
  const int i_q = qb0 + wave;
  const bool live = i_q < q_end;
  const int qi = live ? i_q : -1;
  const int qks = live ? max(ks[i_q], 0) : 0;
  const int qke = live ? window_end(i_q, qks) : 0;
  const int wlo = live ? qks : 0x7fffffff, whi = live ? qke : 0;     // the wave's window
  i32x8 aq[NHT][2];
  float wq[NHT][16];
  load_query(q8, q_w, live ? i_q : qb0, r, g, aq, wq);
  DSA_WAIT_VMCNT(0);
#pragma unroll
  for (int t = 0; t < NHT; t++)
#pragma unroll
    for (int s = 0; s < 2; s++) asm volatile("" : "+v"(aq[t][s]));

  // this part's share of the window union's key tiles: [t_lo, t_hi)
  const int t_first = jlo / BK, t_all = max((jhi + BK - 1) / BK - t_first, 0);
  const int t_lo = t_first + (int)((long)t_all * part / parts), t_hi = t_first + (int)((long)t_all * (part + 1) / parts);
  const unsigned lds0 = (unsigned)(uintptr_t)smem;
  const int gkey = tid >> 3, gsub = tid & 7;                  // 8 NWAVE key rows per DMA instruction
  auto issue = [&](int t) {
    const unsigned lb = lds0 + (unsigned)((t & 1) * TILE_BYTES + wave * 1024);
#pragma unroll
    for (int c = 0; c < BK / (8 * NWAVE); c++) {
      const int key = c * 8 * NWAVE + gkey;
      const int row = min(t * BK + key, Sk - 1);
      dma16(lb + c * 1024 * NWAVE, (unsigned)row * D + (unsigned)((gsub ^ swz(key)) * 16), k8);
    }
    if (wave < BK / 64) {   // the tile's per-key scales
      const unsigned sb = lds0 + (unsigned)(2 * TILE_BYTES + (t & 1) * BK * 4 + wave * 256);
      dma4(sb, (unsigned)min(t * BK + wave * 64 + lane, Sk - 1) * 4u, k_scale);
    }
  };
  // B operand of sub-tile c: key row 32c + r, bytes [64s + 32g, +32) = 16-byte slots 4s+2g, 4s+2g+1
  unsigned b_off[2][2];
#pragma unroll
  for (int s = 0; s < 2; s++)
#pragma unroll
    for (int x = 0; x < 2; x++) b_off[s][x] = (unsigned)(r * D + (((4 * s + 2 * g + x) ^ swz(r)) << 4));

  if (t_lo < t_hi) issue(t_lo);
  for (int t = t_lo; t < t_hi; t++) {
    DSA_WAIT_VMCNT(0);
    __syncthreads();
    if (t + 1 < t_hi) issue(t + 1);
    const unsigned char* tb = smem + (t & 1) * TILE_BYTES;
    const float* ksc_s = (const float*)(smem + 2 * TILE_BYTES) + (t & 1) * BK;
#pragma unroll 1
    for (int c = 0; c < BK / 32; c++) {
      const int j0 = t * BK + c * 32;
      if (j0 >= whi || j0 + 32 <= wlo) continue;               // scalar: nothing of this wave's windows here
      const int j = j0 + r;
      const unsigned char* cb = tb + c * 32 * D;
      i32x8 bk[2];
#pragma unroll
      for (int s = 0; s < 2; s++) {
        const i32x4 lo = *(const i32x4*)(cb + b_off[s][0]);
        const i32x4 hi = *(const i32x4*)(cb + b_off[s][1]);
        bk[s] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      }
      const float ksc = ksc_s[c * 32 + r];
      float sum = 0.f;
#pragma unroll
      for (int tt = 0; tt < NHT; tt++) sum = head_sum(aq[tt], bk, wq[tt], sum);
      sum = add_halves(sum) * ksc;
      if (g == 0 && j >= qks && j < qke) {
        const int col = RELATIVE ? j - qks : j;
        logits[(size_t)(qi - q_begin) * ld + col] = sum;
      }
    }
  }
}

}  // namespace

// q_begin/q_count select a block of queries; row 0 of `logits` is query q_begin.
int dsa_indexer_logits_block(const void* q8, const float* q_w, const void* k8, const float* k_scale,
                             const int32_t* ks, const int32_t* ke, int S, int Hi, int Sk, float* logits,
                             int64_t ld, int width, int relative, int clean, int q_begin, int q_count,
                             hipStream_t st) {
  DSA_REQUIRE(Hi == 32 || Hi == 64, "dsa_indexer_logits: head count must be 32 or 64, got %d", Hi);
  DSA_REQUIRE(S >= 0 && Sk > 0 && width > 0 && ld >= width, "dsa_indexer_logits: bad sizes S=%d Sk=%d width=%d", S, Sk, width);
  DSA_REQUIRE((size_t)Sk * D <= 0xffffffffull, "dsa_indexer_logits: key array too large");
  DSA_REQUIRE(((uintptr_t)q8 % 16) == 0 && ((uintptr_t)k8 % 16) == 0 && ((uintptr_t)q_w % 16) == 0,
              "dsa_indexer_logits: misaligned pointer");
  DSA_REQUIRE(q_begin >= 0 && q_begin + q_count <= S, "dsa_indexer_logits: bad query block");
  if (q_count <= 0) return DSA_OK;
  if (clean) {
    fill_neg_inf_kernel<<<dim3(2048), dim3(256), 0, st>>>(logits, q_count, (long)ld, width);
    DSA_CHECK_LAUNCH("dsa_indexer_logits(fill)");
  }
  // Two workgroups of 128 registers fit a compute unit.  With too few blocks of queries to fill them their windows are
  // cut into parts, for one round of workgroups where that leaves none over (under 128 blocks) and about one and a half
  // of shorter ones beyond (us before -> after, 64 heads: one query x 4096 keys 52 -> 5, 61 x 20000 292 -> 18, 48
  // unrelated windows of 7000 keys 807 -> 15, 500 x 8000 129 -> 39, 1500 x 7500 131 -> 89, 3000 x 7500 200 -> 166).
  const int nblk = (q_count + QB - 1) / QB;
  if (!relative && width < Sk) Sk = width;                   // the keys beyond have no column
  int parts = (nblk < 128 ? 512 : 768) / nblk;
  if (parts > (Sk + BK - 1) / BK) parts = (Sk + BK - 1) / BK;
  if (parts < 1) parts = 1;
  dim3 grid(nblk * parts), block(64 * QB);
#define DSA_IDX_LAUNCH(N, R) indexer_logits_kernel<N, R><<<grid, block, 0, st>>>( \
    (const unsigned char*)q8, q_w, (const unsigned char*)k8, k_scale, ks, ke, S, Sk, width, logits, (long)ld, q_begin, q_count, parts)
  if (Hi == 32) { if (relative) DSA_IDX_LAUNCH(1, true); else DSA_IDX_LAUNCH(1, false); }
  else { if (relative) DSA_IDX_LAUNCH(2, true); else DSA_IDX_LAUNCH(2, false); }
#undef DSA_IDX_LAUNCH
  DSA_CHECK_LAUNCH("dsa_indexer_logits");
  return DSA_OK;
}

extern "C" int dsa_indexer_logits(const void* q8, const float* q_w, const void* k8, const float* k_scale,
                                  const int32_t* ks, const int32_t* ke, int S, int Hi, int Sk, float* logits,
                                  int64_t ld, int width, int relative, void* stream) {
  return dsa_indexer_logits_block(q8, q_w, k8, k_scale, ks, ke, S, Hi, Sk, logits, ld, width, relative, 1, 0, S,
                                  (hipStream_t)stream);
}
