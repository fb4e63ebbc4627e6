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
// VALU ops per element inside a lane plus one exchange between the two half-waves, which serves two
// sub-tiles at a time.
//
// Per sub-tile of 64 heads that is 4 MFMAs of 64 cycles beside some 76 VALU issues of 4: both ports are
// nearly equally busy, so a wave interleaves the products of one head group with the sums of the one
// before, half a group at a time.  Left to the waves of a SIMD to overlap each other's phases, with masked stores that
// every tile waited for and the windows read one after the other by each wave: 8192 queries x 64 heads 505 000
// cycles (MFMA busy 52 %, both ports at once 34 %) and, launched by itself again and again, 300 us; as it is now 455 000 (58 and
// 44 %) and 275, at the 1.7 GHz that the part's power leaves both then.  Inside the pass of a prompt of 8192 257 and 247,
// of 1500 behind 6692 keys 100 and 96.  us, by itself, before and after: 1500 queries behind 6692 keys 95.5
// and 90, 3000 behind 5000 161 and 151, 2077 in four documents 18.2 and 16.5, 61 behind 20 000 18.0 and 16.2,
// 48 unrelated windows of 7000 14.5 and 13.5; 32 heads, 5000 behind 500 82 and 80.5, 50 x 4 windows of 2500 8.5 and
// 7.8.  HBM is far from binding (q8 / k8 are read once, logits written once).
#include <type_traits>

#include "dsa_common.h"

namespace {

constexpr int D = 128;          // indexer head dim (bytes per fp8 row)
constexpr int BK = 128;         // keys per LDS tile
constexpr int TILE_BYTES = BK * D;
constexpr int QB = 8;           // queries per workgroup
constexpr unsigned NOWHERE = 0x40000000u;   // a store offset behind any row, also when added twice

__device__ __forceinline__ int swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

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

// Sums over the two half-waves (lanes l and l ^ 32): that of x in the lower half, that of y in the upper one.
// v_permlane32_swap exchanges the upper half of its first operand with the lower half of its second: afterwards one
// register holds the lower-half values and the other the upper-half values.  (Written as inline assembly: given the same
// value for both operands the compiler's builtin is folded as if both results were equal.)
__device__ __forceinline__ float add_pair(float x, float y) {
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(x), "+v"(y));
  return x + y;
}
__device__ __forceinline__ float add_halves(float x) { return add_pair(x, x); }

__device__ __forceinline__ f32x16 mfma_fp8(const i32x8& a, const i32x8& b, const f32x16& acc) {
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, acc, 0, 0, 0, 0, 0, 0);
}

// weighted ReLU-sum of heads [E, E + 8) of the 16 that a lane holds of a head group
template <int E>
__device__ __forceinline__ float weigh(const f32x16& acc, const float (&wq)[16], float sum) {
#pragma unroll
  for (int e = E; e < E + 8; e++) sum = fmaf(wq[e], relu1(acc[e]), sum);
  return sum;
}

// 32 heads x 32 keys of fp8 products into the weighted ReLU-sum of a lane's key
__device__ __forceinline__ float head_sum(const i32x8 (&aq)[2], const i32x8 (&bk)[2], const float (&wq)[16], float sum) {
  f32x16 acc = {};
  acc = mfma_fp8(aq[0], bk[0], acc);
  acc = mfma_fp8(aq[1], bk[1], acc);
  return weigh<8>(acc, wq, weigh<0>(acc, wq, sum));
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
  // two tiles of rows, two of scales, and so much more that the reads behind a tile's last row stay inside
  __shared__ __attribute__((aligned(1024))) unsigned char smem[2 * TILE_BYTES + 32 * D];
  constexpr int NWAVE = QB;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // scalar: window tests below become scalar branches
  const int r = lane & 31, g = lane >> 5;
  const int nblk = (q_count + QB - 1) / QB;
  const int blk = nblk - 1 - (int)blockIdx.x / parts, part = (int)blockIdx.x % parts;            // longest windows first
  const int qb0 = q_begin + blk * QB;
  const int q_end = q_begin + q_count;
  // The windows of the block's queries, one per lane, from one pair of loads: [first key, end), where no key has a column beyond
  // the row's (absolute columns: Sk is at most the width).
  const int n_q = min(QB, q_end - qb0);
  const int w_first = ks[qb0 + min(lane & (QB - 1), n_q - 1)], w_start = max(w_first, 0);
  int w_end = min(ke[qb0 + min(lane & (QB - 1), n_q - 1)], Sk);
  if (RELATIVE && w_end - w_start > width) w_end = w_start + width;
  auto start_of = [&](int t) { return __builtin_amdgcn_readlane(w_start, t); };
  auto end_of = [&](int t) { return __builtin_amdgcn_readlane(w_end, t); };

  // window union of the block
  int jlo = 0x7fffffff, jhi = 0, total = 0;
#pragma unroll
  for (int t = 0; t < QB; t++) {
    const int lo = start_of(t), hi = end_of(t);
    jlo = min(jlo, lo);
    jhi = max(jhi, hi);
    total += t < n_q ? (max(hi - lo, 0) + 31) / 32 : 0;
  }

  if (2 * total < 3 * ((jhi - jlo + 31) / 32)) {
    // Unrelated windows (the sequences of a batch, or a single query): a key tile in LDS would serve one wave.  The
    // block's 32-key sub-tiles are numbered through and every wave of its workgroups takes an equal run of them,
    // whatever the lengths of the windows, with the key operand straight from global memory one sub-tile ahead.
    const int my = part * NWAVE + wave;
    const int a = (int)((long)total * my / (parts * NWAVE)), b = (int)((long)total * (my + 1) / (parts * NWAVE));
    int before = 0;
#pragma unroll 1
    for (int i = qb0; i < qb0 + n_q; i++) {
      const int w_lo = start_of(i - qb0), w_hi = end_of(i - qb0), n = (max(w_hi - w_lo, 0) + 31) / 32;
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
  const int qks = live ? start_of(wave) : 0, qke = live ? end_of(wave) : 0;

  // this part's share of the window union, in sub-tiles of 32 keys: [s_lo, s_hi), and the wave's own of them [u_lo, u_hi)
  const int s_first = jlo / 32, s_all = max((jhi + 31) / 32 - s_first, 0);
  const int s_lo = s_first + (int)((long)s_all * part / parts), s_hi = s_first + (int)((long)s_all * (part + 1) / parts);
  const int u_lo = max(qks / 32, s_lo), u_hi = qke > qks ? min((qke + 31) / 32, s_hi) : 0;
  const int n_tiles = (s_hi - s_lo + BK / 32 - 1) / (BK / 32);
  const unsigned lds0 = (unsigned)(uintptr_t)smem;
  auto issue = [&](int t) {
    int me = tid;
    asm volatile("" : "+v"(me));                              // no registers for what one tile in four sub-tiles needs
    const int gkey = me >> 3, gsub = me & 7;                  // 8 NWAVE key rows per DMA instruction
    const int first = 32 * s_lo + t * BK;
    const unsigned lb = lds0 + (unsigned)((t & 1) * TILE_BYTES + wave * 1024);
#pragma unroll
    for (int c = 0; c < BK / (8 * NWAVE); c++) {
      const int key = c * 8 * NWAVE + gkey;
      const int row = min(first + key, Sk - 1);
      dma16(lb + c * 1024 * NWAVE, (unsigned)row * D + (unsigned)((gsub ^ swz(key)) * 16), k8);
    }
    if (wave < BK / 64) {   // the tile's per-key scales
      const unsigned sb = lds0 + (unsigned)(2 * TILE_BYTES + (t & 1) * BK * 4 + wave * 256);
      dma4(sb, (unsigned)min(first + me, Sk - 1) * 4u, k_scale);
    }
  };
  if (n_tiles > 0) issue(0);
  i32x8 aq[NHT][2];
  float wq[NHT][16];
  load_query(q8, q_w, live ? i_q : qb0, r, g, aq, wq);
  DSA_WAIT_VMCNT(0);
#pragma unroll
  for (int t = 0; t < NHT; t++)
#pragma unroll
    for (int s = 0; s < 2; s++) asm volatile("" : "+v"(aq[t][s]));

  // B operand of a sub-tile: key row r, bytes [64s + 32g, +32) = 16-byte slots 4s+2g, 4s+2g+1.  Few registers are left: what
  // an address is made of passes through empty assembly, so that it is made where it is used and not carried.
  const unsigned b_off = (unsigned)(r * D + (((2 * g) ^ swz(r)) << 4));
  struct KeyAddr { unsigned at[2][2]; };
  auto key_addr = [&](unsigned base) {
    asm volatile("" : "+s"(base));
    KeyAddr k;
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
      for (int x = 0; x < 2; x++) k.at[s][x] = (b_off ^ (unsigned)(64 * s + 16 * x)) + base;
    return k;
  };
  auto read_keys = [&](const KeyAddr& k, int s, int off) {
    const i32x4 lo = *(const i32x4*)(smem + k.at[s][0] + off);
    const i32x4 hi = *(const i32x4*)(smem + k.at[s][1] + off);
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  const unsigned lane4 = 4u * (unsigned)lane;
  auto scale_of = [&](unsigned base) {
    asm volatile("" : "+s"(base));
    return *(const float*)(smem + 2 * TILE_BYTES + (lane4 + base));
  };
  // A row's stores go through a descriptor of exactly its window, counted from its first key: keys in front of it (a huge
  // offset) and keys behind it are dropped by the bounds check, with neither compares nor masks.  Every pair of sub-tiles so
  // issues exactly one store, which is what lets the wait in front of the barrier leave them in flight.
  const __amdgpu_buffer_rsrc_t row_out = __builtin_amdgcn_make_buffer_rsrc(
      logits + (size_t)((live ? i_q : qb0) - q_begin) * ld + (RELATIVE ? 0 : qks), 0, 4 * max(qke - qks, 0), 0x00027000);
  auto store = [&](float v, unsigned at, bool lower) {         // lower: of the lower half-wave only
    asm volatile("" : "+s"(at));
    unsigned o = lane4;
    if (lower) {
      asm volatile("" : "+v"(o));
      o |= (o & 128u) << 23;
      static_assert(NOWHERE == 128u << 23, "");
    }
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), row_out, (int)(o + at), 0, 0);
  };

  // What the next sub-tile's products overlap: the second head group's products of the last one (acc1) and the first group's sum.
  f32x16 acc1 = {};
  float sum1 = 0.f;
  // the pair of sub-tiles it belongs to: the first one's sum, the scales, the place
  float sum_a = 0.f, ksc1 = 0.f;
  unsigned out1 = NOWHERE;

  bool steady = false;
  unsigned kb = 0, sb = 0;                                     // where a tile's rows and scales lie
#pragma unroll 1
  for (int t = 0; t < n_tiles; t++, kb ^= TILE_BYTES, sb ^= BK * 4) {
    if (steady) DSA_WAIT_VMCNT(BK / (32 * NHT));                      // the tile's rows, not the stores behind them
    else DSA_WAIT_VMCNT(0);
    __syncthreads();
    if (t + 1 < n_tiles) issue(t + 1);
    const int first = s_lo + t * (BK / 32);
    const int c_lo = max(u_lo - first, 0), c_hi = min(u_hi - first, BK / 32);
    steady = c_hi - c_lo == BK / 32;
    if (c_lo >= c_hi) continue;
    const unsigned ob = 128u * (unsigned)first - 4u * (unsigned)qks;
    int c = c_lo;
    const KeyAddr ka = key_addr(kb + c * 32 * D);
    i32x8 bk0 = read_keys(ka, 0, 0), bk1 = read_keys(ka, 1, 0);
    if constexpr (NHT == 2) {
      // One sub-tile: each product of 64 cycles is followed by half a head group's weighted sums, which take as long to issue, of a
      // product that ended before; a wave alone keeps both ports busy.  B: the second one of a pair.
      auto sub_tile = [&](const KeyAddr& k, auto b) {
        constexpr bool B = decltype(b)::value;
        f32x16 acc0 = {};
        acc0 = mfma_fp8(aq[0][0], bk0, acc0);
        __builtin_amdgcn_sched_barrier(0);
        sum1 = weigh<0>(acc1, wq[1], sum1);
        __builtin_amdgcn_sched_barrier(0);
        acc0 = mfma_fp8(aq[0][1], bk1, acc0);
        __builtin_amdgcn_sched_barrier(0);
        sum1 = weigh<8>(acc1, wq[1], sum1);
        if constexpr (B) sum_a = sum1;
        else store(add_pair(sum_a, sum1) * ksc1, out1, false);
        __builtin_amdgcn_sched_barrier(0);
        acc1 = f32x16{};
        acc1 = mfma_fp8(aq[1][0], bk0, acc1);
        __builtin_amdgcn_sched_barrier(0);
        bk0 = read_keys(k, 0, (B ? 2 : 1) * 32 * D);
        if constexpr (!B) ksc1 = scale_of(sb + c * 128);
        sum1 = weigh<0>(acc0, wq[0], 0.f);
        __builtin_amdgcn_sched_barrier(0);
        acc1 = mfma_fp8(aq[1][1], bk1, acc1);
        __builtin_amdgcn_sched_barrier(0);
        bk1 = read_keys(k, 1, (B ? 2 : 1) * 32 * D);
        sum1 = weigh<8>(acc0, wq[0], sum1);
        __builtin_amdgcn_sched_barrier(0);
      };
#pragma unroll 1
      for (; c < c_hi; c += 2) {
        const KeyAddr k = key_addr(kb + c * 32 * D);
        sub_tile(k, std::false_type{});
        out1 = ob + c * 128u;
        if (c + 1 < c_hi) sub_tile(k, std::true_type{});
        else {                                                 // a last one without a partner: nothing of it stays open
          sum1 = weigh<8>(acc1, wq[1], weigh<0>(acc1, wq[1], sum1));
          store(add_pair(sum1, sum1) * ksc1, out1, true);
          out1 = NOWHERE;
        }
      }
    } else {
#pragma unroll 1
      for (; c < c_hi; c++) {
        const i32x8 bk[2] = {bk0, bk1};
        const float sum = head_sum(aq[0], bk, wq[0], 0.f);
        const KeyAddr kn = key_addr(kb + min(c + 1, BK / 32 - 1) * 32 * D);
        bk0 = read_keys(kn, 0, 0);
        bk1 = read_keys(kn, 1, 0);
        store(add_halves(sum) * scale_of(sb + c * 128), ob + c * 128u, true);
      }
    }
  }
  if constexpr (NHT == 2) store(add_pair(sum_a, weigh<8>(acc1, wq[1], weigh<0>(acc1, wq[1], sum1))) * ksc1, out1, false);
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
