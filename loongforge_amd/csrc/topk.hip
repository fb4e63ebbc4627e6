// Per-row top-k selection (radix select with the candidate histograms in LDS) for gfx950.
//
// One workgroup per row.  General path: the row's window is read once into LDS as order-preserving
// 32-bit keys (or re-read from global memory when it does not fit); three histogram passes
// (12 + 10 + 10 bits, most significant first) locate the k-th largest key exactly, a prefix-sum
// compaction then emits every key above it plus the first ties in ascending column order, so the
// result is deterministic; an optional sorting network orders the K outputs by descending score.
// Sorted rows whose values spread over a range take a single sweep instead (linear_select_sort*):
// a histogram over equal-width value bins, a counting-sort scatter and a rank inside each bin; rows
// of up to 8192 columns are held in registers for it, which leaves room for four workgroups per
// compute unit.  HBM-bound by design (4 bytes read per candidate, 8 bytes written per output slot);
// in practice the LDS atomics of the histogram and the scatter set the pace.
#include <type_traits>

#include "dsa_common.h"

namespace {

constexpr int HBINS = 4096;
// Every routine takes the workgroup size BL (256, or 1024 for few or long rows).  `scratch` holds three ints per wave for
// reductions and four more for what they find.
template <int BL> constexpr int NWAVES = BL / 64;
template <int BL> constexpr int SCRATCH = 3 * (BL / 64) + 4;

__device__ __forceinline__ unsigned f2key(float f) {       // larger float <-> larger unsigned
  unsigned u = __builtin_bit_cast(unsigned, f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float key2f(unsigned k) {
  unsigned u = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
  return __builtin_bit_cast(float, u);
}

// Reductions and scans over a wave whose lanes are all active, by moves inside its rows of 16 lanes and from row to row: a shuffle
// is a trip through LDS, and rows are bound by the chain of such trips and barriers (one row of 4096, top-k 2048:
// 7.2 -> 6.0 us with both cut; 200 of 2500 7.0 -> 6.0, 8192 of 2048 58.6 -> 52.7, 8192 of 8192 137 -> 130).
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_add(int x) { return x + __builtin_amdgcn_update_dpp(0, x, CTRL, ROWS, 0xf, false); }
__device__ __forceinline__ int wave_inclusive_sum(int x) {
  x = dpp_add<0x111, 0xf>(x);                // row_shr:1, 2, 4, 8
  x = dpp_add<0x112, 0xf>(x);
  x = dpp_add<0x114, 0xf>(x);
  x = dpp_add<0x118, 0xf>(x);
  x = dpp_add<0x142, 0xa>(x);                // the last lane of rows 0 and 2 to the row behind
  return dpp_add<0x143, 0xc>(x);             // lane 31 to the upper half
}
template <class F>
__device__ __forceinline__ float wave_fold(float x, F f) {   // f commutative; the result in every lane
#pragma unroll
  for (int m = 1; m < 16; m <<= 1) x = f(x, xor16(x, m));
  auto lane = [&](int l) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), l)); };
  return f(f(lane(0), lane(16)), f(lane(32), lane(48)));
}

// exclusive prefix sum over the block (thread order), also returns the block total.  FRESH: there is a barrier behind the last use of scratch.
template <int BL, bool FRESH>
__device__ __forceinline__ int block_exscan(int v, int* scratch, int& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int inc = wave_inclusive_sum(v);
  if (!FRESH) __syncthreads();
  if (lane == 63) scratch[wave] = inc;
  __syncthreads();
  int base = 0, tot = 0;
#pragma unroll
  for (int w = 0; w < NWAVES<BL>; w++) { int s = scratch[w]; if (w < wave) base += s; tot += s; }
  total = tot;
  return base + inc - v;
}

// minimum, maximum and sum over the waves' entries (mn at 0, mx at NWAVES, count at 2 NWAVES)
template <int BL>
__device__ __forceinline__ void row_range(const int* scratch, float& mn, float& mx, int& count) {
  const float* f = (const float*)scratch;
  mn = f[0]; mx = f[NWAVES<BL>]; count = scratch[2 * NWAVES<BL>];
#pragma unroll
  for (int w = 1; w < NWAVES<BL>; w++) {
    mn = fminf(mn, f[w]);
    mx = fmaxf(mx, f[NWAVES<BL> + w]);
    count += scratch[2 * NWAVES<BL> + w];
  }
}

struct Pick { int bin; int above; };

// Finds, scanning bins from the highest down, the bin in which the running count reaches `need`.
// hist has nb bins (nb % BL == 0).  Result: that bin and the number of keys in higher bins.
template <int BL>
__device__ __forceinline__ Pick pick_bin(const int* hist, int nb, int need, int* scratch, int* res) {
  const int per = nb / BL;
  const int hi = nb - 1 - (int)threadIdx.x * per;          // this thread owns bins hi, hi-1, ..., hi-per+1
  int local = 0;
  for (int b = 0; b < per; b++) local += hist[hi - b];
  int total;
  int before = block_exscan<BL, true>(local, scratch, total);
  if (before < need && before + local >= need) {
    int run = before;
    for (int b = 0; b < per; b++) {
      int c = hist[hi - b];
      if (run + c >= need) { res[0] = hi - b; res[1] = run; break; }
      run += c;
    }
  }
  __syncthreads();
  Pick p = {res[0], res[1]};
  __syncthreads();
  return p;
}

// Order of the sorted output: descending score, ascending id among equal scores (id -1 last).
__device__ __forceinline__ bool comes_first(float a, int ia, float b, int ib) {
  return (a > b) || (a == b && (unsigned)ia < (unsigned)ib);
}

// Bitonic sort of Kp2 = EPT * BL (score, id) pairs held in LDS.  A pair becomes one 64-bit
// key whose unsigned order is the output order (descending score, then ascending id, id -1 last),
// so a compare-exchange is one 64-bit compare and two selects.  Thread t keeps
// elements [t*EPT, (t+1)*EPT) in registers: strides below EPT are register compare-exchanges,
// strides inside a wave's span exchange through LDS without a workgroup barrier (LDS operations
// of one wave complete in order), and only the strides that cross waves need barriers.  The
// exchange buffer holds element j of thread t at j * BL + t, so every LDS access of a wave is
// bank-conflict free; the sorted elements go straight from registers to global memory.
__device__ __forceinline__ unsigned long long sort_key(float score, int id) {
  const unsigned bits = __builtin_bit_cast(unsigned, score + 0.0f);          // -0 -> +0
  const unsigned asc = bits ^ ((bits >> 31) ? 0xffffffffu : 0x80000000u);    // ascending with the score
  return ((unsigned long long)(~asc) << 32) | (unsigned)id;
}
__device__ __forceinline__ float sort_key_score(unsigned long long key) {
  const unsigned asc = ~(unsigned)(key >> 32);
  return __builtin_bit_cast(float, asc ^ ((asc >> 31) ? 0x80000000u : 0xffffffffu));
}

template <int BL, int EPT>
__device__ __forceinline__ void bitonic_regs(float* outv, int* outi, unsigned long long* xbuf, int Kp2, float* sv, int* si, int K) {
  const int tid = threadIdx.x;
  const int base = tid * EPT;
  unsigned long long key[EPT];
#pragma unroll
  for (int j = 0; j < EPT; j++) key[j] = sort_key(outv[base + j], outi[base + j]);
  __syncthreads();                             // the buffer is reused as the exchange buffer below
  for (int size = 2; size <= Kp2; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      if (stride >= EPT) {
        const int pt = tid ^ (stride / EPT);
        const bool cross_wave = stride / EPT >= 64;
#pragma unroll
        for (int j = 0; j < EPT; j++) xbuf[j * BL + tid] = key[j];
        if (cross_wave) __syncthreads(); else __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        unsigned long long pk[EPT];
#pragma unroll
        for (int j = 0; j < EPT; j++) pk[j] = xbuf[j * BL + pt];
        if (cross_wave) __syncthreads(); else __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        // this lane keeps the smaller key when it holds the lower element of an ascending pair or
        // the upper element of a descending one (size > stride >= EPT: the same for all j)
        const bool keep_small = ((base & stride) == 0) == ((base & size) == 0);
#pragma unroll
        for (int j = 0; j < EPT; j++) key[j] = ((key[j] < pk[j]) == keep_small) ? key[j] : pk[j];
      } else {
#pragma unroll
        for (int st = EPT >> 1; st > 0; st >>= 1) {
          if (st != stride) continue;
#pragma unroll
          for (int j = 0; j < EPT; j++) {
            if (j & st) continue;
            const bool asc = ((base + j) & size) == 0;
            const unsigned long long x = key[j], y = key[j | st];
            const bool x_first = (x < y) == asc;
            key[j] = x_first ? x : y;
            key[j | st] = x_first ? y : x;
          }
        }
      }
    }
  }
#pragma unroll
  for (int j = 0; j < EPT; j++)
    if (base + j < K) { sv[base + j] = sort_key_score(key[j]); si[base + j] = (int)(unsigned)key[j]; }
}

// Sorted top-K of a staged row in one sweep, for rows whose finite values spread over a range:
// a histogram over HBINS equal-width value bins (bin 0 = largest values) finds the bin that holds
// the K-th largest value; every element of a better bin, plus all elements of that bin, is
// scattered into its bin's segment of an LDS buffer (a counting sort, segments in descending value
// order), and each scattered element then finds its final position by counting the elements of its
// own segment that precede it in the output order (descending score, ascending column).  Elements
// of the threshold bin that rank beyond the K-th place are dropped.  The result is exact and does
// not depend on the order in which the atomics land.  Returns false without writing anything when
// the row is unsuitable (no spread, or a crowded bin): the caller then takes the general path.
constexpr int LIN_SPARE = 960;               // extra buffer entries for the threshold bin's surplus
constexpr int LIN_PAD = 4;                   // and behind the last element: what the ranking reads at a time
constexpr int REG_ROW = 8192 + 4 * 256;      // longest row (plus alignment slack) the register variant holds
constexpr int REG_ROW_BIG = 32768 + 4 * 256; // the same for the variant with twice the registers
constexpr int REG_ROW_WIDE = 9 * 4 * 1024;   // the same for the 1024-thread variant
constexpr int WIDE_ROWS = 256;               // at most so many rows: the 1024-thread kernel
constexpr int COMPACT_FLIGHT = 8;            // loads in flight per thread of the general path's compaction
constexpr int LIN_MAX_BIN = 256;             // largest segment ranked by pairwise counting

// Threshold bin of a filled histogram (thread t owns bins [PER t, PER t + PER)), then the segment
// starts written over the counts.  False when a bin is too crowded for the ranking step.
template <int BL>
__device__ __forceinline__ bool lin_threshold(int* hist, int* scratch, int keff, int& tbin, int& above, int& c) {
  const int tid = threadIdx.x;
  constexpr int PER = HBINS / BL;
  static_assert(PER % 4 == 0, "a thread's bins go by 16 bytes");
  int* found = scratch + 3 * NWAVES<BL>;
  int cnt[PER], local = 0;
#pragma unroll
  for (int b4 = 0; b4 < PER; b4 += 4) {
    const int4 q4 = *(const int4*)(hist + tid * PER + b4);
    cnt[b4] = q4.x; cnt[b4 + 1] = q4.y; cnt[b4 + 2] = q4.z; cnt[b4 + 3] = q4.w;
  }
#pragma unroll
  for (int b = 0; b < PER; b++) local += cnt[b];
  int total;
  const int before = block_exscan<BL, true>(local, scratch, total);
  if (before < keff && before + local >= keff) {
    int run = before;
#pragma unroll
    for (int b = 0; b < PER; b++) {
      if (run < keff && run + cnt[b] >= keff) { found[0] = tid * PER + b; found[1] = run; found[2] = cnt[b]; }
      run += cnt[b];
    }
  }
  if (tid == 0) found[3] = 0;                // set below by a thread with a crowded bin in front of the threshold's
  __syncthreads();
  tbin = found[0]; above = found[1]; c = found[2];
  int big = 0;
#pragma unroll
  for (int b = 0; b < PER; b++) if (tid * PER + b < tbin) big = max(big, cnt[b]);
  if (big > LIN_MAX_BIN) found[3] = 1;
  {
    int run = before, st[PER];
#pragma unroll
    for (int b = 0; b < PER; b++) { st[b] = run; run += cnt[b]; }
#pragma unroll
    for (int b4 = 0; b4 < PER; b4 += 4) *(int4*)(hist + tid * PER + b4) = make_int4(st[b4], st[b4 + 1], st[b4 + 2], st[b4 + 3]);
  }
  __syncthreads();
  return !found[3] && c <= LIN_SPARE;
}

// Final position of every scattered element: hist[b] is the end of segment b by now.  The elements of later segments come behind it
// and so do the LIN_PAD entries behind the last one, so that counting may run past the end of its segment: four entries at a time for
// two elements of a thread together (of 1024, one where few have a second), as often as the longest segment of the wave asks for.
// (One entry at a time in a loop of every lane's own length is a chain of LDS trips.  us, then / now: top-k 2048, 8192 causal rows 103 / 97,
// 1500 rows of 7500 33.2 / 30.4, 8192 of 2048 83 / 77; top-k 512, 4000 rows of 1000 28.9 / 27.2, 2077 of up to 692 15.6 / 14.9; 200 rows of
// 1000, top-k 256, with all but one in a segment 51 / 35, 62 in pairs.  Fewer bins for short rows, which a row's clearing and scanning of 4096 is a
// quarter of, were 22 at 4000 x 1000, but 106 and not 37 where half of the values are close to zero, and 63 and not 41 with an outlier.)
template <int BL, class BinOf>
__device__ __forceinline__ void lin_rank(const unsigned long long* obuf, const int* hist, int filled, int keff, int K,
                                         int base_id, BinOf bin_of, float* sv, int* si) {
  const int tid = threadIdx.x;
  auto rank_at = [&](int p0, auto pair) {
    constexpr int PAIR = decltype(pair)::value;
    unsigned long long key[PAIR];
    float v[PAIR];
    int start[PAIR], rank[PAIR], longest = 0;
#pragma unroll
    for (int u = 0; u < PAIR; u++) key[u] = obuf[min(p0 + u * BL, filled)];
#pragma unroll
    for (int u = 0; u < PAIR; u++) {
      v[u] = sort_key_score(key[u]);
      const bool in = p0 + u * BL < filled;
      const int b = in ? bin_of(v[u]) : 0;
      start[u] = in ? (b > 0 ? hist[b - 1] : 0) : filled;
      longest = max(longest, (in ? hist[b] : filled) - start[u]);
      rank[u] = 0;
    }
    for (int j = 0; __any(j < longest); j += LIN_PAD) {
#pragma unroll
      for (int u = 0; u < PAIR; u++) {
        const unsigned long long* o = obuf + min(start[u] + j, filled);
#pragma unroll
        for (int i = 0; i < LIN_PAD; i++) rank[u] += o[i] < key[u];
      }
    }
#pragma unroll
    for (int u = 0; u < PAIR; u++) {
      const int pos = start[u] + rank[u];
      if (pos < keff && p0 + u * BL < filled) { sv[pos] = v[u]; si[pos] = base_id + (int)(unsigned)key[u]; }
    }
  };
  const std::integral_constant<int, 1> one;
  const std::integral_constant<int, 2> two;
  if (BL == 1024 && filled <= BL + BL / 2) {
    for (int p = tid; p < filled; p += BL) rank_at(p, one);
  } else {
    for (int p = tid; p < filled; p += 2 * BL) rank_at(p, two);
  }
  for (int t = keff + tid; t < K; t += BL) { sv[t] = -INFINITY; si[t] = -1; }
}
// The entries behind the last scattered one: behind everything.
__device__ __forceinline__ void lin_pad(unsigned long long* obuf, int filled) {
  if (threadIdx.x < LIN_PAD) obuf[filled + threadIdx.x] = ~0ull;
}

// The same for rows of at most 4 NV BL elements, with the row held in registers instead of
// LDS: thread t owns the 16-byte chunks t, t + BL, ... of the row counted from the 16-byte
// boundary at or below its first element, so the whole row is fetched by NV vector loads issued
// together and the workgroup needs only the histogram and the output buffer in LDS.  The row is
// positions [off, m) of that layout; chunk i (positions [4 BL i, 4 BL (i + 1))) is touched only
// while it holds any of them.
template <int BL, int NV>
__device__ __forceinline__ void load_row_regs(const float* __restrict__ src, int n, float (&v)[NV][4], int& off, int& m) {
  const int tid = threadIdx.x;
  off = (int)(((uintptr_t)src >> 2) & 3);                  // elements between that boundary and src
  const float* base = src - off;
  m = n + off;
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const int p = 4 * (tid + BL * i);
    if (p >= off && p + 4 <= m) {
      const float4 x = *(const float4*)(base + p);
      v[i][0] = x.x; v[i][1] = x.y; v[i][2] = x.z; v[i][3] = x.w;
    } else {
#pragma unroll
      for (int j = 0; j < 4; j++) v[i][j] = (p + j >= off && p + j < m) ? base[p + j] : -INFINITY;
    }
  }
}

// Rows of at most SHORT_ROW elements: one element per thread, ranked by counting the elements that precede it.  (The
// first rows of a causal window: a row of one element has no spread, and the sorting network of the general path
// would take 50 us over its 2048 output slots.)  False for rows that hold a NaN or +inf.
constexpr int SHORT_ROW = 256;
template <int BL>
__device__ __forceinline__ bool rank_short_row(const float* __restrict__ src, int n, int K, int base_id, unsigned long long* buf,
                                               float* sv, int* si) {
  const int tid = threadIdx.x;
  const float v = tid < n ? src[tid] : -INFINITY;
  const bool live = v > -INFINITY;
  const unsigned long long key = live ? sort_key(v, tid) : ~0ull;
  if (tid < SHORT_ROW) buf[tid] = key;
  if (__syncthreads_or(!(v < INFINITY))) return false;
  const int nfin = __syncthreads_count(live);
  if (tid < SHORT_ROW) {
    int rank = 0;
#pragma unroll 8
    for (int j = 0; j < n; j++) rank += buf[j] < key;
    if (live && rank < K) { sv[rank] = v; si[rank] = base_id + tid; }
  }
  for (int t = min(K, nfin) + tid; t < K; t += BL) { sv[t] = -INFINITY; si[t] = -1; }
  return true;
}

// min / max of three without the canonicalising v_max that fminf / fmaxf put in front of every operand
__device__ __forceinline__ float min3_raw(float a, float b, float c) {
  float r;
  asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ float max3_raw(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// The selection itself for rows whose values are all finite - the common case.  No per-element
// finiteness tests (an infinity shows in the row's minimum or maximum, a NaN in one unordered compare
// per two elements), min / max three at a time, bins without a clamp ((mx - x) scale < HBINS for every
// x in [mn, mx]), and chunks wholly inside the row need no position tests.  Returns 1 when the row is
// done, 0 when it is unsuitable (no spread, a crowded bin), -1 when it holds a non-finite value (the
// caller then runs the tolerant form below on the same registers).
template <int BL, int NV>
__device__ __forceinline__ int select_regs_finite(const float (&v)[NV][4], int off, int m, int K, int base_id, int* hist,
                                                  int* scratch, unsigned long long* obuf, float* sv, int* si) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  constexpr int CH = 4 * BL;
  const int nch = (m + CH - 1) / CH;                        // chunks that hold any of the row
  auto chunk_full = [&](int i) { return (i > 0 || off == 0) && CH * (i + 1) <= m; };   // the same for all threads
  for (int b = tid; b < HBINS / 4; b += BL) ((int4*)hist)[b] = make_int4(0, 0, 0, 0);
  float mn = INFINITY, mx = -INFINITY;
  bool nan = false;
#pragma unroll
  for (int i = 0; i < NV; i++) {
    if (i >= nch) continue;
    if (chunk_full(i)) {
      mn = min3_raw(mn, v[i][0], v[i][1]); mn = min3_raw(mn, v[i][2], v[i][3]);
      mx = max3_raw(mx, v[i][0], v[i][1]); mx = max3_raw(mx, v[i][2], v[i][3]);
      nan |= __builtin_isunordered(v[i][0], v[i][1]) | __builtin_isunordered(v[i][2], v[i][3]);
    } else {
      const int p = 4 * (tid + BL * i);
#pragma unroll
      for (int j = 0; j < 4; j++)
        if (p + j >= off && p + j < m) {
          mn = min3_raw(mn, v[i][j], v[i][j]); mx = max3_raw(mx, v[i][j], v[i][j]);
          nan |= v[i][j] != v[i][j];
        }
    }
  }
  mn = wave_fold(mn, [](float a, float b) { return fminf(a, b); });
  mx = wave_fold(mx, [](float a, float b) { return fmaxf(a, b); });
  const bool wave_nan = __ballot(nan) != 0ull;
  if (lane == 0) { ((float*)scratch)[wave] = mn; ((float*)scratch)[NWAVES<BL> + wave] = mx; scratch[2 * NWAVES<BL> + wave] = wave_nan; }
  __syncthreads();
  int any_nan;
  row_range<BL>(scratch, mn, mx, any_nan);   // (scratch is written again behind the histogram's barrier)
  if (any_nan || !(mn > -INFINITY) || !(mx < INFINITY)) return -1;
  const float span = mx - mn;
  if (!(span > 0.f) || !(span < INFINITY)) return 0;
  const int keff = min(K, m - off);
  const float scale = ((float)HBINS - 0.5f) / span;
  if (!(scale < INFINITY)) return 0;         // (a span below 1.2e-35: there would be no bin for any value but the largest)
  auto bin_of = [&](float x) { return (int)((mx - x) * scale); };
#pragma unroll
  for (int i = 0; i < NV; i++) {
    if (i >= nch) continue;
    if (chunk_full(i)) {
#pragma unroll
      for (int j = 0; j < 4; j++) atomicAdd(&hist[bin_of(v[i][j])], 1);
    } else {
      const int p = 4 * (tid + BL * i);
#pragma unroll
      for (int j = 0; j < 4; j++)
        if (p + j >= off && p + j < m) atomicAdd(&hist[bin_of(v[i][j])], 1);
    }
  }
  __syncthreads();
  int tbin, above, c;
  if (!lin_threshold<BL>(hist, scratch, keff, tbin, above, c)) return 0;
#pragma unroll
  for (int i = 0; i < NV; i++) {
    if (i >= nch) continue;
    const int p = 4 * (tid + BL * i);
    const bool full = chunk_full(i);
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (full || (p + j >= off && p + j < m)) {
        const int b = bin_of(v[i][j]);
        if (b <= tbin) obuf[atomicAdd(&hist[b], 1)] = sort_key(v[i][j], p + j - off);
      }
  }
  lin_pad(obuf, above + c);
  __syncthreads();
  lin_rank<BL>(obuf, hist, above + c, keff, K, base_id, bin_of, sv, si);
  return 1;
}

// The tolerant form: values that are not finite (-inf marks a column that cannot be selected) are skipped
// one by one.
template <int BL, int NV>
__device__ __forceinline__ bool select_regs_tolerant(const float (&v)[NV][4], int off, int K, int base_id, int* hist,
                                                     int* scratch, unsigned long long* obuf, float* sv, int* si) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int b = tid; b < HBINS / 4; b += BL) ((int4*)hist)[b] = make_int4(0, 0, 0, 0);
  float mn = INFINITY, mx = -INFINITY;
  int nfin = 0;
#pragma unroll
  for (int i = 0; i < NV; i++)
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (fabsf(v[i][j]) < INFINITY) { mn = fminf(mn, v[i][j]); mx = fmaxf(mx, v[i][j]); nfin++; }
      else if (!(v[i][j] < INFINITY)) mx = INFINITY;   // +inf or NaN: the general path takes the row
  mn = wave_fold(mn, [](float a, float b) { return fminf(a, b); });
  mx = wave_fold(mx, [](float a, float b) { return fmaxf(a, b); });
  nfin = __builtin_amdgcn_readlane(wave_inclusive_sum(nfin), 63);
  if (lane == 0) { ((float*)scratch)[wave] = mn; ((float*)scratch)[NWAVES<BL> + wave] = mx; scratch[2 * NWAVES<BL> + wave] = nfin; }
  __syncthreads();
  row_range<BL>(scratch, mn, mx, nfin);
  const float span = mx - mn;
  if (!(span > 0.f) || !(span < INFINITY)) return false;
  const int keff = min(K, nfin);
  const float scale = ((float)HBINS - 0.5f) / span;
  auto bin_of = [&](float x) { return min(HBINS - 1, (int)((mx - x) * scale)); };
#pragma unroll
  for (int i = 0; i < NV; i++)
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (fabsf(v[i][j]) < INFINITY) atomicAdd(&hist[bin_of(v[i][j])], 1);
  __syncthreads();
  int tbin, above, c;
  if (!lin_threshold<BL>(hist, scratch, keff, tbin, above, c)) return false;
#pragma unroll
  for (int i = 0; i < NV; i++)
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (fabsf(v[i][j]) < INFINITY) {
        const int b = bin_of(v[i][j]);
        if (b <= tbin) obuf[atomicAdd(&hist[b], 1)] = sort_key(v[i][j], 4 * (tid + BL * i) + j - off);
      }
  lin_pad(obuf, above + c);
  __syncthreads();
  lin_rank<BL>(obuf, hist, above + c, keff, K, base_id, bin_of, sv, si);
  return true;
}

template <int BL, int NV>
__device__ __forceinline__ bool linear_select_sort_regs(const float* __restrict__ src, int n, int K, int base_id,
                                                        int* hist, int* scratch, unsigned long long* obuf, float* sv, int* si) {
  float v[NV][4];
  int off, m;
  load_row_regs<BL, NV>(src, n, v, off, m);
  const int r = select_regs_finite<BL, NV>(v, off, m, K, base_id, hist, scratch, obuf, sv, si);
  if (r >= 0) return r == 1;
  __syncthreads();
  return select_regs_tolerant<BL, NV>(v, off, K, base_id, hist, scratch, obuf, sv, si);
}

// LEAN 0: unsorted output, the row staged in LDS where it fits.  1, 2, 3: sorted output, rows held in registers.  1: rows of up
// to REG_ROW elements, the kernel keeps to 128 registers so that four workgroups share a compute unit.  2: rows of up to
// REG_ROW_BIG elements at up to 256 registers (two workgroups per compute unit).  3: BL = 1024, rows of up to REG_ROW_WIDE
// elements at up to 128 registers: one row per compute unit, four times as fast (between the two limits, 300 rows of
// 34000, top-k 64: 171 us on the general path, 25 here).  A launch looks only at the rows whose length lies in
// (n_above, n_upto] and leaves the others to the launch of the other variant.  Rows that the single-sweep path turns down or
// that are too long for it take the general path on global memory and a sorting network: in LDS with 256 threads, whose
// registers are the row's, in registers with 1024 (us, top-k 2048, in LDS / in registers: one row of 40000 81 / 73, 48 of
// 131072 210 / 202, 300 of 65536 398 / 382).  Rows are taken in ascending order (with causal windows the short ones first:
// 0.118 ms at 8192 x 8192 against 0.161 ms longest first and 0.141 ms with short and long rows alternating).
template <int BL, bool STAGED, int LEAN>
__global__ __launch_bounds__(BL, LEAN == 1 ? 4 : LEAN == 2 ? 2 : LEAN == 3 ? 4 : 1) void topk_kernel(
    const float* __restrict__ logits, long ld, const int* __restrict__ row_begin, const int* __restrict__ row_end,
    int width, const int* __restrict__ id_base, int K, int Kp2, float* __restrict__ scores, int* __restrict__ ids,
    int n_above, int n_upto) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  int* hist = (int*)smem;                          // HBINS
  int* scratch = hist + HBINS;                     // SCRATCH<BL>
  float* outv = (float*)(scratch + SCRATCH<BL>);   // Kp2
  int* outi = (int*)(outv + Kp2);                  // Kp2
  unsigned* keys = (unsigned*)(outi + Kp2 + 2 * (LIN_SPARE + LIN_PAD));   // width (STAGED only); the gap extends the (score, id) buffer
  const int tid = threadIdx.x;
  const long row = blockIdx.x;
  const int cb = max(row_begin ? row_begin[row] : 0, 0);
  const int ce = min(row_end ? row_end[row] : width, width);
  const int n = max(ce - cb, 0);
  if (n <= n_above || n > n_upto) return;
  const int base_id = (id_base ? id_base[row] : 0) + cb;
  const float* src = logits + row * ld + cb;
  float* sv = scores + row * (long)K;
  int* si = ids + row * (long)K;

  auto key_at = [&](int e) -> unsigned { return STAGED ? keys[e] : f2key(src[e]); };

  if (LEAN != 0 && n > 0 && n <= SHORT_ROW) {
    if (rank_short_row<BL>(src, n, K, base_id, (unsigned long long*)outv, sv, si)) return;
    __syncthreads();
  } else if (LEAN != 0 && n > 0) {   // single-sweep path, also for rows shorter than K
    if (LEAN == 1 && n + 3 <= REG_ROW) {
      bool done;
      unsigned long long* obuf = (unsigned long long*)outv;
      if (n + 3 <= 4 * BL) done = linear_select_sort_regs<BL, 1>(src, n, K, base_id, hist, scratch, obuf, sv, si);
      else if (n + 3 <= 8 * BL) done = linear_select_sort_regs<BL, 2>(src, n, K, base_id, hist, scratch, obuf, sv, si);
      else if (n + 3 <= 16 * BL) done = linear_select_sort_regs<BL, 4>(src, n, K, base_id, hist, scratch, obuf, sv, si);
      else done = linear_select_sort_regs<BL, REG_ROW / (4 * BL)>(src, n, K, base_id, hist, scratch, obuf, sv, si);
      if (done) return;
      __syncthreads();
    } else if (LEAN == 2 && n + 3 <= REG_ROW_BIG) {
      bool done;
      unsigned long long* obuf = (unsigned long long*)outv;
      if (n + 3 <= 16 * 4 * BL) done = linear_select_sort_regs<BL, 16>(src, n, K, base_id, hist, scratch, obuf, sv, si);
      else if (n + 3 <= 24 * 4 * BL) done = linear_select_sort_regs<BL, 24>(src, n, K, base_id, hist, scratch, obuf, sv, si);
      else done = linear_select_sort_regs<BL, REG_ROW_BIG / (4 * BL)>(src, n, K, base_id, hist, scratch, obuf, sv, si);
      if (done) return;
      __syncthreads();
    } else if (LEAN == 3 && n + 3 <= REG_ROW_WIDE) {
      bool done;
      unsigned long long* obuf = (unsigned long long*)outv;
      if (n + 3 <= 4 * BL) done = linear_select_sort_regs<BL, 1>(src, n, K, base_id, hist, scratch, obuf, sv, si);
      else if (n + 3 <= 2 * 4 * BL) done = linear_select_sort_regs<BL, 2>(src, n, K, base_id, hist, scratch, obuf, sv, si);
      else if (n + 3 <= 4 * 4 * BL) done = linear_select_sort_regs<BL, 4>(src, n, K, base_id, hist, scratch, obuf, sv, si);
      else done = linear_select_sort_regs<BL, REG_ROW_WIDE / (4 * BL)>(src, n, K, base_id, hist, scratch, obuf, sv, si);
      if (done) return;
      __syncthreads();
    }
  }
  if (n <= K) {
    for (int t = tid; t < Kp2; t += BL) {
      float v = t < n ? src[t] : -INFINITY;
      outv[t] = v;
      outi[t] = (t < n && v != -INFINITY) ? base_id + t : -1;
    }
  } else {
    if (STAGED) {
      for (int e = tid; e < n; e += BL) keys[e] = f2key(src[e]);
    }
    // ---- pass 1: bits [31:20] ------------------------------------------------------------
    for (int b = tid; b < HBINS; b += BL) hist[b] = 0;
    __syncthreads();
    for (int e = tid; e < n; e += BL) atomicAdd(&hist[key_at(e) >> 20], 1);
    __syncthreads();
    Pick p1 = pick_bin<BL>(hist, 4096, K, scratch, scratch + 3 * NWAVES<BL>);
    int need = K - p1.above;
    // ---- pass 2: bits [19:10] among keys in bin p1 -----------------------------------------
    for (int b = tid; b < 1024; b += BL) hist[b] = 0;
    __syncthreads();
    for (int e = tid; e < n; e += BL) {
      unsigned k = key_at(e);
      if ((int)(k >> 20) == p1.bin) atomicAdd(&hist[(k >> 10) & 1023], 1);
    }
    __syncthreads();
    Pick p2 = pick_bin<BL>(hist, 1024, need, scratch, scratch + 3 * NWAVES<BL>);
    need -= p2.above;
    // ---- pass 3: bits [9:0] ----------------------------------------------------------------
    const unsigned pre22 = ((unsigned)p1.bin << 10) | (unsigned)p2.bin;
    for (int b = tid; b < 1024; b += BL) hist[b] = 0;
    __syncthreads();
    for (int e = tid; e < n; e += BL) {
      unsigned k = key_at(e);
      if ((k >> 10) == pre22) atomicAdd(&hist[k & 1023], 1);
    }
    __syncthreads();
    Pick p3 = pick_bin<BL>(hist, 1024, need, scratch, scratch + 3 * NWAVES<BL>);
    const unsigned thr = (pre22 << 10) | (unsigned)p3.bin;   // the K-th largest key
    const int ties = need - p3.above;                         // how many keys == thr to keep (>= 1)
    // ---- compaction in ascending column order ------------------------------------------------
    if constexpr (STAGED || LEAN == 1) {     // a run of columns per thread: the row is in LDS or fits the first cache
      const int cs = (n + BL - 1) / BL;
      const int e0 = min(tid * cs, n), e1 = min(e0 + cs, n);
      int ngt = 0, neq = 0;
      for (int e = e0; e < e1; e++) { unsigned k = key_at(e); ngt += k > thr; neq += k == thr; }
      int tot;
      const int eq_before = block_exscan<BL, true>(neq, scratch, tot);
      const int eq_take = max(0, min(neq, ties - eq_before));
      int pos = block_exscan<BL, false>(ngt + eq_take, scratch, tot);
      int eq_seen = 0;
      for (int e = e0; e < e1; e++) {
        unsigned k = key_at(e);
        bool take = k > thr;
        if (k == thr) { take = eq_seen < eq_take; eq_seen++; }
        if (take) {
          float v = key2f(k);
          outv[pos] = v;
          outi[pos] = v != -INFINITY ? base_id + e : -1;
          pos++;
        }
      }
    } else {
      // A run per wave, 64 consecutive columns per load.  (With a run per thread every lane's load touches a line of its own,
      // and a workgroup's lines do not fit the first cache.  us, top-k 2048, per thread / per wave: one row of 65536 106 / 79,
      // 300 rows 385 / 209, 1024 rows 1201 / 501, 300 rows of 131072 unsorted 785 / 680.  From LDS a run per thread is the
      // better one: 1024 rows of 7000 unsorted 52 / 58, and from the first cache: 300 rows of 2500 with ties 70 / 73.)
      const int lane = tid & 63, wave = tid >> 6;
      const int run = ((n + NWAVES<BL> - 1) / NWAVES<BL> + 63) / 64 * 64;
      const int e0 = min(wave * run, n), e1 = min(e0 + run, n);
      // fn(first column, their keys, whether this lane's column is one) for 64 columns of the run after the other
      auto each = [&](auto fn) {
        for (int e = e0; e < e1; e += 64 * COMPACT_FLIGHT) {
          unsigned k[COMPACT_FLIGHT];
#pragma unroll
          for (int u = 0; u < COMPACT_FLIGHT; u++) k[u] = key_at(min(e + 64 * u + lane, e1 - 1));
#pragma unroll
          for (int u = 0; u < COMPACT_FLIGHT; u++)
            if (e + 64 * u < e1) fn(e + 64 * u, k[u], e + 64 * u + lane < e1);
        }
      };
      int ngt = 0, neq = 0;
      each([&](int, unsigned k, bool in) {
        ngt += (int)__popcll(__ballot(in && k > thr));
        neq += (int)__popcll(__ballot(in && k == thr));
      });
      if (lane == 0) { scratch[wave] = ngt; scratch[NWAVES<BL> + wave] = neq; }
      __syncthreads();
      int pos = 0, left = ties;                // output position and ties left at the wave's first column
      for (int w = 0; w < wave; w++) {
        const int q = min(scratch[NWAVES<BL> + w], left);
        pos += scratch[w] + q;
        left -= q;
      }
      const unsigned long long below = (1ull << lane) - 1ull;
      each([&](int e, unsigned k, bool in) {
        const unsigned long long eq = __ballot(in && k == thr);
        const int eq_before = (int)__popcll(eq & below), eq_here = (int)__popcll(eq);
        const bool take = in && (k > thr || (k == thr && eq_before < left));
        const unsigned long long all = __ballot(take);
        if (take) {
          const int p = pos + (int)__popcll(all & below);
          const float v = key2f(k);
          outv[p] = v;
          outi[p] = v != -INFINITY ? base_id + e + lane : -1;
        }
        pos += (int)__popcll(all);
        left = max(left - eq_here, 0);
      });
    }
    for (int t = K + tid; t < Kp2; t += BL) { outv[t] = -INFINITY; outi[t] = -1; }
  }
  __syncthreads();

  if (LEAN != 0) {   // bitonic sort, descending score, ascending id among equal scores
    // in registers where the kernel has them to spare: every row too long for the single sweep comes this way
    if (LEAN == 3 && Kp2 >= BL) {
      unsigned long long* xbuf = (unsigned long long*)outv;
      if (Kp2 == BL) bitonic_regs<BL, 1>(outv, outi, xbuf, Kp2, sv, si, K);
      else if (Kp2 == 2 * BL) bitonic_regs<BL, 2>(outv, outi, xbuf, Kp2, sv, si, K);
      else if (Kp2 == 4 * BL) bitonic_regs<BL, 4>(outv, outi, xbuf, Kp2, sv, si, K);
      else bitonic_regs<BL, 8>(outv, outi, xbuf, Kp2, sv, si, K);
      return;
    }
    for (int size = 2; size <= Kp2; size <<= 1) {
      for (int stride = size >> 1; stride > 0; stride >>= 1) {
        for (int t = tid; t < (Kp2 >> 1); t += BL) {
          const int lo = 2 * t - (t & (stride - 1));
          const int hi = lo + stride;
          const bool desc = ((lo & size) == 0);
          const float a = outv[lo], b = outv[hi];
          const int ia = outi[lo], ib = outi[hi];
          if (comes_first(a, ia, b, ib) != desc) { outv[lo] = b; outv[hi] = a; outi[lo] = ib; outi[hi] = ia; }
        }
        __syncthreads();
      }
    }
  }
  for (int t = tid; t < K; t += BL) { sv[t] = outv[t]; si[t] = outi[t]; }
}

}  // namespace

int dsa_topk_launch(const float* logits, int S, int64_t ld, const int32_t* row_begin, const int32_t* row_end,
                    int width, const int32_t* id_base, int K, int sorted, float* scores, int32_t* ids,
                    hipStream_t st) {
  DSA_REQUIRE(S >= 0 && width > 0 && ld >= width && K > 0, "dsa_topk: bad sizes S=%d width=%d K=%d", S, width, K);
  DSA_REQUIRE(K <= 8192, "dsa_topk: K=%d exceeds the supported maximum 8192", K);
  if (S == 0) return DSA_OK;
  int Kp2 = 1;
  while (Kp2 < K) Kp2 <<= 1;
  const size_t buffers = (size_t)HBINS * 4 + (size_t)Kp2 * 8 + (size_t)(LIN_SPARE + LIN_PAD) * 8;
  const size_t fixed = buffers + SCRATCH<256> * 4, wide = buffers + SCRATCH<1024> * 4;
  const size_t staged = fixed + (size_t)width * 4;
  // Sorted rows that fit a register variant need no staging buffer: rows of up to REG_ROW elements go to the
  // 128-register kernel (four workgroups per compute unit), longer ones to a second launch; each launch skips the
  // other's rows.  Only the device knows how long they are (a window of a wide key array may be short).  With no more rows
  // than compute units the 1024-thread kernel takes them all and finishes a row sooner (us, top-k 2048: one row of 4096
  // 11.5 -> 7.7, of 32768 29 -> 13.7, 48 windows of 7000 in a wide array 65 -> 10; 300 rows of 8000 16.5 against 17.6).
  const int none = 0x7fffffff, split = REG_ROW - 3;
  auto launch = [&](auto kern, int block, size_t smem, int n_above, int n_upto) {
    if (dsa_reserve_lds((const void*)kern, smem) != hipSuccess) return false;
    kern<<<dim3(S), dim3(block), smem, st>>>(logits, (long)ld, row_begin, row_end, width, id_base, K, Kp2, scores, ids,
                                             n_above, n_upto);
    return true;
  };
  bool ok;
  if (sorted && S <= WIDE_ROWS) {
    ok = launch(topk_kernel<1024, false, 3>, 1024, wide, -1, none);
  } else if (sorted) {
    ok = launch(topk_kernel<256, false, 1>, 256, fixed, -1, split);
    if (ok && width > split) {
      if (width + 3 <= REG_ROW_BIG) ok = launch(topk_kernel<256, false, 2>, 256, fixed, split, none);
      else ok = launch(topk_kernel<1024, false, 3>, 1024, wide, split, none);
    }
  } else if (staged <= 160 * 1024) {
    ok = launch(topk_kernel<256, true, 0>, 256, staged, -1, none);
  } else {
    ok = launch(topk_kernel<256, false, 0>, 256, fixed, -1, none);
  }
  if (!ok) DSA_FAIL(DSA_ERR_LAUNCH, "dsa_topk: cannot reserve LDS");
  DSA_CHECK_LAUNCH("dsa_topk");
  return DSA_OK;
}

extern "C" int dsa_topk(const float* logits, int S, int64_t ld, const int32_t* row_begin, const int32_t* row_end,
                        int width, const int32_t* id_base, int K, int sorted, float* scores, int32_t* ids,
                        void* stream) {
  return dsa_topk_launch(logits, S, ld, row_begin, row_end, width, id_base, K, sorted, scores, ids,
                         (hipStream_t)stream);
}

// ---- fused indexer forward: logits of one query block at a time, then its top-k ----------------
int dsa_indexer_logits_block(const void* q8, const float* q_w, const void* k8, const float* k_scale,
                             const int32_t* ks, const int32_t* ke, int S, int Hi, int Sk, float* logits,
                             int64_t ld, int width, int relative, int clean, int q_begin, int q_count,
                             hipStream_t st);

static int fused_block_rows(int Sk) {
  // one block's logits stay within the 256 MiB memory-side cache where that still leaves a block 8192 queries:
  // 1024 workgroups of 8 queries, four rounds over the 256 compute units (blocks of 2048 queries - one workgroup per
  // compute unit, half of what fits - took 2.6 ms for 32768 packed tokens where blocks of 8192 take 1.9 ms)
  long rows = (256l << 20) / ((long)(Sk > 0 ? Sk : 1) * 4);         // (no keys: refused by the logits kernel's checks)
  rows = rows < 8192 ? 8192 : rows;
  return (int)(rows / 8 * 8);
}

extern "C" size_t dsa_indexer_topk_workspace_bytes(int S, int Sk, int K) {
  (void)K;
  int rows = fused_block_rows(Sk);
  if (rows > S) rows = (S + 7) / 8 * 8;
  return (size_t)rows * (size_t)Sk * 4;
}

// Logits of `rows` queries at a time into lg ([rows][Sk] floats), then their top-k.
static int indexer_topk_blocks(const void* q8, const float* q_w, const void* k8, const float* k_scale, const int32_t* ks,
                               const int32_t* ke, int S, int Hi, int Sk, int K, int sorted, float* scores, int32_t* ids,
                               float* lg, int rows, hipStream_t st) {
  for (int q0 = 0; q0 < S; q0 += rows) {
    const int cnt = S - q0 < rows ? S - q0 : rows;
    int rc = dsa_indexer_logits_block(q8, q_w, k8, k_scale, ks, ke, S, Hi, Sk, lg, Sk, Sk, 0, 0, q0, cnt, st);
    if (rc != DSA_OK) return rc;
    rc = dsa_topk_launch(lg, cnt, Sk, ks + q0, ke + q0, Sk, nullptr, K, sorted, scores + (size_t)q0 * K,
                         ids + (size_t)q0 * K, st);
    if (rc != DSA_OK) return rc;
  }
  return DSA_OK;
}

extern "C" int dsa_indexer_topk_fwd(const void* q8, const float* q_w, const void* k8, const float* k_scale,
                                    const int32_t* ks, const int32_t* ke, int S, int Hi, int Sk, int K, int sorted,
                                    float* scores, int32_t* ids, void* workspace, size_t workspace_bytes,
                                    void* stream) {
  if (S == 0) return DSA_OK;
  DSA_REQUIRE(workspace != nullptr && workspace_bytes >= dsa_indexer_topk_workspace_bytes(S, Sk, K),
              "dsa_indexer_topk_fwd: workspace of %zu bytes is too small", workspace_bytes);
  return indexer_topk_blocks(q8, q_w, k8, k_scale, ks, ke, S, Hi, Sk, K, sorted, scores, ids, (float*)workspace,
                             fused_block_rows(Sk), (hipStream_t)stream);
}

// ---- the same without any allocation by anyone: the logits blocks live in a device array of the library ----
// For callers that cannot allocate device memory (code under HIP graph capture, tight serving loops):
// they pass inputs and outputs only.  Every GPU the library runs on holds its own copy of the array
// until the process ends; calls that overlap on one GPU share it and race - order them on one stream.
constexpr size_t STATIC_SCRATCH_BYTES = (size_t)64 << 20;
constexpr int STATIC_MIN_ROWS = 256;           // a block of fewer queries would leave most compute units idle
static __device__ __align__(256) unsigned char scratch[STATIC_SCRATCH_BYTES];

#include <mutex>
static std::mutex scratch_mutex;
static void* scratch_ptr[64];                  // per device: the array's address on that device (0 = not asked yet)

extern "C" int dsa_indexer_topk_fwd_static(const void* q8, const float* q_w, const void* k8, const float* k_scale,
                                           const int32_t* ks, const int32_t* ke, int S, int Hi, int Sk, int K,
                                           int sorted, float* scores, int32_t* ids, void* stream) {
  if (S == 0) return DSA_OK;
  DSA_REQUIRE(Sk > 0 && (size_t)Sk * 4 * STATIC_MIN_ROWS <= STATIC_SCRATCH_BYTES,
              "dsa_indexer_topk_fwd_static: at most %zu keys fit the library's %zu MiB scratch array, got %d "
              "(use dsa_indexer_topk_fwd with a workspace)",
              STATIC_SCRATCH_BYTES / (4 * STATIC_MIN_ROWS), STATIC_SCRATCH_BYTES >> 20, Sk);
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64)
    DSA_FAIL(DSA_ERR_LAUNCH, "dsa_indexer_topk_fwd_static: no current device");
  void* base;
  {
    std::lock_guard<std::mutex> lock(scratch_mutex);
    if (scratch_ptr[dev] == nullptr) {         // first call on this device: the array's address here
      void* p = nullptr;
      const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
      if (e != hipSuccess || p == nullptr)
        DSA_FAIL(DSA_ERR_LAUNCH, "dsa_indexer_topk_fwd_static: hipGetSymbolAddress failed: %s", hipGetErrorString(e));
      scratch_ptr[dev] = p;
    }
    base = scratch_ptr[dev];
  }
  int rows = (int)(STATIC_SCRATCH_BYTES / ((size_t)Sk * 4)) / 8 * 8;
  // (nothing in the array has to start at zero: the logits kernel writes columns [ks, ke) of every row of a block
  // and the selection reads no others)
  return indexer_topk_blocks(q8, q_w, k8, k_scale, ks, ke, S, Hi, Sk, K, sorted, scores, ids, (float*)base, rows,
                             (hipStream_t)stream);
}
