// Key-sorted order of the valid (query, slot) pairs of a block of queries, built with integer
// work only (bitmap over queries per key, prefix popcounts over the queries, exclusive scan over keys), so it is
// identical from run to run.  Used by the deterministic scatter-accumulations of the backward
// kernels: pair (q, slot) with key v gets row  start[v] + #{q' < q : q' selects v}.
// Ids within one query row must be distinct (any top-k guarantees it): a repeated id has one bit and
// one row like any other, so one of its contributions would be lost.  The first kernel notices a
// repeated id (the bit it sets is set already) and raises *dup_flag; the callers' last kernels then
// fill their outputs with NaN instead of returning sums that silently miss a term.
#pragma once
#include <type_traits>

#include "dsa_common.h"

namespace order {

static __global__ void zero_u32_kernel(unsigned* __restrict__ p, size_t n) {
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) p[e] = 0u;
}

// bitmap[w][key] bit b  <=>  local query 32w + b selects key (keys contiguous: the kernels behind it read it along the keys).
// Built without global atomics, in two steps.  (1) One workgroup per query sets the query's bits
// over the keys in LDS and writes them out as one row of qmap[query][key / 32] (Wk words).
// (2) A transpose of the bit matrix: a wave loads the words of 64 consecutive queries for 64 keys and turns them in its registers.
static __global__ __launch_bounds__(256) void qmap_kernel(const int* __restrict__ ids, int q0, int cnt, int K, int Skv,
                                                          int q_start, unsigned* __restrict__ qmap, int Wk,
                                                          int* __restrict__ sorted, int* __restrict__ dup_flag) {
  extern __shared__ unsigned qbits[];        // Wk words; with `sorted`, Wk more for the prefix counts and K for the list
  __shared__ int wave_tot[4];
  const int ql = blockIdx.x;
  for (int w = threadIdx.x; w < Wk; w += 256) qbits[w] = 0u;
  __syncthreads();
  for (int t0 = threadIdx.x; t0 < K; t0 += 8 * 256) {
    int v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = t0 + i * 256 < K ? ids[(size_t)(q0 + ql) * K + t0 + i * 256] : -1;
#pragma unroll
    for (int i = 0; i < 8; i++)
      if (v[i] >= 0 && v[i] < Skv && v[i] <= q_start + q0 + ql) {
        const unsigned bit = 1u << (v[i] & 31);
        if (atomicOr(&qbits[v[i] >> 5], bit) & bit) *dup_flag = 1;      // every writer stores the same value
      }
  }
  __syncthreads();
  for (int w = threadIdx.x; w < Wk; w += 256) qmap[(size_t)ql * Wk + w] = qbits[w];
  if (sorted == nullptr) return;
  // The query's valid ids in ascending order, -1 after them: id v goes to position (set bits below v).
  // Thread t counts the words [t * per, (t + 1) * per); an exclusive scan over the threads gives each
  // thread its base, from which it writes the per-word prefix counts.
  unsigned* pre = qbits + Wk;
  const int per = (Wk + 255) / 256;
  const int w0 = threadIdx.x * per;
  int mine = 0;
  for (int w = w0; w < w0 + per && w < Wk; w++) mine += __popc(qbits[w]);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int inc = mine;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) { int n = __shfl_up(inc, o, 64); if (lane >= o) inc += n; }
  if (lane == 63) wave_tot[wave] = inc;
  __syncthreads();
  int base = inc - mine;
  for (int w = 0; w < wave; w++) base += wave_tot[w];
  const int total = wave_tot[0] + wave_tot[1] + wave_tot[2] + wave_tot[3];
  for (int w = w0; w < w0 + per && w < Wk; w++) { pre[w] = (unsigned)base; base += __popc(qbits[w]); }
  __syncthreads();
  int* list = (int*)(pre + Wk);              // K ints: the list is put together in LDS and written out in order
  for (int t = total + threadIdx.x; t < K; t += 256) list[t] = -1;
  for (int t = threadIdx.x; t < K; t += 256) {
    const int v = ids[(size_t)(q0 + ql) * K + t];
    if (v >= 0 && v < Skv && v <= q_start + q0 + ql)
      list[pre[v >> 5] + __popc(qbits[v >> 5] & ((1u << (v & 31)) - 1u))] = v;
  }
  __syncthreads();
  int* row = sorted + (size_t)ql * K;
  for (int t = threadIdx.x; t < K; t += 256) row[t] = list[t];
}

// ---- groups of G consecutive queries that may be worked as one unit ----
// bad[w] bit b  <=>  row 32 w + b of kv (row16 pieces of 16 bytes, bf16) holds a value that is not finite.  Also clears the flags
// of repeated ids and of units.
static __global__ __launch_bounds__(256) void kv_check_kernel(const uint4* __restrict__ kv, int Skv, int row16, unsigned* __restrict__ bad,
                                                              int* __restrict__ flags) {
  __shared__ unsigned word;
  if (threadIdx.x == 0) {
    word = 0u;
    if (blockIdx.x == 0) flags[0] = flags[1] = 0;
  }
  __syncthreads();
  const int n = min(32, Skv - 32 * (int)blockIdx.x) * row16;
  const uint4* p = kv + (size_t)blockIdx.x * 32 * row16;
  constexpr int AHEAD = 9;                   // all of 32 rows of 576 values
  for (int e0 = threadIdx.x; e0 < n; e0 += AHEAD * 256) {
    uint4 v[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; i++) v[i] = p[min(e0 + i * 256, n - 1)];
#pragma unroll
    for (int i = 0; i < AHEAD; i++) {
      const unsigned w[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
      bool inf = false;
#pragma unroll
      for (int j = 0; j < 4; j++) inf |= (w[j] & 0x7f80u) == 0x7f80u || (w[j] & 0x7f800000u) == 0x7f800000u;
      if (inf) atomicOr(&word, 1u << (min(e0 + i * 256, n - 1) / row16));
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) bad[blockIdx.x] = word;
}

// What a group costs as one unit and as single queries: a fixed part and a part per 32 slots each
struct UnitCost { int unit_fixed, unit_tile, fixed, tile; };

// Words of a key bitmap in LDS: whole 16-byte pieces
__host__ __device__ inline int unit_words(int n) { return (n + 3) / 4 * 4; }
// qmap_kernel for a group of G queries per workgroup.  dup_flag[1]: there is a unit.  units[group] = slots of the unit, a multiple of 32,
// or 0 for single queries.  A unit has the bits of all its queries in its first one's row of qmap, so that it counts as one query in
// everything behind; its list (G K places from the first query's on) holds key | queries << 24.  Not a unit: groups that lack a query
// at the end, without a key or with more than max_slots, keys with values that are not finite (a product over the slots would carry
// them to the queries that do not have them), and what costs less query by query.
// Like qmap_kernel it goes over the words of the key bitmap, four at a time, and over the ids; it is bound by latency, LDS traffic and the
// workgroups that the LDS leaves room for.  us, with the lists made by a walk over all keys / as they are; qmap_kernel, for queries by
// themselves: 8000 queries x 256 slots of 8000 keys in pairs 43 / 22; 16, of 131072 312 / 68; 100; 3000 x 2048 of 32768 48 / 22; 18; in fours
// 8000 x 256 of 32768 69 / 22; 21, 2000 x 512 of 131072 144 / 27; 31.
template <int G, int BL>
static __global__ __launch_bounds__(BL) void qmap_unit_kernel(const int* __restrict__ ids, int q0, int cnt, int K, int Skv, int q_start,
                                                               unsigned* __restrict__ qmap, int Wk, int* __restrict__ sorted,
                                                               int* __restrict__ dup_flag, const unsigned* __restrict__ bad,
                                                               int* __restrict__ units, int max_slots, UnitCost cost) {
  extern __shared__ __attribute__((aligned(16))) unsigned qbits[];      // [G][WL] bits, [G / 2][WL] prefix counts, 16 bits each, [G][K] list
  __shared__ unsigned wave_tot[G / 2 + 1][BL / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ql0 = blockIdx.x * G, nq = min(G, cnt - ql0), n_ids = nq * K;
  const int WL = unit_words(Wk);
  unsigned* pre = qbits + G * WL;
  int* list = (int*)(pre + G / 2 * WL);
  const int* src = ids + (size_t)(q0 + ql0) * K;
  // f(id, query) for every valid id, the first 8 of a thread requested ahead
  int v[8];
  auto request = [&](int t0) {
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = src[min(t0 + i * BL, n_ids - 1)];
  };
  auto each_id = [&](bool have, auto f) {
    for (int t0 = tid; t0 < n_ids; t0 += 8 * BL) {
      if (!have || t0 >= 8 * BL) request(t0);
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int t = t0 + i * BL, j = __builtin_amdgcn_readfirstlane(t / K);        // (K is a multiple of 64: the same for a wave)
        if (t < n_ids && v[i] >= 0 && v[i] < Skv && v[i] <= q_start + q0 + ql0 + j) f(v[i], j);
      }
    }
  };
  request(tid);
  for (int w = 4 * tid; w < G * WL; w += 4 * BL) *(uint4*)(qbits + w) = make_uint4(0u, 0u, 0u, 0u);
  __syncthreads();
  each_id(true, [&](int id, int j) {
    const unsigned bit = 1u << (id & 31);
    if (atomicOr(&qbits[j * WL + (id >> 5)], bit) & bit) *dup_flag = 1;
  });
  __syncthreads();
  // one scan over the threads: the queries' counts in pairs (a query has at most 2048 keys), then the union's beside the number of
  // threads that saw a key with values that are not finite
  const int per = unit_words((Wk + BL - 1) / BL), w0 = min(tid * per, WL), w1 = min(w0 + per, WL);
  constexpr int NC = G / 2 + 1;
  unsigned mine[NC], inc[NC], total[NC];
#pragma unroll
  for (int c = 0; c < NC; c++) mine[c] = 0u;
  bool sees_bad = false;
  struct Words { unsigned own[G][4], any[4]; };
  auto words = [&](int w) {                  // of four neighbouring words: the queries' bits and their union
    Words x;
#pragma unroll
    for (int j = 0; j < G; j++) {
      const uint4 b = *(const uint4*)(qbits + j * WL + w);
      const unsigned y[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
      for (int i = 0; i < 4; i++) {
        x.own[j][i] = y[i];
        x.any[i] = j ? x.any[i] | y[i] : y[i];
      }
    }
    return x;
  };
  for (int w = w0; w < w1; w += 4) {
    const Words x = words(w);
    const uint4 b = *(const uint4*)(bad + w);
    sees_bad |= ((x.any[0] & b.x) | (x.any[1] & b.y) | (x.any[2] & b.z) | (x.any[3] & b.w)) != 0u;
#pragma unroll
    for (int i = 0; i < 4; i++) {
#pragma unroll
      for (int j = 0; j < G; j++) mine[j / 2] += (unsigned)__popc(x.own[j][i]) << (16 * (j & 1));
      mine[NC - 1] += __popc(x.any[i]);
    }
  }
  if (sees_bad) mine[NC - 1] |= 0x10000u;
#pragma unroll
  for (int c = 0; c < NC; c++) {
    inc[c] = mine[c];
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) { const unsigned x = __shfl_up(inc[c], o, 64); if (lane >= o) inc[c] += x; }
    if (lane == 63) wave_tot[c][wave] = inc[c];
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < NC; c++) {
    inc[c] -= mine[c];
    total[c] = 0u;
#pragma unroll
    for (int w = 0; w < BL / 64; w++) {
      if (w < wave) inc[c] += wave_tot[c][w];
      total[c] += wave_tot[c][w];
    }
  }
  const int keys = (int)(total[NC - 1] & 0xffffu), tiles = (keys + 31) / 32;
  int n[G], apart = 0;
#pragma unroll
  for (int j = 0; j < G; j++) {
    n[j] = (int)(total[j / 2] >> (16 * (j & 1)) & 0xffffu);
    apart += n[j] ? cost.fixed + cost.tile * ((n[j] + 31) / 32) : 0;
  }
  const bool unit = nq == G && keys > 0 && 32 * tiles <= max_slots && total[NC - 1] >> 16 == 0u && cost.unit_fixed + cost.unit_tile * tiles <= apart;
  if (tid == 0) {
    units[blockIdx.x] = unit ? 32 * tiles : 0;
    if (unit) dup_flag[1] = 1;
  }
  inc[NC - 1] &= 0xffffu;
  for (int w = w0; w < w1; w += 4) {
    const Words x = words(w);
    unsigned p[NC - 1][4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      if (unit) {
        p[0][i] = inc[NC - 1];
        inc[NC - 1] += __popc(x.any[i]);
      } else {
#pragma unroll
        for (int c = 0; c < NC - 1; c++) {
          p[c][i] = inc[c];
          inc[c] += (unsigned)__popc(x.own[2 * c][i]) + ((unsigned)__popc(x.own[2 * c + 1][i]) << 16);
        }
      }
    }
#pragma unroll
    for (int c = 0; c < NC - 1; c++)
      if (!unit || c == 0) *(uint4*)(pre + c * WL + w) = make_uint4(p[c][0], p[c][1], p[c][2], p[c][3]);
  }
  auto any = [&](int w) {
    unsigned b = qbits[w];
#pragma unroll
    for (int j = 1; j < G; j++) b |= qbits[j * WL + w];
    return b;
  };
  for (int j = 0; j < nq; j++)
    for (int w = tid; w < Wk; w += BL) qmap[(size_t)(ql0 + j) * Wk + w] = !unit ? qbits[j * WL + w] : j == 0 ? any(w) : 0u;
  __syncthreads();
  // the lists, ascending: an id's place is the number of set bits below it (an id of several queries of a unit is put there by each)
  each_id(n_ids <= 8 * BL, [&](int id, int j) {
    const int w = id >> 5, b = id & 31;
    const unsigned below = (1u << b) - 1u;
    if (unit) {
      unsigned bits = 0u;
      int entry = id;
#pragma unroll
      for (int k = 0; k < G; k++) {
        const unsigned own = qbits[k * WL + w];
        bits |= own;
        entry |= (int)(own >> b & 1u) << (24 + k);
      }
      list[pre[w] + __popc(bits & below)] = entry;
    } else {
      list[j * K + (int)(pre[(j >> 1) * WL + w] >> (16 * (j & 1)) & 0xffffu) + __popc(qbits[j * WL + w] & below)] = id;
    }
  });
  if (unit) {
    for (int t = keys + tid; t < n_ids; t += BL) list[t] = -1;
  } else {
#pragma unroll
    for (int j = 0; j < G; j++)
      if (j < nq)
        for (int t = n[j] + tid; t < K; t += BL) list[j * K + t] = -1;
  }
  __syncthreads();
  int* row = sorted + (size_t)ql0 * K;
  for (int t = 4 * tid; t < n_ids; t += 4 * BL) *(int4*)(row + t) = *(const int4*)(list + t);
}

// A 64 x 64 bit matrix across a wave, lane = row with columns 0 - 31 in `lo` and 32 - 63 in `hi`, becomes its transpose.
__device__ __forceinline__ void transpose64(unsigned& lo, unsigned& hi, int lane) {
  // the off-diagonal quarters: the upper half-wave's lo against the lower one's hi
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(lo), "+v"(hi));
  // then bit o of lane and column for o = 16 .. 1: half of the bits are the partner's, from o columns to the right or left
  auto step = [&](auto o_c, unsigned m) {
    constexpr int o = decltype(o_c)::value;
    const bool up = lane & o;
    const unsigned take = up ? m : ~m, by = up ? o : 32 - o;
    auto swap = [&](unsigned& x) {
      const unsigned y = (unsigned)__builtin_amdgcn_ds_swizzle((int)x, o << 10 | 0x1f);
      x = (x & ~take) | (__builtin_amdgcn_alignbit(y, y, by) & take);
    };
    swap(lo);
    swap(hi);
  };
  step(std::integral_constant<int, 16>{}, 0x0000ffffu);
  step(std::integral_constant<int, 8>{}, 0x00ff00ffu);
  step(std::integral_constant<int, 4>{}, 0x0f0f0f0fu);
  step(std::integral_constant<int, 2>{}, 0x33333333u);
  step(std::integral_constant<int, 1>{}, 0x55555555u);
}

// inclusive sums over the lanes of a wave, within the vector unit (rows of 16 lanes, then their ends to the rows behind them)
__device__ __forceinline__ int wave_sums(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);       // row_shr 1, 2, 4, 8
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);      // row_bcast 15, into rows 1 and 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);      // row_bcast 31, into rows 2 and 3
  return x;
}

// What there is to do where some groups of G queries are units: work[2 ..] = first query << 8 | tiles of 32 slots for the units, query << 8
// for the queries by themselves, both from the last query on; work[0] entries in all, work[1] those of the kind that comes first, which
// is the rarer one (a few long queries behind everything else would end alone).  The two kinds apart, because a workgroup that does the
// one and its neighbour that does the other displace each other's code from the instruction cache that they share.
struct WorkList { const int* units; int cnt, G; int* work; };

// One workgroup of 1024 threads, each with a run of the groups, which it counts and then, from the counts of those before it, writes.
__device__ __forceinline__ void make_work_list(const WorkList& list) {
  __shared__ int wave_units[16], wave_apart[16];
  const int G = list.G, groups = (list.cnt + G - 1) / G, per = (groups + 1023) / 1024;
  const int k0 = min((int)threadIdx.x * per, groups), k1 = min(k0 + per, groups);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int units = 0, apart = 0;
  for (int k = k0; k < k1; k++) {
    if (list.units[groups - 1 - k] / 32) units++;
    else apart += min(G, list.cnt - (groups - 1 - k) * G);
  }
  int at_u = wave_sums(units), at_a = wave_sums(apart);
  if (lane == 63) { wave_units[wave] = at_u; wave_apart[wave] = at_a; }
  __syncthreads();
  at_u -= units;
  at_a -= apart;
  int n_units = 0, n_apart = 0;
  for (int w = 0; w < 16; w++) {
    if (w < wave) { at_u += wave_units[w]; at_a += wave_apart[w]; }
    n_units += wave_units[w];
    n_apart += wave_apart[w];
  }
  const bool units_first = n_units <= n_apart;
  int* to_u = list.work + 2 + (units_first ? 0 : n_apart) + at_u;
  int* to_a = list.work + 2 + (units_first ? n_units : 0) + at_a;
  for (int k = k0; k < k1; k++) {
    const int g = groups - 1 - k, tiles = list.units[g] / 32;
    if (tiles) *to_u++ = (g * G) << 8 | tiles;
    else for (int j = min(G, list.cnt - g * G) - 1; j >= 0; j--) *to_a++ = (g * G + j) << 8;
  }
  if (threadIdx.x == 0) {
    list.work[0] = n_units + n_apart;
    list.work[1] = min(n_units, n_apart);
  }
}

// A share of the clearing of `marks` (n_marks of 16 bytes), which are read if there is a unit: it goes beside kernels that leave most of
// the chip idle.
struct Marks { const int* flags; uint4* at; size_t n; int blocks; };
__device__ __forceinline__ void clear_marks(const Marks& m, int block) {
  if (m.flags[1])
    for (size_t e = (size_t)block * 1024 + threadIdx.x; e < m.n; e += (size_t)m.blocks * 1024) m.at[e] = make_uint4(0u, 0u, 0u, 0u);
}

// BITS: bitmap from qmap.  COUNTS: prefix[w][key] = number of set bits of the key in words < w; count[key] = total.  A workgroup takes 64
// keys; its 16 waves turn and count a part of the queries each, 64 at a time, then write the prefixes of that part.  Others clear marks,
// and a last one makes the work list, if there is one.  Both at once where
// qmap does not lie in the prefixes' place.  An XCD has a run of keys, and so its L2 the 128-byte lines of qmap that 16 workgroups share.
template <bool BITS, bool COUNTS>
static __global__ __launch_bounds__(1024) void key_bits_kernel(const unsigned* qmap, int cnt, int Skv, int Wk, unsigned* bitmap,
                                                               unsigned* prefix, int* __restrict__ count, int W, int per_xcd, WorkList list, Marks marks) {
  __shared__ int part[16][64];
  const int beside = (int)blockIdx.x - 8 * per_xcd, kb = ((int)blockIdx.x & 7) * per_xcd + ((int)blockIdx.x >> 3);
  if (beside >= 0) {
    if (beside < marks.blocks) clear_marks(marks, beside);
    else make_work_list(list);
    return;
  }
  if (64 * kb >= Skv) return;
  const int lane = threadIdx.x & 63, seg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int key = kb * 64 + lane, kw = 2 * kb;
  const bool live = key < Skv;
  unsigned* bits = bitmap + min(key, Skv - 1);
  const int pairs = (W + 1) / 2, per = (pairs + 15) / 16;
  const int p0 = min(seg * per, pairs), p1 = min(p0 + per, pairs), w1 = min(2 * p1, W);
  unsigned lo[4], hi[4];
  int n = 0;
  if (BITS) {
    for (int p = p0; p < p1; p += 4) {
      const unsigned* src = qmap + (size_t)(64 * p + lane) * Wk + kw;
      const int left = cnt - 64 * p - lane;             // queries from the lane's first on
      if (Wk & 1) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const bool in = p + i < p1 && 64 * i < left;
          lo[i] = in ? src[(size_t)64 * i * Wk] : 0u;
          hi[i] = in && kw + 1 < Wk ? src[(size_t)64 * i * Wk + 1] : 0u;
        }
      } else {
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const uint2 v = p + i < p1 && 64 * i < left ? *(const uint2*)(src + (size_t)64 * i * Wk) : make_uint2(0u, 0u);
          lo[i] = v.x;
          hi[i] = v.y;
        }
      }
#pragma unroll
      for (int i = 0; i < 4; i++) {
        if (p + i >= p1) break;
        transpose64(lo[i], hi[i], lane);
        const int w = 2 * (p + i);
        if (live) {
          bits[(size_t)w * Skv] = lo[i];
          if (w + 1 < W) bits[(size_t)(w + 1) * Skv] = hi[i];        // (else of queries beyond the last: none)
        }
        n += __popc(lo[i]) + __popc(hi[i]);
      }
    }
  } else {
#pragma unroll 8
    for (int w = 2 * p0; w < w1; w++) n += __popc(bits[(size_t)w * Skv]);
  }
  if (!COUNTS) return;
  part[seg][lane] = n;
  __syncthreads();
  int run = 0;
  for (int s = 0; s < seg; s++) run += part[s][lane];
  if (!live) return;
  if (BITS && per <= 4) {                               // (all in registers)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int w = 2 * (p0 + i);
      if (w >= w1) break;
      prefix[(size_t)w * Skv + key] = (unsigned)run;
      run += __popc(lo[i]);
      if (w + 1 < w1) prefix[(size_t)(w + 1) * Skv + key] = (unsigned)run;
      run += __popc(hi[i]);
    }
  } else {
    for (int w0 = 2 * p0; w0 < w1; w0 += 8) {
      unsigned b[8];
#pragma unroll
      for (int i = 0; i < 8; i++) b[i] = bits[(size_t)min(w0 + i, w1 - 1) * Skv];
#pragma unroll
      for (int i = 0; i < 8; i++) {
        if (w0 + i >= w1) break;
        prefix[(size_t)(w0 + i) * Skv + key] = (unsigned)run;
        run += __popc(b[i]);
      }
    }
  }
  if (seg == 15) count[key] = run;
}

// Keys whose bits and first rows the last kernel holds in LDS at a time
constexpr int RANK_KEYS = 16384;
// dst[ql][slot] = row of the pair in key-sorted order (-1 for invalid slots).  A workgroup takes the 32 queries of a word, or
// a part of them (blockIdx.y) where there are few words, and has the word's bits and first rows of `range` keys at a time in
// LDS, where the lookups by id go: from memory they were two dependent random reads of 4 bytes per pair (8192 queries x 2048 slots
// 0.165 ms; 32768 x 2048 1.29 ms).  With `units` the ids are the lists of qmap_unit_kernel, and the pairs of a unit are its first
// query's; workgroups behind the others clear marks.
// start[key], the exclusive prefix sums of count, every workgroup works out for itself under the loads of the bits (two barriers a range)
// and one writes: in a kernel of its own between this one and the counts it was a launch of one workgroup.
static __global__ __launch_bounds__(1024) void rank_kernel(const int* __restrict__ ids, int row0, int q0, int cnt, int K, int Skv, int q_start,
                                                           const unsigned* __restrict__ bitmap, const unsigned* __restrict__ prefix,
                                                           const int* __restrict__ count, int* __restrict__ start, int range,
                                                           int* __restrict__ dst, int words, const int* __restrict__ units, int G, Marks marks) {
  extern __shared__ uint2 tab[];             // {first row of the word's queries, bits}
  constexpr int ROUNDS = RANK_KEYS / 1024;
  __shared__ int sums[16 * ROUNDS + 1];      // counts of 64 keys, then of all keys before them; of all keys up to the range's end
  const int w = blockIdx.x;
  if (w >= words) { clear_marks(marks, (w - words) * (int)gridDim.y + (int)blockIdx.y); return; }
  const bool writes = w == 0 && blockIdx.y == 0;
  const int share = 32 / gridDim.y;
  const int q_lo = 32 * w + blockIdx.y * share, q_hi = min(q_lo + share, cnt);
  const int sub = threadIdx.x >> 8, lane = threadIdx.x & 255;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wl = threadIdx.x & 63;
  int before = 0;                            // pairs of the ranges before
  for (int k0 = 0; k0 < Skv; k0 += range) {
    const int nk = min(range, Skv - k0), rounds = (nk + 1023) / 1024;
    if (k0) __syncthreads();
    for (int r0 = 0; r0 < rounds; r0 += 4) {
      int c[4], inc[4];
      uint2 e[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int k = min(1024 * (r0 + i) + (int)threadIdx.x, nk - 1);
        c[i] = count[k0 + k];
        e[i] = make_uint2(prefix[(size_t)w * Skv + k0 + k], bitmap[(size_t)w * Skv + k0 + k]);
      }
#pragma unroll
      for (int i = 0; i < 4; i++) {
        c[i] = 1024 * (r0 + i) + (int)threadIdx.x < nk ? c[i] : 0;
        inc[i] = wave_sums(c[i]);
      }
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int k = 1024 * (r0 + i) + threadIdx.x;
        if (k < nk) tab[k] = make_uint2(e[i].x + (unsigned)(inc[i] - c[i]), e[i].y);
        if (wl == 63 && r0 + i < rounds) sums[16 * (r0 + i) + wave] = inc[i];
      }
    }
    __syncthreads();
    if (wave == 0) {
      int c[4], all = 0;
#pragma unroll
      for (int i = 0; i < 4; i++) { c[i] = 4 * wl + i < 16 * rounds ? sums[4 * wl + i] : 0; all += c[i]; }
      int sum = before + wave_sums(all) - all;
#pragma unroll
      for (int i = 0; i < 4; i++) { if (4 * wl + i < 16 * rounds) sums[4 * wl + i] = sum; sum += c[i]; }
      if (wl == 63) sums[16 * ROUNDS] = sum;
    }
    static_assert(16 * ROUNDS == 4 * 64, "one wave has the sums of a range");
    __syncthreads();
    before = sums[16 * ROUNDS];
    if (writes)                              // (the first word has no queries before it)
      for (int k = threadIdx.x; k < nk; k += 1024) start[k0 + k] = (int)tab[k].x + sums[k >> 6];
    for (int ql = q_lo + sub; ql < q_hi; ql += 4) {
      const int owner = units && units[ql / G] ? ql / G * G : ql;
      const unsigned below = (1u << (owner & 31)) - 1u;
      const int last = units ? Skv - 1 : min(Skv - 1, q_start + q0 + ql);
      const int* row = ids + (size_t)(row0 + ql) * K;       // row0: row of local query 0 in the id array handed in
      for (int t0 = lane; t0 < K; t0 += 8 * 256) {
        int v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = t0 + i * 256 < K ? row[t0 + i * 256] : -1;
#pragma unroll
        for (int i = 0; i < 8; i++) {
          if (t0 + i * 256 >= K) break;
          const int id = units && v[i] >= 0 ? v[i] & 0xffffff : v[i];
          const bool ok = id >= 0 && id <= last;
          const int k = id - k0;
          if (ok && k >= 0 && k < nk) {
            const uint2 e = tab[k];
            dst[(size_t)ql * K + t0 + i * 256] = (int)e.x + sums[k >> 6] + __popc(e.y & below);
          } else if (!ok && k0 == 0) {
            dst[(size_t)ql * K + t0 + i * 256] = -1;
          }
        }
      }
    }
  }
  if (writes && threadIdx.x == 0) start[Skv] = before;
}

// Launches the kernels above for queries [q0, q0 + cnt).  A slot counts when its id v is in
// [0, Skv) and v <= q_start + (query index); pass a huge q_start to accept every id in range.
// With `sorted` ([cnt][K] ints) the first kernel also writes every query's valid ids in ascending
// order (-1 after them) and dst refers to the slots of that list: a caller that is free to choose
// its slot order uses the list instead of ids, which makes concurrently running queries gather
// neighbouring key rows at the same time (the rows then hit in the L2 of the XCD).
// qmap (cnt * ceil(Skv / 32) words) lies in `room`, memory of the caller that is free until the order is made, where that is large enough:
// then one kernel makes the bitmap and counts.  Else it lies in the prefix buffer, which the prefixes are written over afterwards: size that
// with prefix_words().
struct Room { void* at; size_t bytes; };
inline unsigned* qmap_place(const Room& room, unsigned* prefix, int cnt, int Wk) {
  return (size_t)cnt * Wk * 4 <= room.bytes ? (unsigned*)room.at : prefix;
}
inline size_t prefix_words(int chunk, int Skv) {
  const size_t W = (size_t)(chunk + 31) / 32, Wk = (size_t)(Skv + 31) / 32;
  return (size_t)Skv * W > (size_t)chunk * Wk ? (size_t)Skv * W : (size_t)chunk * Wk;
}
// The first kernel keeps one bit per key in LDS: the largest key count the builder takes
constexpr int MAX_KEYS = 150 * 1024 * 8;
// LDS of the first kernel with the sorted list: bitmap and prefix counts over all keys plus the list
inline bool sorted_list_fits(int Skv, int K) {
  return (size_t)((Skv + 31) / 32) * 8 + (size_t)K * 4 <= (size_t)150 * 1024;
}
// dup_flag: one int the caller has cleared (clear_flag) before the first block of queries of a call.
inline void clear_flag(int* dup_flag, hipStream_t st) { zero_u32_kernel<<<dim3(1), dim3(64), 0, st>>>((unsigned*)dup_flag, 1); }
inline void build_ranks(const int* lists, int row0, int q0, int cnt, int K, int Skv, int q_start, const unsigned* qmap, unsigned* bitmap,
                        unsigned* prefix, int* count, int* start, int* dst, int W, WorkList list, hipStream_t st, const int* flags = nullptr,
                        uint4* marks = nullptr, size_t n_marks = 0) {
  // Two kernels; they are short, so their number and the trips to memory in each are what they cost.  us in kernels as four (bits, counts,
  // one workgroup's scan, rows) / as two, a launch each besides: 2077 queries x 512 slots in pairs 26.3 / 21.5, 3072 x 640 32.1 / 23.9, 8192 x 2048
  // by themselves 72 / 52.  (The work list, in one pass over the groups instead of three, beside the counts or the rows: the same.)
  const int Wk = (Skv + 31) / 32, per_xcd = ((Skv + 63) / 64 + 7) / 8;
  // every word of the bitmap is written (zeros beyond the last query), so no clearing pass is needed
  const int words = (cnt + 31) / 32, parts = words >= 256 ? 1 : words >= 128 ? 2 : words >= 64 ? 4 : 8;
  const size_t half = n_marks / 2, rest = n_marks - half, each = (rest + 4095) / 4096 < 256 ? (rest + 4095) / 4096 : 256;
  const Marks first{flags, marks, half, (int)each}, second{flags, marks + half, rest, (int)(each + parts - 1) / parts * parts};
  if (qmap != prefix) {
    key_bits_kernel<true, true><<<dim3(8 * per_xcd + first.blocks + (list.units ? 1 : 0)), dim3(1024), 0, st>>>(qmap, cnt, Skv, Wk, bitmap, prefix, count, W, per_xcd, list, first);
  } else {
    key_bits_kernel<true, false><<<dim3(8 * per_xcd), dim3(1024), 0, st>>>(qmap, cnt, Skv, Wk, bitmap, prefix, count, W, per_xcd, list, first);
    key_bits_kernel<false, true><<<dim3(8 * per_xcd + first.blocks + (list.units ? 1 : 0)), dim3(1024), 0, st>>>(qmap, cnt, Skv, Wk, bitmap, prefix, count, W, per_xcd, list, first);
  }
  const int range = Skv < RANK_KEYS ? Skv : RANK_KEYS;
  if (range * 8 > 48 * 1024) (void)dsa_reserve_lds((const void*)rank_kernel, (size_t)range * 8);
  rank_kernel<<<dim3(words + second.blocks / parts, parts), dim3(1024), (size_t)range * 8, st>>>(
      lists, row0, q0, cnt, K, Skv, q_start, bitmap, prefix, count, start, range, dst, words, list.units, list.G, second);
}
inline void build(const int* ids, int q0, int cnt, int K, int Skv, int q_start, unsigned* bitmap, unsigned* prefix,
                  int* count, int* start, int* dst, int W, Room room, hipStream_t st, int* dup_flag, int* sorted = nullptr) {
  const int Wk = (Skv + 31) / 32;
  const size_t lds = (size_t)Wk * 4 * (sorted ? 2 : 1) + (sorted ? (size_t)K * 4 : 0);
  if (lds > 48 * 1024) (void)dsa_reserve_lds((const void*)qmap_kernel, lds);
  unsigned* qmap = qmap_place(room, prefix, cnt, Wk);
  qmap_kernel<<<dim3(cnt), dim3(256), lds, st>>>(ids, q0, cnt, K, Skv, q_start, qmap, Wk, sorted, dup_flag);
  // with `sorted` (rows of the block's queries, [cnt][K]) the ranks are those of the sorted slots
  build_ranks(sorted ? sorted : ids, sorted ? 0 : q0, q0, cnt, K, Skv, q_start, qmap, bitmap, prefix, count, start, dst, W, WorkList{nullptr, cnt, 1, nullptr}, st);
}
// LDS of qmap_unit_kernel
inline size_t unit_lists_lds(int G, int Skv, int K) { return (size_t)unit_words((Skv + 31) / 32) * 4 * (G + G / 2) + (size_t)G * K * 4; }
// build with the sorted lists, for groups of G (2 or 4) queries that may be units; 16 bytes of `marks` for every row (cnt K at most) are
// cleared if there are any.  work: cnt + 2 ints
inline void build_units(const int* ids, int q0, int cnt, int K, int Skv, int q_start, unsigned* bitmap, unsigned* prefix, int* count, int* start,
                        int* dst, int W, Room room, hipStream_t st, int* dup_flag, int* sorted, int G, const unsigned* bad, int* units, int max_slots,
                        UnitCost cost, uint4* marks, int* work) {
  const int Wk = (Skv + 31) / 32;
  const size_t lds = unit_lists_lds(G, Skv, K);
  const bool small = G * K <= 2048 && Wk <= 1024;      // (one round of ids for 256 threads, and then twice the workgroups on a compute unit)
  auto kernel = G == 2 ? (small ? qmap_unit_kernel<2, 256> : qmap_unit_kernel<2, 512>) : small ? qmap_unit_kernel<4, 256> : qmap_unit_kernel<4, 512>;
  if (lds > 48 * 1024) (void)dsa_reserve_lds((const void*)kernel, lds);
  unsigned* qmap = qmap_place(room, prefix, cnt, Wk);
  kernel<<<dim3((cnt + G - 1) / G), dim3(small ? 256 : 512), lds, st>>>(ids, q0, cnt, K, Skv, q_start, qmap, Wk, sorted, dup_flag, bad, units, max_slots, cost);
  build_ranks(sorted, 0, q0, cnt, K, Skv, q_start, qmap, bitmap, prefix, count, start, dst, W, WorkList{units, cnt, G, work}, st, dup_flag, marks, (size_t)cnt * K);
}

}  // namespace order
