// The integer work of packed sequences that more than one kernel does: which sequence a token belongs to, and the indexer's windows.
#pragma once
#include "dsa_common.h"

namespace {

// Index of the sequence that token t of the packed batch belongs to: the first one that ends behind t (ncu - 1 if none does).
template <typename T>
__device__ __forceinline__ int sequence_of(const T* cu, int ncu, long long t) {
  int lo = 0, hi = ncu - 1;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if ((long long)cu[mid + 1] > t) hi = mid; else lo = mid + 1;
  }
  return lo;
}

// The windows of queries 256 block .. 256 block + 255, one per thread of 256, and from the first block the summed length of the sequences (-1
// if the cumulative lengths decrease).  A query behind the last sequence has an empty window, not the keys of another sequence:
// nothing stops a captured launch.
template <typename T>
__device__ __forceinline__ void window_part(int block, const T* __restrict__ cu, int ncu, int S, int chunk_offset, int* __restrict__ ks,
                                            int* __restrict__ ke, int* __restrict__ total) {
  if (total && block == 0) {
    bool falls = false;
    for (int k = threadIdx.x; k + 1 < ncu; k += 256) falls |= cu[k + 1] < cu[k];
    falls = __syncthreads_or(falls);
    if (threadIdx.x == 0) *total = falls ? -1 : ncu > 0 ? (int)min((long long)cu[ncu - 1] - (long long)cu[0], 0x7fffffffll) : 0;
  }
  const int i = block * 256 + (int)threadIdx.x;
  if (i >= S) return;
  int start = 0, end = chunk_offset + i + 1;
  if (ncu > 0) {
    const int seq = sequence_of(cu, ncu, (long long)i + chunk_offset + (long long)cu[0]);   // lengths count from cu[0]
    if (seq < ncu - 1) start = (int)cu[seq];
    else end = 0;
  }
  ks[i] = start;
  ke[i] = end;
}

}  // namespace
