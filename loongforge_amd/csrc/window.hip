// Integer work around packed sequences: the indexer's windows and the rotary positions.  One thread per token, a binary
// search over the cumulative lengths (a few KB that stay in the caches).  Bound by its launch; it takes the place of 8 - 10
// small tensor operations, one of which made the host wait for the device.
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

// A query behind the last sequence has an empty window, not the keys of another sequence: nothing stops a captured launch.
template <typename T>
__global__ __launch_bounds__(256) void window_kernel(const T* __restrict__ cu, int ncu, int S, int chunk_offset, int* __restrict__ ks,
                                                     int* __restrict__ ke, int* __restrict__ total) {
  if (total && blockIdx.x == 0) {
    bool falls = false;
    for (int k = threadIdx.x; k + 1 < ncu; k += blockDim.x) falls |= cu[k + 1] < cu[k];
    falls = __syncthreads_or(falls);
    if (threadIdx.x == 0) *total = falls ? -1 : ncu > 0 ? (int)min((long long)cu[ncu - 1] - (long long)cu[0], 0x7fffffffll) : 0;
  }
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
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

template <typename T>
__global__ void positions_kernel(const T* __restrict__ cu, int ncu, int tokens, long long offset, int* __restrict__ pos) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= tokens) return;
  const long long t = i + offset;
  const int seq = sequence_of(cu, ncu, t);
  pos[i] = seq < ncu - 1 ? (int)(t - (long long)cu[seq]) : 0;
}

}  // namespace

extern "C" int dsa_indexer_window(const void* cu, int cu_i64, int ncu, int S, int chunk_offset, int32_t* ks, int32_t* ke, int32_t* total,
                                  void* stream) {
  DSA_REQUIRE(S >= 0 && ncu >= 0, "indexer_window: bad sizes");
  DSA_REQUIRE(cu != nullptr || ncu == 0, "indexer_window: null pointer");
  const dim3 grid(dsa_cdiv(S > 0 ? S : 1, 256));
  if (cu_i64) window_kernel<long long><<<grid, 256, 0, (hipStream_t)stream>>>((const long long*)cu, ncu, S, chunk_offset, ks, ke, total);
  else window_kernel<int><<<grid, 256, 0, (hipStream_t)stream>>>((const int*)cu, ncu, S, chunk_offset, ks, ke, total);
  DSA_CHECK_LAUNCH("indexer_window");
  return DSA_OK;
}

extern "C" int dsa_thd_positions(const void* cu, int cu_i64, int ncu, int tokens, int64_t offset, int32_t* positions, void* stream) {
  DSA_REQUIRE(tokens >= 0 && ncu >= 1 && cu != nullptr, "thd_positions: bad sizes");
  if (tokens == 0) return DSA_OK;
  const dim3 grid(dsa_cdiv(tokens, 256));
  if (cu_i64) positions_kernel<long long><<<grid, 256, 0, (hipStream_t)stream>>>((const long long*)cu, ncu, tokens, offset, positions);
  else positions_kernel<int><<<grid, 256, 0, (hipStream_t)stream>>>((const int*)cu, ncu, tokens, offset, positions);
  DSA_CHECK_LAUNCH("thd_positions");
  return DSA_OK;
}
