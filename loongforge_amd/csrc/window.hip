// Integer work around packed sequences: the indexer's windows and the rotary positions.  One thread per token, a binary
// search over the cumulative lengths (a few KB that stay in the caches).  Bound by its launch; it takes the place of 8 - 10
// small tensor operations, one of which made the host wait for the device.
#include "window.h"

namespace {

template <typename T>
__global__ __launch_bounds__(256) void window_kernel(const T* __restrict__ cu, int ncu, int S, int chunk_offset, int* __restrict__ ks,
                                                     int* __restrict__ ke, int* __restrict__ total) {
  window_part(blockIdx.x, cu, ncu, S, chunk_offset, ks, ke, total);
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
