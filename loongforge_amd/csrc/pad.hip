// Zero heads behind the real ones of every token: the attention kernels take heads in groups of 32.  One launch at the copy rate
// (1024 tokens x 16 heads x 576: 12 us) where a fill of the padded tensor and a strided copy into it took 20.
#include "dsa_common.h"

namespace {

constexpr int PER_THREAD = 3;              // 16-byte pieces: 32 rows of 576 or 512 elements are 9 or 8 times 256 of them

__global__ __launch_bounds__(256) void pad_heads_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst, int pieces_in, int pieces_out, int parts) {
  const long tok = blockIdx.x / parts;
  const int first = ((int)blockIdx.x % parts) * 256 * PER_THREAD + (int)threadIdx.x;
  uint4 v[PER_THREAD];
#pragma unroll
  for (int i = 0; i < PER_THREAD; i++) {
    const int p = first + 256 * i;
    v[i] = p < pieces_in ? src[tok * pieces_in + p] : make_uint4(0, 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < PER_THREAD; i++) {
    const int p = first + 256 * i;
    if (p < pieces_out) dst[tok * pieces_out + p] = v[i];
  }
}

}  // namespace

extern "C" int dsa_pad_heads(const void* src, int tokens, int heads, int heads_out, int row_bytes, void* dst, void* stream) {
  DSA_REQUIRE(tokens >= 0 && heads > 0 && heads <= heads_out && heads_out <= 1024 && row_bytes > 0 && row_bytes <= 65536 && row_bytes % 16 == 0,
              "dsa_pad_heads: bad sizes");
  DSA_REQUIRE(((uintptr_t)src % 16) == 0 && ((uintptr_t)dst % 16) == 0, "dsa_pad_heads: misaligned pointer");
  if (tokens == 0) return DSA_OK;
  const int pieces_in = heads * (row_bytes / 16), pieces_out = heads_out * (row_bytes / 16), parts = dsa_cdiv(pieces_out, 256 * PER_THREAD);
  DSA_REQUIRE((int64_t)tokens * parts < (1ll << 31), "dsa_pad_heads: too many tokens");
  pad_heads_kernel<<<dim3((unsigned)(tokens * parts)), dim3(256), 0, (hipStream_t)stream>>>((const uint4*)src, (uint4*)dst, pieces_in, pieces_out, parts);
  DSA_CHECK_LAUNCH("dsa_pad_heads");
  return DSA_OK;
}
