// KL loss of the indexer against the attention distribution, with its gradient, in one pass (gfx950).
//
// Per query row, over the K selected slots:
//   pred = softmax(score)        u = target + eps
//   loss_row = sum_t u_t (log u_t - log(pred_t + eps))                       (F.kl_div(log(pred + eps), u, "sum"))
//   grad_t   = d loss_row / d score_t = pred_t (sum_j w_j pred_j - w_t),     w_t = u_t / (pred_t + eps)
// One workgroup per row; the row's scores and targets stay in registers between the three reductions
// (maximum, normaliser, loss and sum_j w_j pred_j), so each array crosses HBM once and the gradient is
// written once.  A padded slot (score -inf, target 0) has pred = 0, contributes eps (log eps - log eps) = 0
// to the loss and gets gradient 0.  HBM-bound: 12 bytes per slot, 10 with targets in bf16, which are read as they are (3072 x 512: 7.8 us
// behind a pass of 6.1 that makes them 32 bits wide, 8.3 us by itself).
#include "dsa_common.h"

namespace {

constexpr int BLOCK = 256;

// sums (or maxima) over the workgroup; every thread gets the result.  `scratch` holds 8 floats.
__device__ __forceinline__ float block_max(float v, float* scratch) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, o > 8 ? __shfl_xor(v, o, 64) : xor16(v, o));
  __syncthreads();                                   // the previous reduction's reads are done
  if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
  __syncthreads();
  return fmaxf(fmaxf(scratch[0], scratch[1]), fmaxf(scratch[2], scratch[3]));
}
__device__ __forceinline__ void block_sum2(float& a, float& b, float* scratch) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) { a += o > 8 ? __shfl_xor(a, o, 64) : xor16(a, o); b += o > 8 ? __shfl_xor(b, o, 64) : xor16(b, o); }
  __syncthreads();
  if ((threadIdx.x & 63) == 0) { scratch[threadIdx.x >> 6] = a; scratch[4 + (threadIdx.x >> 6)] = b; }
  __syncthreads();
  a = (scratch[0] + scratch[1]) + (scratch[2] + scratch[3]);
  b = (scratch[4] + scratch[5]) + (scratch[6] + scratch[7]);
}

// Sums over the threads that share a row: a workgroup, or a wave by itself.
struct BlockRow {
  float* scratch;
  __device__ float max(float v) const { return block_max(v, scratch); }
  __device__ void sum2(float& a, float& b) const { block_sum2(a, b, scratch); }
};
struct WaveRow {
  __device__ float max(float v) const {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, o > 8 ? __shfl_xor(v, o, 64) : xor16(v, o));
    return v;
  }
  __device__ void sum2(float& a, float& b) const {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) { a += o > 8 ? __shfl_xor(a, o, 64) : xor16(a, o); b += o > 8 ? __shfl_xor(b, o, 64) : xor16(b, o); }
  }
};

// Sum of a thread's four or eight values in pairs, for a wave that has a row by itself to round no more than a workgroup's 256 threads
template <int N>
__device__ __forceinline__ float pairs_sum(const float (&v)[N]) {
  static_assert(N == 4 || N == 8);
  const float a = (v[0] + v[1]) + (v[2] + v[3]);
  if constexpr (N == 8) return a + ((v[4] + v[5]) + (v[6] + v[7]));
  return a;
}

// a target slot as it is or from bf16
__device__ __forceinline__ float slot(float x) { return x; }
__device__ __forceinline__ float slot(unsigned short x) { return bf16_bits_to_f32(x); }

// thread tid of the NT that share a row has its slots tid, tid + NT, ..: K <= NE * NT
template <int NE, int NT, class T, class Row>
__device__ __forceinline__ void kl_row(const Row& over, int tid, int64_t row, const float* __restrict__ scores, int64_t ld_s,
                                       const T* __restrict__ target, int64_t ld_t, int K, float eps, float factor, float* __restrict__ row_loss,
                                       float* __restrict__ grad) {
  const float* sp = scores + row * ld_s;
  const T* tp = target + row * ld_t;
  float s[NE], u[NE];
  T raw[NE];
  float mx = -INFINITY;
  // No lane's branch between the loads, and nothing that waits for one of them.  (Loads beyond the row are left out by a branch of the whole
  // wave with targets in fp32: 8192 rows of 2500 slots 95.5 -> 93.4 us, 3000 40.4 -> 39.6.  In bf16 each would be waited for: 97 and 100.6, 2000
  // rows of 8192 33.7 and 45.)
#pragma unroll
  for (int i = 0; i < NE; i++) {
    s[i] = 0.f;
    raw[i] = T(0);
    if (NE > 8 && sizeof(T) == 4 && NT * i >= K) continue;
    const int t = min(tid + NT * i, K - 1);
    s[i] = sp[t];
    raw[i] = tp[t];
  }
#pragma unroll
  for (int i = 0; i < NE; i++) {
    const int t = tid + NT * i;
    s[i] = t < K ? s[i] : -INFINITY;
    u[i] = (t < K ? slot(raw[i]) : 0.f) + eps;
    mx = fmaxf(mx, s[i]);
  }
  mx = over.max(mx);
  constexpr bool WAVE = NT == 64;
  float z = 0.f, unused = 0.f;
#pragma unroll
  for (int i = 0; i < NE; i++) {                                          // a row of -inf only: NaN, as torch.softmax
    s[i] = expf(s[i] - mx);
    if (!WAVE) z += s[i];
  }
  if constexpr (WAVE) z = pairs_sum(s);
  over.sum2(z, unused);
  const float inv = 1.0f / z;
  float loss = 0.f, inner = 0.f, l[WAVE ? NE : 1], n[WAVE ? NE : 1];
#pragma unroll
  for (int i = 0; i < NE; i++) {
    const int t = tid + NT * i;
    const float p = s[i] * inv;
    const float w = u[i] / (p + eps);
    if constexpr (WAVE) {
      l[i] = t < K ? u[i] * (logf(u[i]) - logf(p + eps)) : 0.f;
      n[i] = t < K ? w * p : 0.f;
    } else if (t < K) {
      loss += u[i] * (logf(u[i]) - logf(p + eps));
      inner += w * p;
    }
    s[i] = p;
    u[i] = w;
  }
  if constexpr (WAVE) {
    loss = pairs_sum(l);
    inner = pairs_sum(n);
  }
  over.sum2(loss, inner);
#pragma unroll
  for (int i = 0; i < NE; i++) {
    const int t = tid + NT * i;
    if (t < K) grad[row * K + t] = (s[i] * (inner - u[i])) * factor;
  }
  if (tid == 0) row_loss[row] = loss;
}

template <int NE, class T>
__global__ __launch_bounds__(BLOCK) void kl_loss_kernel(const float* __restrict__ scores, int64_t ld_s,
                                                        const T* __restrict__ target, int64_t ld_t, int K, float eps, float factor,
                                                        float* __restrict__ row_loss, float* __restrict__ grad) {
  __shared__ float scratch[8];
  kl_row<NE, BLOCK>(BlockRow{scratch}, threadIdx.x, blockIdx.x, scores, ld_s, target, ld_t, K, eps, factor, row_loss, grad);
}

// Up to 512 slots: a row to a wave.  A workgroup to a row spent its time in three reductions with barriers and on eight slots a thread of
// which one or two were there (7951 x 256 slots 30.4 us and 7.6 so, 2077 x 512 11.3 and 6.1, 300 x 256 4.8 and 3.3; beyond, four
// slots a thread where that is enough: 4000 x 1024 18.8 and 13.8).
template <int NE, class T>
__global__ __launch_bounds__(BLOCK) void kl_loss_wave_kernel(const float* __restrict__ scores, int64_t ld_s, const T* __restrict__ target,
                                                             int64_t ld_t, int S, int K, float eps, float factor, float* __restrict__ row_loss,
                                                             float* __restrict__ grad) {
  const int row = __builtin_amdgcn_readfirstlane(blockIdx.x * (BLOCK / 64) + (threadIdx.x >> 6));
  if (row >= S) return;
  kl_row<NE, 64>(WaveRow{}, threadIdx.x & 63, row, scores, ld_s, target, ld_t, K, eps, factor, row_loss, grad);
}

// *out = factor * sum of the rows' losses, in a fixed order and 64 bits, so that the result is rounded and not the sums on the way.  One
// launch for the sum and the scaling behind it (5 us each).  Bound by its latency: 2.4 us at 1024 - 8192 rows, 3.7 at 32 768 (32-bit
// sums 2.0 and 2.6).  Relative error over 200 draws of 300 - 32 768 rows 2.8 - 3.5e-8; 32-bit sums 5.0 - 6.7e-8, torch's 4.2 - 5.7e-8.
__global__ __launch_bounds__(1024) void kl_total_kernel(const float* __restrict__ row_loss, int S, float factor, float* __restrict__ out) {
  __shared__ double part[16];
  double s = 0.0;
  for (int i0 = threadIdx.x; i0 < S; i0 += 8 * 1024) {
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = row_loss[min(i0 + 1024 * k, S - 1)];
#pragma unroll
    for (int k = 0; k < 8; k++) s += i0 + 1024 * k < S ? (double)v[k] : 0.0;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x != 0) return;
  s = 0.0;
#pragma unroll
  for (int i = 0; i < 16; i++) s += part[i];
  *out = (float)s * factor;
}

// y = x * (*g * factor): the loss's gradient carried on to the scores, bound by memory.
__global__ __launch_bounds__(256) void kl_scale_kernel(const f32x4* __restrict__ x, const float* __restrict__ g, float factor, f32x4* __restrict__ y, int64_t n) {
  const float f = *g * factor;
  const int64_t n4 = n / 4, i0 = (int64_t)blockIdx.x * 1024 + threadIdx.x;
  f32x4 v[4];
#pragma unroll
  for (int i = 0; i < 4; i++)
    if (i0 + 256 * i < n4) v[i] = x[i0 + 256 * i];
#pragma unroll
  for (int i = 0; i < 4; i++)
    if (i0 + 256 * i < n4) y[i0 + 256 * i] = v[i] * f;
  if (blockIdx.x == 0 && (int64_t)threadIdx.x < n % 4) ((float*)y)[4 * n4 + threadIdx.x] = ((const float*)x)[4 * n4 + threadIdx.x] * f;
}

template <class T>
void launch_rows(const float* scores, int64_t ld_s, const T* target, int64_t ld_t, int S, int K, float eps, float factor, float* row_loss, float* grad,
                 hipStream_t st) {
  const dim3 waves(dsa_cdiv(S, BLOCK / 64));
  if (K <= 256) kl_loss_wave_kernel<4, T><<<waves, dim3(BLOCK), 0, st>>>(scores, ld_s, target, ld_t, S, K, eps, factor, row_loss, grad);
  else if (K <= 512) kl_loss_wave_kernel<8, T><<<waves, dim3(BLOCK), 0, st>>>(scores, ld_s, target, ld_t, S, K, eps, factor, row_loss, grad);
  else if (K <= 4 * BLOCK) kl_loss_kernel<4, T><<<dim3(S), dim3(BLOCK), 0, st>>>(scores, ld_s, target, ld_t, K, eps, factor, row_loss, grad);
  else if (K <= 8 * BLOCK) kl_loss_kernel<8, T><<<dim3(S), dim3(BLOCK), 0, st>>>(scores, ld_s, target, ld_t, K, eps, factor, row_loss, grad);
  else kl_loss_kernel<32, T><<<dim3(S), dim3(BLOCK), 0, st>>>(scores, ld_s, target, ld_t, K, eps, factor, row_loss, grad);
}

}  // namespace

extern "C" int dsa_indexer_kl_total(const float* row_loss, int S, float factor, float* out, void* stream) {
  DSA_REQUIRE(S >= 0 && out != nullptr && (S == 0 || row_loss != nullptr), "dsa_indexer_kl_total: bad arguments");
  kl_total_kernel<<<dim3(1), dim3(1024), 0, (hipStream_t)stream>>>(row_loss, S, factor, out);
  DSA_CHECK_LAUNCH("dsa_indexer_kl_total");
  return DSA_OK;
}

extern "C" int dsa_indexer_kl_scale(const float* grad, const float* g, float factor, float* out, int64_t n, void* stream) {
  DSA_REQUIRE(n >= 0 && (n == 0 || (grad && g && out)), "dsa_indexer_kl_scale: bad arguments");
  DSA_REQUIRE(((uintptr_t)grad % 16) == 0 && ((uintptr_t)out % 16) == 0, "dsa_indexer_kl_scale: misaligned pointer");
  if (n == 0) return DSA_OK;
  const int64_t blocks = (n / 4 + 1024) / 1024;
  DSA_REQUIRE(blocks < (1ll << 31), "dsa_indexer_kl_scale: too many elements");
  kl_scale_kernel<<<dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream>>>((const f32x4*)grad, g, factor, (f32x4*)out, n);
  DSA_CHECK_LAUNCH("dsa_indexer_kl_scale");
  return DSA_OK;
}

extern "C" int dsa_indexer_kl_loss(const float* scores, int64_t ld_s, const float* target, int64_t ld_t, int S, int K,
                                   float eps, float* row_loss, float* grad, void* stream) {
  return dsa_indexer_kl_loss_scaled(scores, ld_s, target, 0, ld_t, S, K, eps, 1.0f, row_loss, grad, stream);
}

extern "C" int dsa_indexer_kl_loss_scaled(const float* scores, int64_t ld_s, const void* target, int target_bf16, int64_t ld_t, int S, int K,
                                          float eps, float factor, float* row_loss, float* grad, void* stream) {
  DSA_REQUIRE(S >= 0 && K > 0 && K <= 32 * BLOCK, "dsa_indexer_kl_loss: K must lie in [1, %d], got %d", 32 * BLOCK, K);
  DSA_REQUIRE(ld_s >= K && ld_t >= K, "dsa_indexer_kl_loss: row strides %lld / %lld below K = %d", (long long)ld_s,
              (long long)ld_t, K);
  if (S == 0) return DSA_OK;
  if (target_bf16) launch_rows(scores, ld_s, (const unsigned short*)target, ld_t, S, K, eps, factor, row_loss, grad, (hipStream_t)stream);
  else launch_rows(scores, ld_s, (const float*)target, ld_t, S, K, eps, factor, row_loss, grad, (hipStream_t)stream);
  DSA_CHECK_LAUNCH("dsa_indexer_kl_loss");
  return DSA_OK;
}
