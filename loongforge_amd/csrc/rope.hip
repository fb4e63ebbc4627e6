// Rotary position embedding for the MLA query / key rows around the sparse attention kernels,
// fused with the copies (layout permutation, concatenation) that surround it.  HBM-bound
// elementwise work: every row is read once and written once in 16-byte pieces.
//
// One kernel covers the whole family.  Per (token, head) it
//   * copies a "main" part of d_main elements from one strided tensor to another, and
//   * rotates a "pe" part of emb_dim elements: pair i is (x1_i, x2_i) with
//         y1_i = x1_i * c1_i - x2_i * s1_i          y2_i = x2_i * c2_i + x1_i * s2_i      (forward)
//         y1_i = x1_i * c1_i + x2_i * s2_i          y2_i = x2_i * c2_i - x1_i * s1_i      (inverse: the transpose)
//     in fp32 without fused multiply-adds, rounded once to bf16.
// Where the pair sits in a row is the "pairing": adjacent (elements 2i, 2i+1) or split
// (elements i, i + emb_dim/2); source and destination pairings are independent, and the cos / sin
// rows are indexed with the pairing of the rotated side (destination in the forward direction,
// source in the inverse one): c1_i = cos[2i], c2_i = cos[2i+1] or c1_i = cos[i], c2_i = cos[i + emb_dim/2].
#include "rope_quad.h"

namespace {

using namespace rope;

struct RopeArgs {
  const unsigned short* main_src; long ms_tok, ms_head;     // strides in elements; nullptr: no main part
  unsigned short* main_dst; long md_tok, md_head;
  int d_main;
  const unsigned short* pe_src; long ps_tok, ps_head;
  unsigned short* pe_dst; long pd_tok, pd_head;
  int emb;
  const void* cos; const void* sin; int cs_f32;             // [positions][emb], fp32 or bf16
  const int* positions; int batch;                          // position of a token: positions[t] or t / batch
  int tokens, heads;
};

template <int IN, int OUT, bool INVERSE>
__global__ __launch_bounds__(256) void rope_rows_kernel(RopeArgs a) {
  const int main_chunks = a.main_src ? a.d_main >> 3 : 0;
  const int quads = a.emb >> 3;                       // groups of four pairs
  const int per_head = main_chunks + quads;
  const int items = a.heads * per_head;
  for (long tok = blockIdx.x; tok < a.tokens; tok += gridDim.x) {
    const long pos = a.emb == 0 ? 0 : (a.positions ? a.positions[tok] : tok / a.batch);
    for (int it = threadIdx.x; it < items; it += 256) {
      const int head = it / per_head, c = it - head * per_head;
      if (c < main_chunks) {
        const uint4 v = *(const uint4*)(a.main_src + tok * a.ms_tok + head * a.ms_head + 8 * c);
        *(uint4*)(a.main_dst + tok * a.md_tok + head * a.md_head + 8 * c) = v;
        continue;
      }
      const int q = c - main_chunks;
      const unsigned short* src = a.pe_src + tok * a.ps_tok + head * a.ps_head;
      unsigned short* dst = a.pe_dst + tok * a.pd_tok + head * a.pd_head;
      rotate_quad<IN, OUT, INVERSE>(src, dst, q, a.emb, pos, a.cos, a.sin, a.cs_f32);
    }
  }
}

// The same for the rows of the absorbed MLA layouts, 512 main and 64 rotary elements.  Bound by memory: 4 B per element.  The
// kernel above has one 16-byte load per thread in flight behind an integer division, 3.2 TB/s; here a workgroup takes a tile
// of 32 rows, 2^tok_log2 tokens by the rest in heads, and a wave eight of them: the 64 lanes move a 1 KB main part per
// instruction and the eight rotary parts in one, all loads requested before the first store.  us, HSD -> SHD / back:
// 4096 tokens x 128 heads 379 / 383 -> 216 / 228 (5.6 TB/s), 700 x 128 63 / 62 -> 30 / 30, 8192 x 32 183 / 177 -> 108 / 109,
// 60 x 128 33 / 33 -> 4.7 / 5.1.  Tiles of 1, 2, 4 or 8 tokens measured within 2 %, of 32 tokens 5 % slower.
constexpr int MLA_MAIN = 512, MLA_EMB = 64, TILE_ROWS = 32, TOK_LOG2 = 1;
// Where the rows read and written exceed the memory-side cache, loads and stores of the main parts are non-temporal (STREAMED): both parts
// are whole lines, used once.  us, forward and backward of query and key: 4096 tokens x 128 heads 469 with plain ones, 462 with such loads,
// 446 with such stores, 420 with both (5.8 TB/s); 8192 x 64 466 -> 431, 1500 x 128 190 -> 167, 2600 x 64 167 -> 140 - 156.  Below that size
// the data may still be there from the kernel that wrote it, or for the one that reads it (700 x 128, forward: 34 against 30 us with such
// loads).  It is a template's argument because of a choice at run time the compiler makes one plain load or store.
constexpr long CACHE_BYTES = 256l << 20;
template <int IN, int OUT, bool INVERSE, bool STREAMED>
__global__ __launch_bounds__(256) void rope_mla_rows_kernel(RopeArgs a, int tok_log2, int head_tiles) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tok0 = ((int)blockIdx.x / head_tiles) << tok_log2;
  const int head0 = ((int)blockIdx.x % head_tiles) * (TILE_ROWS >> tok_log2);
  auto token = [&](int row) { return tok0 + (row & ((1 << tok_log2) - 1)); };
  auto head = [&](int row) { return head0 + (row >> tok_log2); };
  // rows beyond the end are read as the last one and not written
  auto at = [&](const unsigned short* base, long per_tok, long per_head, int row) {
    return base + min(token(row), a.tokens - 1) * per_tok + min(head(row), a.heads - 1) * per_head;
  };
  auto there = [&](int row) { return token(row) < a.tokens && head(row) < a.heads; };
  const int pe_row = wave * 8 + (lane >> 3), q = lane & 7;
  const int t = min(token(pe_row), a.tokens - 1);
  const long pos = a.positions ? a.positions[t] : t / a.batch;
  i32x4 v[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const i32x4* src = (const i32x4*)at(a.main_src, a.ms_tok, a.ms_head, wave * 8 + i) + lane;
    if constexpr (STREAMED) v[i] = __builtin_nontemporal_load(src);
    else v[i] = *src;
  }
  const Quad x = load_quad<IN>(at(a.pe_src, a.ps_tok, a.ps_head, pe_row), q, MLA_EMB);
  const QuadTables tables = load_tables<INVERSE ? IN : OUT>(a.cos, a.sin, a.cs_f32, pos, q, MLA_EMB);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 8; i++)
    if (there(wave * 8 + i)) {
      i32x4* dst = (i32x4*)(a.main_dst + (long)token(wave * 8 + i) * a.md_tok + (long)head(wave * 8 + i) * a.md_head) + lane;
      if constexpr (STREAMED) __builtin_nontemporal_store(v[i], dst);
      else *dst = v[i];
    }
  if (there(pe_row))
    store_quad<OUT>(rotate<INVERSE>(x, tables), a.pe_dst + (long)token(pe_row) * a.pd_tok + (long)head(pe_row) * a.pd_head, q, MLA_EMB);
}

// Gradient of a pe row that the forward broadcast to every head: the head-sum of the incoming
// gradient (fp32, heads added in ascending order within 256 / emb_dim interleaved groups, the groups
// then in order), rounded to bf16, then the inverse rotation; written with adjacent pairing.
template <int IN>
__global__ __launch_bounds__(256) void rope_headsum_inverse_kernel(
    const unsigned short* __restrict__ g, long g_tok, long g_head, unsigned short* __restrict__ d_emb, long de_tok,
    int emb, const void* cos, const void* sin, int cs_f32, const int* __restrict__ positions, int batch,
    int tokens, int heads) {
#pragma clang fp contract(off)
  __shared__ float part[256];
  __shared__ float tot[256];
  const int half = emb >> 1;
  const int groups = 256 / emb;
  const int e = threadIdx.x % emb, grp = threadIdx.x / emb;
  for (long tok = blockIdx.x; tok < tokens; tok += gridDim.x) {
    const long pos = positions ? positions[tok] : tok / batch;
    float s = 0.f;
    if (grp < groups)
      for (int h = grp; h < heads; h += groups) s += bf16_bits_to_f32(g[tok * g_tok + h * g_head + e]);
    part[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x < emb) {
      float t = 0.f;
      for (int k = 0; k < groups; k++) t += part[k * emb + e];
      tot[e] = bf16_bits_to_f32(f32_to_bf16_bits(t));
    }
    __syncthreads();
    if (threadIdx.x < half) {
      const int i = threadIdx.x;
      const int i1 = IN == ADJ ? 2 * i : i, i2 = IN == ADJ ? 2 * i + 1 : i + half;
      const float x1 = tot[i1], x2 = tot[i2];
      float c1, c2, s1, s2;
      const long crow = pos * emb;
      if (cs_f32) {
        c1 = ((const float*)cos)[crow + i1]; c2 = ((const float*)cos)[crow + i2];
        s1 = ((const float*)sin)[crow + i1]; s2 = ((const float*)sin)[crow + i2];
      } else {
        c1 = bf16_bits_to_f32(((const unsigned short*)cos)[crow + i1]); c2 = bf16_bits_to_f32(((const unsigned short*)cos)[crow + i2]);
        s1 = bf16_bits_to_f32(((const unsigned short*)sin)[crow + i1]); s2 = bf16_bits_to_f32(((const unsigned short*)sin)[crow + i2]);
      }
      const float y1 = x1 * c1 + x2 * s2;
      const float y2 = (-x1) * s1 + x2 * c2;
      *(unsigned*)(d_emb + tok * de_tok + 2 * i) = pack_bf16x2(y1, y2);
    }
    __syncthreads();
  }
}

bool aligned16(const void* p) { return ((uintptr_t)p % 16) == 0; }
bool aligned8(const void* p) { return ((uintptr_t)p % 8) == 0; }

}  // namespace

extern "C" int dsa_rope_rows(const void* main_src, int64_t ms_tok, int64_t ms_head, void* main_dst, int64_t md_tok,
                             int64_t md_head, int d_main, const void* pe_src, int64_t ps_tok, int64_t ps_head,
                             void* pe_dst, int64_t pd_tok, int64_t pd_head, int emb_dim, const void* cos,
                             const void* sin, int cos_sin_f32, const int32_t* positions, int batch, int tokens,
                             int heads, int in_pairing, int out_pairing, int inverse, void* stream) {
  DSA_REQUIRE(tokens >= 0 && heads > 0, "dsa_rope_rows: bad sizes tokens=%d heads=%d", tokens, heads);
  DSA_REQUIRE(emb_dim >= 0 && emb_dim % 8 == 0, "dsa_rope_rows: emb_dim must be a multiple of 8, got %d", emb_dim);
  DSA_REQUIRE(emb_dim > 0 || main_src != nullptr, "dsa_rope_rows: nothing to do (no main part and emb_dim = 0)");
  DSA_REQUIRE((in_pairing == 0 || in_pairing == 1) && (out_pairing == 0 || out_pairing == 1),
              "dsa_rope_rows: pairing must be 0 (adjacent) or 1 (split)");
  DSA_REQUIRE(emb_dim == 0 || (pe_src && pe_dst && cos && sin), "dsa_rope_rows: null pointer");
  DSA_REQUIRE(emb_dim == 0 || positions != nullptr || batch > 0, "dsa_rope_rows: batch must be positive when no positions are given");
  DSA_REQUIRE(emb_dim == 0 || aligned16(pe_src) && aligned16(pe_dst) && aligned16(cos) && aligned16(sin) && ps_tok % 8 == 0 &&
              ps_head % 8 == 0 && pd_tok % 8 == 0 && pd_head % 8 == 0,
              "dsa_rope_rows: pe rows must start on 16-byte boundaries");
  if (main_src) {
    DSA_REQUIRE(main_dst != nullptr && d_main > 0 && d_main % 8 == 0, "dsa_rope_rows: d_main must be a positive multiple of 8, got %d", d_main);
    DSA_REQUIRE(aligned16(main_src) && aligned16(main_dst) && ms_tok % 8 == 0 && ms_head % 8 == 0 && md_tok % 8 == 0 &&
                md_head % 8 == 0, "dsa_rope_rows: main rows must start on 16-byte boundaries");
  }
  if (tokens == 0) return DSA_OK;
  RopeArgs a;
  a.main_src = (const unsigned short*)main_src; a.ms_tok = ms_tok; a.ms_head = ms_head;
  a.main_dst = (unsigned short*)main_dst; a.md_tok = md_tok; a.md_head = md_head; a.d_main = d_main;
  a.pe_src = (const unsigned short*)pe_src; a.ps_tok = ps_tok; a.ps_head = ps_head;
  a.pe_dst = (unsigned short*)pe_dst; a.pd_tok = pd_tok; a.pd_head = pd_head; a.emb = emb_dim;
  a.cos = cos; a.sin = sin; a.cs_f32 = cos_sin_f32; a.positions = positions; a.batch = batch;
  a.tokens = tokens; a.heads = heads;
  hipStream_t st = (hipStream_t)stream;
  const dim3 block(256);
  const int sel = (in_pairing << 2) | (out_pairing << 1) | (inverse ? 1 : 0);
  int tok_log2 = TOK_LOG2;
  while (tok_log2 < 5 && heads <= (TILE_ROWS >> (tok_log2 + 1))) tok_log2++;
  const int head_tiles = dsa_cdiv(heads, TILE_ROWS >> tok_log2);
  const long tiles = (long)dsa_cdiv(tokens, 1 << tok_log2) * head_tiles;
  const bool mla = main_src && d_main == MLA_MAIN && emb_dim == MLA_EMB && tiles < (1 << 24);
  const bool streamed = (long)tokens * heads * (MLA_MAIN + MLA_EMB) * 4 > CACHE_BYTES;
  const dim3 grid(mla ? (unsigned)tiles : tokens < (1 << 20) ? tokens : (1 << 20));
#define DSA_ROPE(IN, OUT, INV) do { \
    if (mla && streamed) rope_mla_rows_kernel<IN, OUT, INV, true><<<grid, block, 0, st>>>(a, tok_log2, head_tiles); \
    else if (mla) rope_mla_rows_kernel<IN, OUT, INV, false><<<grid, block, 0, st>>>(a, tok_log2, head_tiles); \
    else rope_rows_kernel<IN, OUT, INV><<<grid, block, 0, st>>>(a); \
  } while (0)
  switch (sel) {
    case 0: DSA_ROPE(ADJ, ADJ, false); break;
    case 1: DSA_ROPE(ADJ, ADJ, true); break;
    case 2: DSA_ROPE(ADJ, SPLIT, false); break;
    case 3: DSA_ROPE(ADJ, SPLIT, true); break;
    case 4: DSA_ROPE(SPLIT, ADJ, false); break;
    case 5: DSA_ROPE(SPLIT, ADJ, true); break;
    case 6: DSA_ROPE(SPLIT, SPLIT, false); break;
    default: DSA_ROPE(SPLIT, SPLIT, true); break;
  }
#undef DSA_ROPE
  DSA_CHECK_LAUNCH("dsa_rope_rows");
  return DSA_OK;
}

extern "C" int dsa_rope_headsum_inverse(const void* grad, int64_t g_tok, int64_t g_head, void* d_emb, int64_t de_tok,
                                        int emb_dim, const void* cos, const void* sin, int cos_sin_f32,
                                        const int32_t* positions, int batch, int tokens, int heads, int in_pairing,
                                        void* stream) {
  DSA_REQUIRE(tokens >= 0 && heads > 0, "dsa_rope_headsum_inverse: bad sizes tokens=%d heads=%d", tokens, heads);
  DSA_REQUIRE(emb_dim >= 2 && emb_dim <= 256 && (emb_dim & (emb_dim - 1)) == 0,
              "dsa_rope_headsum_inverse: emb_dim must be a power of two up to 256, got %d", emb_dim);
  DSA_REQUIRE(in_pairing == 0 || in_pairing == 1, "dsa_rope_headsum_inverse: pairing must be 0 (adjacent) or 1 (split)");
  DSA_REQUIRE(positions != nullptr || batch > 0, "dsa_rope_headsum_inverse: batch must be positive when no positions are given");
  DSA_REQUIRE(grad && d_emb && cos && sin, "dsa_rope_headsum_inverse: null pointer");
  DSA_REQUIRE(((uintptr_t)d_emb % 4) == 0 && de_tok % 2 == 0, "dsa_rope_headsum_inverse: d_emb rows must start on 4-byte boundaries");
  if (tokens == 0) return DSA_OK;
  hipStream_t st = (hipStream_t)stream;
  dim3 grid(tokens < (1 << 20) ? tokens : (1 << 20)), block(256);
  if (in_pairing == 0)
    rope_headsum_inverse_kernel<ADJ><<<grid, block, 0, st>>>((const unsigned short*)grad, g_tok, g_head, (unsigned short*)d_emb,
                                                            de_tok, emb_dim, cos, sin, cos_sin_f32, positions, batch, tokens, heads);
  else
    rope_headsum_inverse_kernel<SPLIT><<<grid, block, 0, st>>>((const unsigned short*)grad, g_tok, g_head, (unsigned short*)d_emb,
                                                              de_tok, emb_dim, cos, sin, cos_sin_f32, positions, batch, tokens, heads);
  DSA_CHECK_LAUNCH("dsa_rope_headsum_inverse");
  return DSA_OK;
}
