// Dense attention for gfx950 on feature-major operands: q, k, v and the output are (heads * HD, tokens) matrices whose
// columns are `seqs` sequences of `length` tokens -- what the projections W_csr @ X of a decoder layer leave and take --
// so no head is ever split off or merged, and neither scores nor probabilities exist outside registers.
//
// By separate kernels (heads split into token-major copies, scores, softmax, context, merge) the attention of the layer of
// 16 x 512 tokens, 32 heads of 128, moved 1.7 GB and took 0.9 ms; the two products alone are 69 GFLOP.
//
// A workgroup of four wavefronts owns 128 queries of one head and sequence, a wavefront 32 of them; keys go by in tiles of
// 64, k and v of a tile loaded straight into LDS while the tile before is worked on (two stages of 2 * HD * 128 bytes: two
// workgroups per CU).  Per wavefront and tile:
//   S^T = K^T Q   MFMA rows = keys, columns = queries, the sum over HD.  k lies [d][key] in LDS, its fragments come by
//                 transpose reads; q's stay in registers.  Key 4..7 and 8..11 of every 16 change places on the way in, so
//                 that a lane's 8 sums of 16 keys are 8 consecutive keys ...
//   P^T = exp2    per lane one query: maximum and sum over its registers, one exchange between the two lanes that share a
//                 query for the maximum, none for the sum until the end
//   O^T += V P    ... and so its probabilities, rounded and packed, ARE the MFMA operand, no lane exchange; v lies [d][key]
//                 in LDS like a row-major operand.  Rows = features, columns = queries: rescaling by a new maximum is one
//                 factor per lane, and done only when some query's maximum has grown.
// What bounds it: per wavefront and tile 32 MFMAs (1024 clocks of the matrix core) beside more clocks of vector instructions
// (exponentials at a quarter rate among them) on two wavefronts per SIMD: vector units busy 54 %, matrix cores 33 %, 33 % of the
// time waiting (profiles/kernel_counters_of_the_cases.txt).  The layer's 32 heads of 128, 16 x 512 tokens: 97 us.
#pragma once
#include "gemm_dma_device.cuh"
#include "online_softmax_device.cuh"

namespace iex {

struct AttentionParams {
  int heads, seqs, length;
  const void* q;
  const void* k;
  const void* v;
  void* out;
  float scale_log2;   // scale * log2(e), > 0
};

// v of keys past a sequence's end: weight 0 times an infinity would be NaN.
static __device__ __align__(16) const unsigned attention_no_values[4] = {0u, 0u, 0u, 0u};

constexpr int kAttnQ = 128, kAttnKeys = 64, kAttnThreads = 256;

template <int HD>
constexpr int attention_lds_bytes() { return 2 * 2 * HD * kAttnKeys * 2; }

template <bool BF16, int HD>
__global__ __launch_bounds__(kAttnThreads, 2) void attention_kernel(AttentionParams p) {
  constexpr int KS = HD / 16, DT = HD / 32;         // sub-steps of the sum over HD, blocks of 32 features
  constexpr int TILE = HD * kAttnKeys * 2;          // bytes of one operand's tile
  constexpr int INSTR = TILE / 1024 / 4;            // direct loads per wavefront, tile and operand (8 rows of 128 bytes each)
  static_assert(HD * kAttnQ * 2 <= attention_lds_bytes<HD>(), "the queries fit the stages");
  typedef unsigned short u16;
  typedef __attribute__((address_space(3))) unsigned char lds_u8;
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = lane >> 5, col = lane & 31;
  const int L = p.length;
  const size_t T = (size_t)p.seqs * L;
  // workgroups go to the XCDs round-robin; renumbered so that an XCD gets all query blocks of a (head, sequence)
  const int blocks = (L + kAttnQ - 1) / kAttnQ, total = gridDim.x;
  const int id = total % kXcds == 0 ? (blockIdx.x % kXcds) * (total / kXcds) + blockIdx.x / kXcds : blockIdx.x;
  const int q0 = (id % blocks) * kAttnQ, head = (id / blocks) % p.heads, seq = id / blocks / p.heads;
  const size_t at = (size_t)head * HD * T + (size_t)seq * L;   // element (feature 0, token 0) of this head and sequence
  const u16* q = static_cast<const u16*>(p.q) + at;
  const u16* k = static_cast<const u16*>(p.k) + at;
  const u16* v = static_cast<const u16*>(p.v) + at;
  u16* out = static_cast<u16*>(p.out) + at;
  const unsigned lds0 = (unsigned)(size_t)(lds_u8*)smem;

  // ---- queries: through the (still unused) stages into registers.  Rows of 128 queries, 16 chunks; a chunk past the
  // sequence's end is its last one (length % 8 == 0), its queries are never stored.
#pragma unroll
  for (int i = 0; i < HD * kAttnQ * 2 / 1024 / 4; ++i) {
    const int g = wave * (HD * kAttnQ * 2 / 1024 / 4) + i;   // 4 rows of 256 bytes
    const int d = g * 4 + lane / 16;
    const int c = (lane % 16) ^ kn_swizzle<kAttnQ>(d);
    lds_dma16(q + d * T + min(q0 + c * 8, L - 8), __builtin_amdgcn_readfirstlane(lds0 + g * 1024));
  }
  wait_vmcnt<0>();
  __syncthreads();
  u32x4 fq[KS];
  {
    const int off = kn_fragment_offset<kAttnQ>(lane, wave);
#pragma unroll
    for (int s = 0; s < KS; ++s) fq[s] = kn_fragment<kAttnQ * 2>(smem + off + s * 16 * (kAttnQ * 2));
  }
#pragma unroll
  for (int s = 0; s < KS; ++s) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(fq[s]));
  __syncthreads();

  // ---- direct loads of a key tile: 8 rows (features) of 64 keys per instruction
  const int row_in = lane / 8, chunk_in = lane % 8;
  auto issue = [&](int tile, int stage) {
    const int k0 = tile * kAttnKeys;
#pragma unroll
    for (int i = 0; i < INSTR; ++i) {
      const int g = wave * INSTR + i, d = g * 8 + row_in;
      const unsigned base = lds0 + stage * 2 * TILE + g * 1024;
      lds_dma16(k + d * T + min(k0 + (chunk_in ^ kn_swizzle<kAttnKeys>(d)) * 8, L - 8), __builtin_amdgcn_readfirstlane(base));
      const int at_v = k0 + (chunk_in ^ ((d >> 1) & 7)) * 8;
      lds_dma16(at_v < L ? static_cast<const void*>(v + d * T + at_v) : attention_no_values, __builtin_amdgcn_readfirstlane(base + TILE));
    }
  };
  // where a lane's fragments start: k by transpose reads with the middle quads of every 16 keys exchanged, v as 16 bytes
  // of one feature's keys
  int k_off[2];
  {
    const int kr = half * 8 + ((lane & 15) >> 2), quad = ((lane & 1) << 1) | ((lane >> 1) & 1);   // 0, 2, 1, 3
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int c = (b * 4 + ((lane >> 4) & 1) * 2 + (quad >> 1)) ^ kn_swizzle<kAttnKeys>(kr);
      k_off[b] = kr * (kAttnKeys * 2) + c * 16 + (quad & 1) * 8;
    }
  }

  f32x16 o[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[d][r] = 0.f;
  float top = -INFINITY, sum = 0.f;   // of this lane's query: the maximum so far (both lanes' keys), this lane's share of the sum

  const int tiles = (L + kAttnKeys - 1) / kAttnKeys;
  issue(0, 0);
  for (int t = 0; t < tiles; ++t) {
    wait_vmcnt<0>();
    __syncthreads();   // everybody's loads of tile t have landed, and everybody is done with the other stage
    if (t + 1 < tiles) issue(t + 1, (t + 1) & 1);
    const unsigned char* sk = smem + (t & 1) * 2 * TILE;
    const unsigned char* sv = sk + TILE;

    f32x16 s[2];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[b][r] = 0.f;
#pragma unroll
    for (int e = 0; e < KS; ++e)
#pragma unroll
      for (int b = 0; b < 2; ++b) s[b] = mfma_32x32x16<BF16>(kn_fragment<kAttnKeys * 2>(sk + k_off[b] + e * 16 * (kAttnKeys * 2)), fq[e], s[b]);
    if (t * kAttnKeys + kAttnKeys > L) {   // (uniform) the last tile: keys past the end
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (t * kAttnKeys + b * 32 + (r / 8) * 16 + half * 8 + r % 8 >= L) s[b][r] = -INFINITY;
    }
    softmax_maximum(s, o, top, sum, p.scale_log2);
    u32x4 fp[4];   // the probabilities as MFMA operand: 16 keys each
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      softmax_weights<8>(s[e / 2], e % 2 * 8, top, sum, p.scale_log2);
      fp[e] = probability_operand<BF16>(s[e / 2], e % 2 * 8);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        const int row = d * 32 + col;
        const u32x4 fv = *reinterpret_cast<const u32x4*>(sv + row * (kAttnKeys * 2) + (((e * 2 + half) ^ ((row >> 1) & 7)) * 16));
        o[d] = mfma_32x32x16<BF16>(fv, fp[e], o[d]);
      }
  }
  sum += __shfl_xor(sum, 32);
  const float inv = 1.f / sum;
  const int query = q0 + wave * 32 + col;
  if (query < L) {
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r)   // (32 consecutive queries of one feature per half wavefront: 64 bytes)
        out[(d * 32 + 8 * (r / 4) + 4 * half + r % 4) * T + query] = f32_to_16(o[d][r] * inv, BF16);
  }
}

}  // namespace iex
