// One tile of keys of a softmax that runs over tiles (attention_device.cuh, sparse_attention_device.cuh): a lane holds KB * 16
// scores of one query, shared with the lane 32 further, and DT * 16 sums of what the probabilities weigh.
#pragma once
#include "gemm_device.cuh"

namespace iex {

// The running maximum of the query over both lanes' scores; sums so far follow it (once the first tile is past ever more
// rarely).  top starts below every score: -infinity where every tile has a score for every query, a finite mark where a query
// may have none yet.
template <int KB, int DT>
__device__ __forceinline__ void softmax_maximum(f32x16 (&s)[KB], f32x16 (&o)[DT], float& top, float& sum, float scale_log2) {
  float m = s[0][0];
#pragma unroll
  for (int b = 0; b < KB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) m = fmaxf(m, s[b][r]);
  m = fmaxf(m, __shfl_xor(m, 32));
  if (__ballot(m > top)) {
    const float now = fmaxf(top, m), keep = __builtin_amdgcn_exp2f((top - now) * scale_log2);
    top = now;
    sum *= keep;
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[d][r] *= keep;
  }
}

// R scores from r0 on become exp2((score - maximum) * scale), added to this lane's share of the sum.
template <int R>
__device__ __forceinline__ void softmax_weights(f32x16& s, int r0, float top, float& sum, float scale_log2) {
  const float shift = -top * scale_log2;
#pragma unroll
  for (int r = r0; r < r0 + R; ++r) {
    s[r] = __builtin_amdgcn_exp2f(fmaf(s[r], scale_log2, shift));   // (exp2(-infinity) = 0)
    sum += s[r];
  }
}

// Eight probabilities from r0 on, rounded and packed: an MFMA operand of 16 keys (the other lane has the other eight).
template <bool BF16>
__device__ __forceinline__ u32x4 probability_operand(const f32x16& x, int r0) {
  return u32x4{pack_pair<BF16>(x[r0], x[r0 + 1]), pack_pair<BF16>(x[r0 + 2], x[r0 + 3]), pack_pair<BF16>(x[r0 + 4], x[r0 + 5]),
               pack_pair<BF16>(x[r0 + 6], x[r0 + 7])};
}

}  // namespace iex
