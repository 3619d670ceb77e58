// The fp32 product by three bf16 parts of every entry, as the sparse products use it (gemm_split.hip, gemm_split_device.cuh).
#pragma once
#include "iex_common.h"

namespace iex {

constexpr int kSplitSlots = 512;         // workgroups that make a dense operand's parts, at most
constexpr int kSplitSparseSlots = 2048;  // ... a sparse one's

inline int round32(int x) { return (x + 31) & ~31; }

// src (batch x rows x cols, fp32, at element alignment) as three planes of bf16: high, middle and low parts.  Entry (z, r, c) of a plane lies at
// z * dst_batch + r * ld + c, for r < dst_rows and c < dst_cols (a multiple of 8): zero outside src.
struct SplitDense {
  int batch, rows, cols;
  const float* src;
  int dst_rows, dst_cols, ld;
  long long dst_batch, plane;   // elements
  void* dst;
};
// The dense form of a CSR matrix (columns ascending inside a row) as three planes, rows of ld (a multiple of 32, at least the number of columns).
struct SplitSparse {
  int m, ld;
  const int* row_offsets;
  const int* cols;
  const float* values;
  long long plane;
  void* dst;
};
// Every workgroup leaves the largest magnitude it met, as its bits: at largest[0 ..] those of the second operand (a dense one), from
// largest[kSplitSlots] on those of the first.  How many there are:
int split_dense_blocks(const SplitDense& s);
int split_sparse_blocks(const SplitSparse& s);
int launch_split_operands(const SplitSparse& a, const SplitDense& b, unsigned* largest, hipStream_t stream);
int launch_split_operands(const SplitDense& a, const SplitDense& b, unsigned* largest, hipStream_t stream);

// C = A * B, or with K in parts (gemm_split_parts: more than one) part s's share of it at C + s * stride_part, which the caller adds up.
struct SplitParams {
  int M, N, K;
  const void *A, *B;             // A (M,K), B (N,K) or (K,N): three planes each
  float* C;
  int lda, ldb, ldc;             // row strides in elements
  unsigned plane_a, plane_b;     // bytes from one plane to the next
  long long stride_b, stride_c;  // elements from one batch entry to the next (A is shared)
  const float* row_bias;         // K in one part: C = relu?(A * B + row_bias[row])
  int relu;
  long long stride_part;
  int tiles_m, tiles_n, parts;   // (set by the launcher)
};
int gemm_split_parts(int M, int N, int K, int batch);
double gemm_split_seconds(int M, int N, int K, int batch);   // an estimate, for choices between this product and others
int gemm_split(const SplitParams& p, bool trans_b, int batch, hipStream_t stream);

// out[j] = scores[row of j][cols[j]] (of all parts) for every nonzero j, or the dot product itself where the scores do not stand for it.
struct SplitSample {
  int m, k, n, batch, ld, parts;
  long long stride_part;
  const int* row_offsets;
  const int* cols;
  const float* scores;
  const float *lhs, *rhs;   // (batch, m, k), (batch, n, k)
  float* out;
  const unsigned* largest;
  int slots_a, slots_b;
};
int launch_split_sample(const SplitSample& s, hipStream_t stream);

// From the largest magnitudes of both operands: whether the parts of every entry and product lie inside fp32's normal range (no
// infinities or NaN either), so that the product of the parts stands for the fp32 one.
__device__ __forceinline__ bool split_range_ok(unsigned a, unsigned b) {
  const unsigned inf = 0x7f800000u, least = 37u << 23;   // 2^-90
  if (a == 0u || b == 0u) return a < inf && b < inf;
  if (a >= inf || b >= inf || a < least || b < least) return false;
  const int ea = (int)(a >> 23) - 127, eb = (int)(b >> 23) - 127;
  return ea + eb > -80 && ea + eb < 90 && ea < 126 && eb < 126;
}

}  // namespace iex
