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
// Every workgroup leaves the range of the entries it met, a SplitRange as a word: at ranges[0 ..] those of the second operand (a dense one), from
// ranges[kSplitSlots] on those of the first.  How many there are:
int split_dense_blocks(const SplitDense& s);
int split_sparse_blocks(const SplitSparse& s);
int launch_split_operands(const SplitSparse& a, const SplitDense& b, unsigned* ranges, hipStream_t stream);
int launch_split_operands(const SplitDense& a, const SplitDense& b, unsigned* ranges, hipStream_t stream);

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
  const unsigned* ranges;
  int slots_a, slots_b;
};
int launch_split_sample(const SplitSample& s, hipStream_t stream);

__device__ __forceinline__ unsigned magnitude(float x) { return __float_as_uint(x) & 0x7fffffffu; }

// What is known of an operand's entries: the largest finite magnitude, as its bits, and whether there was an infinity or a NaN.
struct SplitRange {
  unsigned most = 0;
  unsigned odd = 0;   // 0 or 1 << 31
  __device__ __forceinline__ void add(float x) {
    const unsigned size = magnitude(x);
    if (size >= 0x7f800000u) odd = 1u << 31;
    else most = max(most, size);
  }
  __device__ __forceinline__ unsigned word() const { return most | odd; }
  __device__ __forceinline__ void add_word(unsigned w) {
    most = max(most, w & 0x7fffffffu);
    odd |= w & (1u << 31);
  }
  __device__ __forceinline__ void over_wave() {
#pragma unroll
    for (int d = 32; d; d >>= 1) add_word((unsigned)__shfl_xor((int)word(), d));
  }
};

// Whether the largest entries of both operands and their product lie inside fp32's normal range, so that the product of the parts of finite
// entries stands for the fp32 one.
__device__ __forceinline__ bool split_range_ok(const SplitRange& of_a, const SplitRange& of_b) {
  const unsigned a = of_a.most, b = of_b.most, least = 37u << 23;   // 2^-90
  if (a == 0u || b == 0u) return max(a, b) < 253u << 23;   // (beyond 2^126 a part may be an infinity, and its product with zero a NaN)
  if (a < least || b < least) return false;
  const int ea = (int)(a >> 23) - 127, eb = (int)(b >> 23) - 127;
  return ea + eb > -80 && ea + eb < 90 && ea < 126 && eb < 126;
}

}  // namespace iex
