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
// Every workgroup leaves the range of the entries it met, a SplitRange as two words: at ranges[0 ..] those of the second operand (a dense one), from
// ranges[kSplitSlots] on those of the first.  How many there are:
int split_dense_blocks(const SplitDense& s);
int split_sparse_blocks(const SplitSparse& s);
int launch_split_operands(const SplitSparse& a, const SplitDense& b, uint2* ranges, hipStream_t stream);
int launch_split_operands(const SplitDense& a, const SplitDense& b, uint2* ranges, hipStream_t stream);

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
  const uint2* ranges;
  int slots_a, slots_b;
};
int launch_split_sample(const SplitSample& s, hipStream_t stream);

__device__ __forceinline__ unsigned magnitude(float x) { return __float_as_uint(x) & 0x7fffffffu; }

// What is known of an operand's entries: the largest finite magnitude and the smallest but zero, as their bits, and whether there was an
// infinity or a NaN.
struct SplitRange {
  unsigned most = 0;
  unsigned least = ~0u;   // less one: a zero is then the largest of all
  unsigned odd = 0;       // 0 or 1 << 31
  __device__ __forceinline__ void add(float x) {
    const unsigned size = magnitude(x);
    if (size >= 0x7f800000u) odd = 1u << 31;
    else most = max(most, size), least = min(least, size - 1u);
  }
  __device__ __forceinline__ uint2 words() const { return uint2{most | odd, least}; }
  __device__ __forceinline__ void add_words(uint2 w) {
    most = max(most, w.x & 0x7fffffffu);
    least = min(least, w.y);
    odd |= w.x & (1u << 31);
  }
  __device__ __forceinline__ void over_wave() {
#pragma unroll
    for (int d = 32; d; d >>= 1) {
      const uint2 w = words();
      add_words(uint2{(unsigned)__shfl_xor((int)w.x, d), (unsigned)__shfl_xor((int)w.y, d)});
    }
  }
};

// Whether the product of the parts of both operands' finite entries holds what an fp32 one does.  Entries from 2^-110 on have parts that hold
// all their 24 bits (a bit of theirs is worth 2^-133 or more, the least a bf16 can be), and products from 2^-120 on have products of parts that fp32's
// sums, which end at 2^-149, keep to 2^-29 of them.  Rows of 2^-112 beside rows of 1 were off by 1.8e-7, of 2^-120 by 3.7e-5 (row kernel 1.0e-7).  At
// the other end parts, products and their sums stay below infinity.
__device__ __forceinline__ bool split_range_ok(const SplitRange& of_a, const SplitRange& of_b) {
  if (of_a.most == 0u || of_b.most == 0u) return max(of_a.most, of_b.most) < 253u << 23;   // (beyond 2^126 a part may be an infinity, and its product with zero a NaN)
  auto exponent = [](unsigned bits) { return (int)(bits >> 23) - 127; };
  const int least_a = exponent(of_a.least + 1u), least_b = exponent(of_b.least + 1u), most_a = exponent(of_a.most), most_b = exponent(of_b.most);
  return least_a >= -110 && least_b >= -110 && least_a + least_b >= -120 && most_a < 126 && most_b < 126 && most_a + most_b < 90;
}

}  // namespace iex
