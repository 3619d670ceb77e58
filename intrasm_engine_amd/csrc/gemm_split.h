// The fp32 product by three bf16 parts of every entry, as the sparse products use it (gemm_split.hip, gemm_split_device.cuh).
#pragma once
#include "iex_common.h"

namespace iex {

constexpr int kSplitSlots = 512;         // workgroups that make a dense operand's parts, at most
constexpr int kSplitSparseSlots = 2048;  // ... a sparse one's

constexpr int kSplitVerdict = kSplitSlots + kSplitSparseSlots, kSplitRanges = kSplitVerdict + 64;   // (whole 256 bytes)

// The most that a call's workspace for parts may take: 1.4 % of the card's memory.  What would need more runs on the kernels without one.
constexpr size_t kSplitWorkspaceMost = (size_t)4 << 30;

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
// ranges[kSplitSlots] on those of the first.  The product leaves at ranges[kSplitVerdict] whether it stands for the fp32 one; room for kSplitRanges in all.  How many
// there are of each:
int split_dense_blocks(const SplitDense& s);
int split_sparse_blocks(const SplitSparse& s);
int launch_split_operands(const SplitSparse& a, const SplitDense& b, unsigned* ranges, hipStream_t stream);
int launch_split_operands(const SplitDense& a, const SplitDense& b, unsigned* ranges, hipStream_t stream);
int launch_split_operand(const SplitDense& b, unsigned* ranges, hipStream_t stream);   // the second one alone

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
  unsigned* ranges;                 // of the operands' entries, and the verdict: where the range says that the parts do not hold the entries nothing else is written
  int slots_a, slots_b;
  int finite;                    // ... and where there is an infinity or a NaN
  int parts;                     // of K, each with at least a step: gemm_split_parts
  int tiles_m, tiles_n;          // (set by the launcher)
};
int gemm_split_parts(int M, int N, int K, int batch);
double gemm_split_seconds(int M, int N, int K, int batch);   // an estimate, for choices between this product and others
int gemm_split(const SplitParams& p, bool trans_b, int batch, hipStream_t stream);

// out[j] = scores[row of j][cols[j]] (of all parts) for every nonzero j, or the dot product itself where the scores do not stand for it.  wide: a workgroup per row.
struct SplitSample {
  int m, k, n, batch, ld, parts, wide;
  long long stride_part;
  const int* row_offsets;
  const int* cols;
  const float* scores;
  const float *lhs, *rhs;   // (batch, m, k), (batch, n, k)
  float* out;
  const unsigned* ranges;
};
int launch_split_sample(const SplitSample& s, hipStream_t stream);

__device__ __forceinline__ unsigned magnitude(float x) { return __float_as_uint(x) & 0x7fffffffu; }

// What is known of an operand's entries: the exponents of the largest finite magnitude and of the smallest but zero, and whether there was an
// infinity or a NaN.  As a word: the first in the low byte, 255 less the second in the next one, the third above; 0 of no entries or zeros.
struct SplitRange {
  unsigned most = 0, small = 0, odd = 0;
  __device__ __forceinline__ void add_word(unsigned w) {
    most = max(most, w & 0xffu);
    small = max(small, w & 0xff00u);
    odd |= w & 0x10000u;
  }
  __device__ __forceinline__ unsigned word() const { return most | small | odd; }
  __device__ __forceinline__ void over_wave() {
    most = (unsigned)wave_max((float)most);
    small = (unsigned)wave_max((float)small);
    odd = __ballot(odd != 0) ? 0x10000u : 0u;
  }
};
// ... and how it is found, entry by entry
struct SplitExtent {
  unsigned most = 0, least = ~0u, odd = 0;   // magnitudes as their bits (least: less one, a zero is then the largest of all)
  __device__ __forceinline__ void add(float x) {
    const unsigned size = magnitude(x);
    if (size >= 0x7f800000u) odd = 0x10000u;
    else most = max(most, size), least = min(least, size - 1u);
  }
  __device__ __forceinline__ SplitRange range() const { return SplitRange{most >> 23, least == ~0u ? 0u : (255u - ((least + 1u) >> 23)) << 8, odd}; }
};

// Whether the product of the parts of both operands' finite entries holds what an fp32 one does.  Entries from 2^-110 on have parts that hold
// all their 24 bits (a bit of theirs is worth 2^-133 or more, the least a bf16 can be), and products from 2^-120 on have products of parts that fp32's
// sums, which end at 2^-149, keep to 2^-29 of them.  Rows of 2^-112 beside rows of 1 were off by 1.8e-7, of 2^-120 by 3.7e-5 (row kernel 1.0e-7).  At
// the other end parts, products and their sums stay below infinity.
__device__ __forceinline__ bool split_range_ok(const SplitRange& of_a, const SplitRange& of_b) {
  const int most_a = (int)of_a.most - 127, most_b = (int)of_b.most - 127, least_a = 128 - (int)(of_a.small >> 8), least_b = 128 - (int)(of_b.small >> 8);
  if (most_a >= 126 || most_b >= 126) return false;         // (beyond 2^126 a part may be an infinity, and its product with zero a NaN)
  if (of_a.small == 0 || of_b.small == 0) return true;      // (zeros alone)
  return least_a >= -110 && least_b >= -110 && least_a + least_b >= -120 && most_a + most_b < 90;
}

}  // namespace iex
