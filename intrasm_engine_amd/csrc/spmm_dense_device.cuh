// Dense form of a CSR matrix with 16-bit values (fp16 / bf16 bit patterns), for the SpMM path
// that hands the product to the dense GEMM: every workgroup that computes a tile of the output
// of a matrix-core SpMM kernel rebuilds the dense form of its rows of A in LDS, once per column
// tile of the output; when the output has many column tiles it is cheaper to build the dense
// form once, in a workspace of m * k * 2 bytes that stays in L2 / MALL, and let the GEMM read it.
//
// One workgroup of four wavefronts per pair of rows (the loads of both rows in flight together): each row is assembled
// in LDS (zeros, then the nonzeros scattered to their columns, each wavefront taking a contiguous quarter of them) and written with 128-bit stores, so every byte of the
// workspace is written exactly once, by one kind of store, whatever the sparsity.  What a row costs is the chain of
// "load 256 nonzeros, scatter them" steps of its wavefronts, each a round trip to memory: with one wavefront per row
// the longest row set the kernel's time (4096 nonzeros: 16 steps, 24 us where the bytes written take 8).
// Rows longer than the columns in LDS are done in segments, every wavefront with a cursor into its quarter of the
// row's ascending column indices: quarters wait for their segment, so rows of more than 5120 columns have a workgroup and LDS for 12288 of them to themselves
// (4096 x 11008 at 90 %, geometric lengths, 30.4 -> 20.8 us, even ones 21.9 -> 19.9; 500 x 8000 10.7 -> 6.2; not for 11008 x 4160, 20.6 -> 21.1).  k, here the row stride of the dense form, is a multiple of 8 and no less than the number
// of columns (the rest is zero); the workspace is 16-byte aligned; column indices inside a row must ascend strictly
// (canonical CSR).
#pragma once
#include "iex_common.h"

namespace iex {

constexpr int kDenseSeg = 4096;       // columns of a row assembled at a time, two rows to a workgroup (16 KB of LDS)
constexpr int kDenseLongSeg = 12288;  // ... of longer rows, one to a workgroup (24 KB)
constexpr int kDenseWaves = 4;
constexpr int kDenseThreads = kDenseWaves * kWave;

template <typename IT, int ROWS, int SEG>
__global__ __launch_bounds__(kDenseThreads) void csr_to_dense_kernel(int m, int k, const int* __restrict__ row_offsets,
                                                                     const IT* __restrict__ cols,
                                                                     const uint16_t* __restrict__ values,
                                                                     uint16_t* __restrict__ out, int* __restrict__ zero_words,
                                                                     int n_zero_words) {
  __shared__ __align__(16) uint16_t srow[ROWS][SEG];
  // (words that the kernel after this one wants zero at its launch, a few hundred at most: cheaper here than a launch)
  if (blockIdx.x == 0)
    for (int i = threadIdx.x; i < n_zero_words; i += kDenseThreads) zero_words[i] = 0;
  const int lane = lane_id();
  const int wave = uniform(threadIdx.x >> 6);
  // this wavefront's quarter of each row's nonzeros, in whole chunks of 64
  int pos[ROWS], end[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const int row = min((int)blockIdx.x * ROWS + r, m - 1);   // (the grid has ceil(m / ROWS) workgroups)
    const int first = uniform(row_offsets[row]);
    const int last = (int)blockIdx.x * ROWS + r < m ? uniform(row_offsets[row + 1]) : first;   // (past the matrix: an empty row, not stored)
    const int share = ((max(last - first, 0) + kWave * kDenseWaves - 1) / (kWave * kDenseWaves)) * kWave;
    pos[r] = min(first + wave * share, last);
    end[r] = min(pos[r] + share, last);
  }
  for (int c0 = 0; c0 < k; c0 += SEG) {
    const int len = min(SEG, k - c0);  // a multiple of 8
    if (c0) __syncthreads();   // the previous segment has been copied out
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
      for (int i = threadIdx.x * 8; i < len; i += kDenseThreads * 8) *reinterpret_cast<uint4*>(srow[r] + i) = uint4{0u, 0u, 0u, 0u};
    __syncthreads();
    // the nonzeros of this segment: 64 at a time from the cursors, four chunks of each row in flight
    bool more[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) more[r] = pos[r] < end[r];
    static_assert(ROWS <= 2, "the loop below names both rows");
    while (more[0] || more[ROWS - 1]) {
      int c[ROWS][4];
      uint16_t v[ROWS][4];
#pragma unroll
      for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int j = max(min(pos[r] + u * kWave + lane, end[r] - 1), 0);   // (a row without nonzeros: entry 0, never used)
          c[r][u] = (int)cols[j] - c0;
          v[r][u] = values[j];
        }
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        int taken = 0;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          // (canonical CSR: c >= 0, earlier segments took what lies before c0; the test keeps a row whose
          // columns do not ascend inside the row's slice of LDS -- its result is then undefined, not a fault)
          const bool mine = more[r] && pos[r] + u * kWave + lane < end[r] && c[r][u] < len && c[r][u] >= 0;
          if (mine) srow[r][c[r][u]] = v[r][u];
          taken += __popcll(__ballot(mine));
        }
        pos[r] += taken;
        more[r] = taken == 4 * kWave;  // a short take: the quarter ended or its next nonzero lies beyond this segment
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const int row = (int)blockIdx.x * ROWS + r;
      if (row < m)
        for (int i = threadIdx.x * 8; i < len; i += kDenseThreads * 8)
          *reinterpret_cast<uint4*>(out + (size_t)row * k + c0 + i) = *reinterpret_cast<const uint4*>(srow[r] + i);
    }
  }
}

// dst (dst_rows x ld, ld a multiple of 8, 16-byte aligned) = src (rows x cols, at element alignment) with zeros around it:
// a dense operand of any shape as the GEMM's direct loads want it.  One 16-byte chunk of dst per thread.
static __global__ __launch_bounds__(256) void pad_rows_kernel(int rows, int cols, const uint16_t* __restrict__ src, int dst_rows, int ld, uint16_t* __restrict__ dst,
                                                              long long src_stride) {
  struct alignas(2) Any { uint16_t v[8]; };
  struct alignas(16) Whole { uint16_t v[8]; };
  const int chunks = ld / 8;
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long long)dst_rows * chunks) return;
  const int r = (int)(i / chunks), c = (int)(i % chunks) * 8;
  src += (size_t)blockIdx.y * src_stride + (size_t)r * cols;
  dst += (size_t)blockIdx.y * dst_rows * ld + (size_t)r * ld;
  Whole w{};
  if (r < rows && c + 8 <= cols) {
    const Any a = *reinterpret_cast<const Any*>(src + c);
#pragma unroll
    for (int e = 0; e < 8; ++e) w.v[e] = a.v[e];
  } else if (r < rows) {
#pragma unroll
    for (int e = 0; e < 8; ++e) w.v[e] = c + e < cols ? src[c + e] : (uint16_t)0;
  }
  *reinterpret_cast<Whole*>(dst + c) = w;
}

// (k: the row stride of the dense form)
template <typename IT>
inline void launch_csr_to_dense(int m, int k, const int* row_offsets, const void* cols, const void* values, void* out, int* zero_words, int n_zero_words,
                                hipStream_t stream) {
  if (k < kDenseSeg + kDenseSeg / 4)
    hipLaunchKernelGGL((csr_to_dense_kernel<IT, 2, kDenseSeg>), dim3(ceil_div(m, 2)), dim3(kDenseThreads), 0, stream, m, k, row_offsets, static_cast<const IT*>(cols),
                       static_cast<const uint16_t*>(values), static_cast<uint16_t*>(out), zero_words, n_zero_words);
  else
    hipLaunchKernelGGL((csr_to_dense_kernel<IT, 1, kDenseLongSeg>), dim3(m), dim3(kDenseThreads), 0, stream, m, k, row_offsets, static_cast<const IT*>(cols),
                       static_cast<const uint16_t*>(values), static_cast<uint16_t*>(out), zero_words, n_zero_words);
}

inline int round8(int x) { return (x + 7) & ~7; }
inline size_t round256(size_t x) { return (x + 255) & ~size_t(255); }

// rows x cols (`batch` of them, src_stride elements apart) into dst_rows x ld, as above.
inline int launch_pad_rows(int rows, int cols, const void* src, int dst_rows, int ld, void* dst, int batch, long long src_stride, hipStream_t stream) {
  note_kernel("pad_rows_kernel");
  hipLaunchKernelGGL(pad_rows_kernel, dim3(ceil_div((long long)dst_rows * (ld / 8), 256), batch), dim3(256), 0, stream, rows, cols,
                     static_cast<const uint16_t*>(src), dst_rows, ld, static_cast<uint16_t*>(dst), src_stride);
  return check_hip(hipGetLastError(), "padding launch");
}

}  // namespace iex
