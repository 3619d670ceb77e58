// Which bytes of global memory the direct-load GEMM tiles (gemm_dma_device.cuh, gemm_pp_device.cuh) ask for: where a
// buffer ends, which 16-byte chunk a lane of a direct load fetches, how K is dealt to the workgroups of a tile.  Plain
// C++, so that a program on the host can walk every address of a launch (tests/gemm_addresses_check.cpp).
#pragma once
#include <cstddef>

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define IEX_HD __host__ __device__ __forceinline__
#else
#define IEX_HD inline
#endif

namespace iex {

// Bytes from the first element of `rows` rows of `width` elements, ld apart, to the end of the last one.  This and not
// rows * ld is where a buffer has to end: with K in parts a part starts k0 elements into its row, with a row stride above
// the width the last row has no gap behind it, and both would put the end past the allocation.  (16-bit elements; a width
// of no whole chunks has rows padded to whole chunks.)
IEX_HD size_t rows_bytes(int rows, int width, int ld) { return ((size_t)(rows - 1) * ld + (width + 7) / 8 * 8) * 2; }

// A chunk of 8 elements: its byte offset inside the buffer at k = 0, and where it lies along K inside a stage.
struct DirectChunk {
  unsigned offset;
  int k;
};

// Operand whose rows are contiguous along K, a stage of STAGE_K elements of them: direct load `instr` of the workgroup
// fills 64 * 8 / STAGE_K rows of LDS, position c of a row holds chunk c ^ swizzle(row).  `rows`: how many the operand has from
// the buffer's first; a row past them is the last one.
template <int STAGE_K>
IEX_HD DirectChunk row_chunk(int instr, int lane, int rows, int ld) {
  constexpr int CPR = STAGE_K / 8;
  static_assert(CPR == 4 || CPR == 8, "stages of 32 or 64 k");
  const int row = instr * (64 / CPR) + lane / CPR;
  const int k = ((lane % CPR) ^ (CPR == 4 ? (row >> 2) & 3 : (row >> 1) & 7)) * 8;
  return DirectChunk{((unsigned)(row < rows ? row : rows - 1) * ld + k) * 2u, k};
}

// Chunk permutation of k row kr of an operand whose LDS rows hold ROW_ELEMS elements of one k, for fragments of 16 rows
// (columns) x 32 k: a read of 32 lanes covers 4 k rows and the 4 k rows 8 further, 32 bytes of each, and the permutation
// puts them into the eight different 8-bank groups.
template <int ROW_ELEMS>
IEX_HD int kn16_swizzle(int kr) {
  return ROW_ELEMS >= 128 ? ((kr & 3) << 1) | (kr & 8) : (kr & 2) | ((kr & 8) >> 1);
}

// Operand of one row per k, ROW_ELEMS elements of it from column `first` on: a column past the row's stride is its last chunk.
template <int ROW_ELEMS>
IEX_HD DirectChunk column_chunk(int instr, int lane, int first, int ld) {
  constexpr int CPR = ROW_ELEMS / 8;
  static_assert(CPR >= 8 && CPR <= 64, "one direct load fills whole rows");
  const int kr = instr * (64 / CPR) + lane / CPR;
  const int col = first + ((lane % CPR) ^ kn16_swizzle<ROW_ELEMS>(kr)) * 8;
  return DirectChunk{((unsigned)kr * ld + (col < ld - 8 ? col : ld - 8)) * 2u, kr};
}

// A stretch of K: from k0, K elements, of which kb rows of a (K,N) B exist.
struct KPart {
  int k0, K, kb;
};

// Part `part` of `parts` in whole steps of bk; the host has chosen parts so that every part has a step.  (The rows of B that
// are missing are fewer than a chunk: the last part has some.)
IEX_HD KPart k_in_parts(int K, int kb, int bk, int parts, int part) {
  const int per = ((K + bk - 1) / bk + parts - 1) / parts * bk, k0 = part * per;
  const int len = per < K - k0 ? per : K - k0;
  return KPart{k0, len, len < kb - k0 ? len : kb - k0};
}

// The two halves of K in whole steps of bk, the first the shorter one.
IEX_HD KPart k_in_halves(int K, int kb, int bk, int part) {
  const int first = ((K + bk - 1) / bk / 2) * bk, k0 = part ? first : 0, len = part ? K - first : first;
  return KPart{k0, len, len < kb - k0 ? len : kb - k0};
}

}  // namespace iex
