// Host side of the CSR SpMM: kernel wrappers, variant selection, argument checks and
// the C entry points.  The device code is in spmm_device.cuh.
#include <algorithm>
#include <cmath>
#include <mutex>
#include "gemm_split.h"
#include "spmm_dense_device.cuh"
#include "spmm_lds_device.cuh"
#include "spmm_mfma2_device.cuh"
#include "spmm_mfma3_device.cuh"
#include "spmm_mfma_f32_device.cuh"
#include "spmm_smallk_device.cuh"

namespace iex {
namespace {

// SHORT: rows of which a wavefront gets a few dozen nonzeros, see launch_one
template <typename T, typename IT, int VEC, int LPG, int WPR, int NT, bool SHORT>
__global__ __launch_bounds__((WPR > 4 ? WPR : 4) * 64) void spmm_kernel(SpmmParams p) {
  __shared__ float red[spmm_lds_floats<VEC, WPR, NT>()];
  spmm_block<T, IT, VEC, LPG, WPR, (NT > 1 || SHORT ? kSpmmUnroll / 2 : kSpmmUnroll), NT, false, (SHORT || sizeof(T) == 2)>(p, blockIdx.x, blockIdx.y, blockIdx.z, red);
}

template <typename T, typename IT, int VEC, int LPG, int WPR, int NT = 1>
int launch_one(const SpmmParams& p, int batch, hipStream_t stream) {
  constexpr int kWavesPerBlock = (WPR > 4) ? WPR : 4;
  constexpr int kRowsPerBlock = kWavesPerBlock / WPR;
  dim3 grid(ceil_div(p.m, kRowsPerBlock), ceil_div(p.n, NT * LPG * VEC), batch);
  dim3 block(kWavesPerBlock * kWave);
  // Several nonzeros per gather and rows of at most 128 on average, more of them than are resident: windows of four gathers
  // instead of eight.  Fewer registers (n = 64 62 instead of 82 in fp32, n = 128 62 instead of 94 in fp16: 8 wavefronts per SIMD instead of 5; n = 128
  // in fp32 72 instead of 98, 7 instead of 4), and a short share is mostly
  // its last, partial window.  MI355X, us, eight / four: 11008 x 1000, 90 / 95 % sparse, fp32 n = 64 21 / 16 and 21 / 13, n =
  // 128 32 / 25 and 25 / 19, fp16 n = 128 25 / 21 and 25 / 17, n = 256 - and 30 / 24.  Longer rows want the gathers in
  // flight (4096 x 4096, 90 %, fp16 n = 128 22 / 26, fp32 n = 64 22 / 27), few rows leave the registers idle (1024 x 1024, 95 %, fp16 n
  // = 256 4.7 / 5.1).  There the last gathers of a chunk go by fours and twos in 16 bits (1024 - 4096, 90 - 98 %: 3 - 9 % less time); in
  // 32 bits that costs the 4096 x 4096 cells with long rows 5 %.
  const char* const name = "spmm_kernel<%s, %s, %d, %d, %d, %d, %s>";
  if constexpr (LPG < kWave && NT == 1) {
    if (p.nnz <= 128ll * p.m && (long long)p.m * grid.y * batch * WPR > 16384) {
      note_kernel(name, type_name<T>(), type_name<IT>(), VEC, LPG, WPR, NT, "true");
      hipLaunchKernelGGL((spmm_kernel<T, IT, VEC, LPG, WPR, NT, true>), grid, block, 0, stream, p);
      return check_hip(hipGetLastError(), "spmm launch");
    }
  }
  note_kernel(name, type_name<T>(), type_name<IT>(), VEC, LPG, WPR, NT, "false");
  hipLaunchKernelGGL((spmm_kernel<T, IT, VEC, LPG, WPR, NT, false>), grid, block, 0, stream, p);
  return check_hip(hipGetLastError(), "spmm launch");
}

// n not a multiple of the 128-bit vector: full-width tiles with vectors at element alignment
template <typename T, typename IT, int VEC, int WPR>
__global__ __launch_bounds__((WPR > 4 ? WPR : 4) * 64) void spmm_ragged_kernel(SpmmParams p) {
  __shared__ float red[spmm_lds_floats<VEC, WPR, 1>()];
  spmm_block<T, IT, VEC, kWave, WPR, kSpmmUnroll, 1, true>(p, blockIdx.x, blockIdx.y, blockIdx.z, red);
}

template <typename T, typename IT, int VEC, int WPR>
int launch_ragged_one(const SpmmParams& p, int batch, hipStream_t stream) {
  constexpr int kWavesPerBlock = (WPR > 4) ? WPR : 4;
  constexpr int kRowsPerBlock = kWavesPerBlock / WPR;
  dim3 grid(ceil_div(p.m, kRowsPerBlock), ceil_div(p.n, kWave * VEC), batch);
  note_kernel("spmm_ragged_kernel<%s, %s, %d, %d>", type_name<T>(), type_name<IT>(), VEC, WPR);
  hipLaunchKernelGGL((spmm_ragged_kernel<T, IT, VEC, WPR>), grid, dim3(kWavesPerBlock * kWave), 0, stream, p);
  return check_hip(hipGetLastError(), "spmm (ragged rows) launch");
}

template <typename T, typename IT, int VEC>
int launch_ragged(const SpmmParams& p, int batch, int wpr, hipStream_t stream) {
  switch (wpr) {
    case 1: return launch_ragged_one<T, IT, VEC, 1>(p, batch, stream);
    case 4: return launch_ragged_one<T, IT, VEC, 4>(p, batch, stream);
    case 8: return launch_ragged_one<T, IT, VEC, 8>(p, batch, stream);
  }
  return fail(IEX_ERR_BAD_ARGUMENT, "spmm: waves-per-row must be 1, 4 or 8 (got %d)", wpr);
}

// ---- few columns in A, wide output: the dense operand's tile lives in LDS ---------------------
template <typename T, typename IT, int VEC, bool RAGGED, int WAVES, int MOST, bool PLAIN, bool SCALAR>
__global__ __launch_bounds__(WAVES * kWave) void spmm_smallk_kernel(SpmmParams p, int rows_per_wave) {
  extern __shared__ __align__(16) unsigned char smem[];
  spmm_smallk_block<T, IT, VEC, RAGGED, WAVES, MOST, PLAIN, SCALAR>(p, rows_per_wave, blockIdx.x, blockIdx.y, blockIdx.z, smem);
}

// The same with every line of the output written by one wavefront (fp32, no bias, ReLU or accumulation).
template <int WAVES>
__global__ __launch_bounds__(WAVES * kWave) void spmm_smallk_kernel_lines(SpmmParams p, SmallkLines t, int rows_per_wave) {
  extern __shared__ __align__(16) unsigned char smem[];
  spmm_smallk_lines_block<WAVES>(p, t, rows_per_wave, blockIdx.x, blockIdx.y, blockIdx.z, smem);
}

// full vectors at their natural alignment, or (ragged) any n at element alignment
template <typename T>
bool smallk_aligned(const SpmmParams& p) {
  constexpr int kMax = 16 / (int)sizeof(T);
  return p.n % kMax == 0 && aligned(p.dense, 16) && aligned(p.out, 16);
}

// Whole lines per wavefront: fp32 rows that do not start at multiples of 64 bytes.  A dword of LDS per lane, nonzero and 64 columns costs more
// instructions than 128-bit vectors: up to 9 nonzeros a row (us, this / vectors: 384 x 785 x 785, 3.2 per row 252 / 283, 6.4 218 / 295, 9.6
// 331 / 265, 19 429 / 411; 24 x 3133 x 3133, 6.4 215 / 283, 12.8 366 / 344; 64 x 1004 x 1004, 6.4 53 / 89, 12.8 104 / 101).
template <typename T>
bool smallk_by_lines(const SpmmParams& p) {
  return sizeof(T) == 4 && !p.bias && !p.relu && !p.accumulate && (p.n % 16 != 0 || !aligned(p.out, 64)) && p.nnz <= 9ll * p.m && smallk_lines(p.n, p.k).rest > 0;
}

template <typename T>
bool smallk_fits(const SpmmParams& p) {
  constexpr int kMax = 16 / (int)sizeof(T);
  return p.k >= 1 && p.k <= kSmallKMax && p.n >= (sizeof(T) == 2 ? kWave : kWave * kMax) && aligned(p.dense, sizeof(T)) && aligned(p.out, sizeof(T));
}

template <typename T>
bool matrix_core_kernel_applies(const SpmmParams& p, int batch);

// ... and where the library takes it by itself: up to 64 columns (two workgroups per CU), enough rows for
// the tile load (k KB per workgroup) to be a fraction of what the workgroup writes, and rows that gather:
// from 1.8 nonzeros per row the LDS gather wins (fp32, per-batch values: 192 x 784 x 784 outputs,
// k = 32, 2 per row: 107 against 127 us; 8 x 4096 x 4096, k = 64, 6 per row: 126 / 172, 32 per row: 344 / 535);
// almost empty rows are a plain write, which the row kernel does at 6 TB/s with streaming stores
// (96 x 3136 x 3136, 0.5 per row: 627 against 711).
//   (rows that are no multiple of the vector: from 2.5 per row -- 384 x 785 x 785, k = 64: 3.2 per row 377 -> 322 us,
//   1.9 per row 290 -> 313)
// k = 65 .. 128 (one workgroup of 16 wavefronts per CU), fewer rows per dense row, and outputs narrower than a vector per lane
// (fp32 / 16-bit; us by the other kernels -> here, for outputs large enough to fill the chip):
//   k = 128, fp32: 60 x 1000 x 1000, 13 per row 136 -> 99, 2.6 per row 68 -> 91; 24 x 3136 x 3136, 13 per row 450 -> 361, 38 per row
//     2083 -> 782; 200 x 333 x 333, 13 per row 76 -> 72;
//   k = 128, fp16: 24 x 785 x 785, 13 per row 45 -> 30; 200 x 333 x 333, 2.6 per row 30 -> 26, 13 per row 77 -> 49; but where the
//     matrix-core kernels apply they stay ahead (24 x 3136 x 3136, 13 per row 214 / 230, 38 per row 244 / 590);
//   k = 64, m = 333: 13 per row 71 -> 47 (fp32), 78 -> 49 (fp16), 1.9 per row 26 / 28;
//   rows of fp16 narrower than half a tile and no whole vectors, which the row kernel takes in single elements: 384 x 197 x 197
//     64 - 177 -> 26 - 116 whatever k and density; fp32 there: 46 / 53 at 13 per row.
// Where lines are written whole (smallk_by_lines) it is ahead from fewer nonzeros on, outputs of 80 MB and more: any number in rows of 700
// columns, else one a row, three for k > 64 (384 x 785 x 785, k = 64: 1.9 per row 289 -> 203, 0.7 233 -> 201; k = 128, 6.4 437 -> 348, 1.3
// 282 -> 238; 200 x 333 x 333, k = 64, 1 per row 32 -> 28, k = 128, 3.8 47 -> 40; 300 x 500 x 500, k = 64, 1.9 89 -> 79, 0.7 67 / 76, k = 128,
// 1.9 97 / 105; rows of fewer than 256 columns stay with the row kernel: 384 x 197 x 197, k = 64, 6.6 per row 34 / 44).
template <typename T>
bool smallk_wanted(const SpmmParams& p, int batch) {
  constexpr int kMax = 16 / (int)sizeof(T);
  if (!smallk_fits<T>(p)) return false;
  const double per_row = (double)p.nnz / std::max(p.m, 1);
  const bool whole = smallk_aligned<T>(p), large = (double)batch * p.m * p.n >= 8e6;
  const bool wide = p.n >= kWave * kMax / (sizeof(T) == 2 ? 2 : 1);
  if (smallk_by_lines<T>(p) && (double)batch * p.m * p.n >= 2e7 && p.m >= 2 * p.k && per_row >= (p.n >= 700 ? 0.0 : p.k > 64 ? 3.0 : 1.0)) return true;
  if (wide && p.k <= 64 && p.m >= 8 * p.k) return per_row >= (whole ? 1.8 : 2.5);
  if (wide && p.k > 64 && p.m >= 32 * p.k && per_row >= 4.0) return true;
  if (!large) return false;
  if (sizeof(T) == 2 && matrix_core_kernel_applies<T>(p, batch)) return false;
  if (sizeof(T) == 2 && p.n % 8 != 0 && p.n < kWave * kMax / 2) return per_row >= 1.5;
  if (!wide || p.m < 2 * p.k) return false;
  return per_row >= (p.k <= 64 ? 8.0 : sizeof(T) == 2 ? 2.5 : 8.0);
}

// Rows per wavefront of the few-columns kernels, `tiles` column tiles (of all batch entries) and WAVES wavefronts per workgroup.
template <int WAVES>
int smallk_rows(const SpmmParams& p, long long tiles) {
  int rows;
  if constexpr (WAVES == 8) {
    // two workgroups per CU cover for each other's tile load: enough rows for it to be a fraction of what they write
    rows = std::min(64, std::max(16, p.k / 2));
    while (rows > 4 && (long long)ceil_div(p.m, WAVES * rows) * tiles < 1024) rows >>= 1;
  } else {
    // One per CU: rows are dealt evenly to as many as finish first, rounds of workgroups times the rows of a wavefront plus
    // four, about what the tile load costs.  (384 x 785 x 785: one workgroup with 50 rows per wavefront, 301 us, not one of 512
    // rows and one of 273, 328; 96 x 1536 x 1536: four of 24 rows, not two of 48, which are 2.25 rounds: 191 / 227.)
    double least = 0;
    rows = 0;
    for (int blocks = ceil_div(p.m, WAVES * 64), upto = std::max(blocks, ceil_div(p.m, WAVES * 4)); blocks <= upto && blocks < 65536; ++blocks) {
      const int r = ceil_div(p.m, WAVES * blocks);
      const double cost = (double)ceil_div(blocks * tiles, 256) * (r + 4);
      if (rows == 0 || cost < least) rows = r, least = cost;
      if (blocks >= 64) blocks += blocks / 16;   // (long operands: not every count)
    }
  }
  return rows;
}

template <typename T, typename IT, bool RAGGED, int WAVES, int MOST, bool PLAIN, bool SCALAR = false>
int launch_smallk_one(const SpmmParams& p, int batch, int tiles_n, int lds, hipStream_t stream) {
  constexpr int kMax = 16 / (int)sizeof(T);
  if constexpr (!SCALAR && std::is_same<T, float>::value && std::is_same<IT, int>::value) {
    if (p.nnz > (long long)kSmallkScalarRows * p.m) return launch_smallk_one<T, IT, RAGGED, WAVES, MOST, PLAIN, true>(p, batch, tiles_n, lds, stream);
  }
  const int rows = smallk_rows<WAVES>(p, (long long)tiles_n * batch);
  auto kern = spmm_smallk_kernel<T, IT, kMax, RAGGED, WAVES, MOST, PLAIN, SCALAR>;
  if (lds > 64 * 1024) {
    static thread_local bool raised = false;  // per instantiation
    if (!raised) {
      if (int rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024),
                             "hipFuncSetAttribute(LDS size)"))
        return rc;
      raised = true;
    }
  }
  dim3 grid(ceil_div(p.m, WAVES * rows), tiles_n, batch);
  note_kernel("spmm_smallk_kernel<%s, %s, %d, %s, %d, %d>", type_name<T>(), type_name<IT>(), kMax, RAGGED ? "true" : "false", WAVES, MOST);
  hipLaunchKernelGGL(kern, grid, dim3(WAVES * kWave), lds, stream, p, rows);
  return check_hip(hipGetLastError(), "spmm (few columns) launch");
}

// Two vectors per lane where the output is wider than one and two of every dense row fit the LDS.
template <int WAVES>
int launch_smallk_lines(const SpmmParams& p, int batch, const SmallkLines& t, int lds, hipStream_t stream) {
  auto kern = spmm_smallk_kernel_lines<WAVES>;
  static thread_local bool raised = false;  // per instantiation
  if (!raised) {
    if (int rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024),
                           "hipFuncSetAttribute(LDS size)"))
      return rc;
    raised = true;
  }
  const int rows = smallk_rows<WAVES>(p, (long long)(t.tiles + 1) * batch);
  note_kernel("spmm_smallk_kernel_lines<%d> (%d tiles of %d columns, %d at the edges)", WAVES, t.tiles, t.width, t.rest);
  hipLaunchKernelGGL(kern, dim3(ceil_div(p.m, WAVES * rows), t.tiles + 1, batch), dim3(WAVES * kWave), lds, stream, p, t, rows);
  return check_hip(hipGetLastError(), "spmm (few columns, whole lines) launch");
}

template <typename T, typename IT>
int launch_smallk(const SpmmParams& p, int batch, hipStream_t stream) {
  constexpr int kMax = 16 / (int)sizeof(T);
  const bool plain = !p.bias && !p.relu && !p.accumulate;
  if constexpr (std::is_same<T, float>::value && std::is_same<IT, int>::value) {
    if (smallk_by_lines<T>(p)) {
      const SmallkLines t = smallk_lines(p.n, p.k);
      const int lds = smallk_lines_lds(t, p.k);
      return smallk_waves(lds) == 8 ? launch_smallk_lines<8>(p, batch, t, lds, stream) : launch_smallk_lines<16>(p, batch, t, lds, stream);
    }
  }
  const int most = plain && p.n > kWave * kMax && 2 * p.k <= kSmallKMax ? 2 : 1;
  const SmallkTiles t = smallk_tiles(p.n, most, kMax);
  const int last = smallk_row_bytes(t.nv, t.single, sizeof(T)), lds = p.k * (t.tiles > 1 ? std::max(last, smallk_row_bytes(most, false, sizeof(T))) : last);
  const bool eight = smallk_waves(lds) == 8;
  auto pick = [&](auto ragged) {
    constexpr bool R = decltype(ragged)::value;
    if (most == 2) return eight ? launch_smallk_one<T, IT, R, 8, 2, true>(p, batch, t.tiles, lds, stream) : launch_smallk_one<T, IT, R, 16, 2, true>(p, batch, t.tiles, lds, stream);
    if (plain) return eight ? launch_smallk_one<T, IT, R, 8, 1, true>(p, batch, t.tiles, lds, stream) : launch_smallk_one<T, IT, R, 16, 1, true>(p, batch, t.tiles, lds, stream);
    return eight ? launch_smallk_one<T, IT, R, 8, 1, false>(p, batch, t.tiles, lds, stream) : launch_smallk_one<T, IT, R, 16, 1, false>(p, batch, t.tiles, lds, stream);
  };
  return smallk_aligned<T>(p) ? pick(std::false_type{}) : pick(std::true_type{});
}

template <typename T, typename IT, int VEC, int LPG>
int launch_wpr(const SpmmParams& p, int batch, int wpr, int nt, hipStream_t stream) {
  if constexpr (LPG == kWave && VEC * sizeof(T) == 16) {
    // full-width tiles: a wave may cover 2 adjacent tiles (4 waves per row only)
    if (nt == 2 && wpr == 4) return launch_one<T, IT, VEC, LPG, 4, 2>(p, batch, stream);
  }
  switch (wpr) {
    case 1: return launch_one<T, IT, VEC, LPG, 1>(p, batch, stream);
    case 4: return launch_one<T, IT, VEC, LPG, 4>(p, batch, stream);
    case 8: return launch_one<T, IT, VEC, LPG, 8>(p, batch, stream);
  }
  return fail(IEX_ERR_BAD_ARGUMENT, "spmm: waves-per-row must be 1, 4 or 8 (got %d)", wpr);
}

// ---- row kernel with wavefronts per row that follow the row's own length ---------------------------------
template <typename T, typename IT, int VEC, int LPG>
__global__ __launch_bounds__(kRowsWaves * kWave) void spmm_rows_kernel(SpmmParams p, RowClasses rc) {
  __shared__ float red[spmm_rows_lds_floats<VEC>()];
  spmm_rows_block<T, IT, VEC, LPG>(p, rc, blockIdx.x, blockIdx.y, blockIdx.z, red);
}

// From the histogram of row lengths (hist[j] = rows with more than 64 << j nonzeros, j = 0 .. 15) to the five ranges
// of row slots.  A wavefront should get at most `rounds` chunks of 64 nonzeros (a power of two, 1 .. 16): a row of c
// chunks gets the smallest power of two >= c / rounds wavefronts, at most 16.  `rounds` follows the work per
// wavefront slot when every row is cut that way: with fewer chunks than the chip holds wavefronts (256 CUs x 16) one
// chunk per wavefront is the shortest critical path; with more, cutting finer only adds partial sums.
inline RowClasses row_classes(const SpmmParams& p, const int* hist, int tiles, int force_log2_rounds_plus_1, int* rounds_out) {
  const double chunks = (double)p.nnz / kWave * tiles;
  int r = 0;   // log2(rounds)
  while (r < 4 && chunks / (1 << r) > 256.0 * 16) ++r;
  if (force_log2_rounds_plus_1 > 0) r = std::min(force_log2_rounds_plus_1 - 1, 8);
  auto rows_over = [&](int log2_chunks) { return log2_chunks > 15 ? 0 : std::min(p.m, std::max(0, hist[log2_chunks])); };
  RowClasses rc;
  // class c: 16 >> c wavefronts; a row belongs to class c or an earlier one when it has more than (8 >> c) * rounds chunks
  rc.first_row[0] = 0;
  int before = 0;
  for (int c = 0; c < 4; ++c) {
    const int upto = std::max(before, rows_over(3 - c + r));   // rows with more than 64 << (3 - c + r) nonzeros
    rc.first_row[c + 1] = upto;
    before = upto;
  }
  rc.first_row[5] = p.m;
  rc.first_block[0] = 0;
  for (int c = 0; c < 5; ++c) rc.first_block[c + 1] = rc.first_block[c] + ceil_div(rc.first_row[c + 1] - rc.first_row[c], 1 << c);
  rc.log2_rounds = r;
  *rounds_out = 1 << r;
  return rc;
}

template <typename T, typename IT, int VEC, int LPG>
int launch_rows_one(const SpmmParams& p, int batch, const int* hist, int rounds_code, hipStream_t stream) {
  const int tiles = ceil_div(p.n, LPG * VEC);
  int rounds = 1;
  const RowClasses rc = row_classes(p, hist, tiles * batch, rounds_code, &rounds);
  note_kernel("spmm_rows_kernel<%s, %s, %d, %d> (rows by 16/8/4/2/1 waves: %d/%d/%d/%d/%d, %d chunks per wave)", type_name<T>(), type_name<IT>(), VEC, LPG,
              rc.first_row[1], rc.first_row[2] - rc.first_row[1], rc.first_row[3] - rc.first_row[2], rc.first_row[4] - rc.first_row[3],
              rc.first_row[5] - rc.first_row[4], rounds);
  hipLaunchKernelGGL((spmm_rows_kernel<T, IT, VEC, LPG>), dim3(rc.first_block[5], tiles, batch), dim3(kRowsWaves * kWave), 0, stream, p, rc);
  return check_hip(hipGetLastError(), "spmm (rows by length) launch");
}

template <typename T, typename IT>
int launch_rows(const SpmmParams& p, int batch, int lpg, const int* hist, int rounds_code, hipStream_t stream) {
  constexpr int kMax = 16 / (int)sizeof(T);
  switch (lpg) {
    case 8: return launch_rows_one<T, IT, kMax, 8>(p, batch, hist, rounds_code, stream);
    case 16: return launch_rows_one<T, IT, kMax, 16>(p, batch, hist, rounds_code, stream);
    case 32: return launch_rows_one<T, IT, kMax, 32>(p, batch, hist, rounds_code, stream);
    default: return launch_rows_one<T, IT, kMax, 64>(p, batch, hist, rounds_code, stream);
  }
}

// ---- ... by workgroups of four: a wavefront per row, four for the long ones ---------------------------------
// Bound like the row kernel by the gathers' way from L2 into the CUs and, where rows are uneven, by the chain of the longest one.  A whole row per
// wavefront needs no partial sums and lets the wavefronts of an XCD walk through the dense operand's rows together (2048 x 8192, even rows of 409,
// n = 512 fp32: 125 us by four wavefronts a row, 68 by one); four for a long row shorten its chain without the cost for the others.
// (Registers for four wavefronts per SIMD, six with full fp32 tiles: what a row by one wavefront has.)
template <typename T, typename IT, int VEC, int LPG, bool RAGGED>
__global__ __launch_bounds__(4 * kWave, LPG < kWave ? 4 : sizeof(T) == 2 ? 4 : 6) void spmm_rows_kernel4(SpmmParams p, LongRows lr) {
  __shared__ float red[spmm_lds_floats<VEC, 4>()];
  spmm_long_rows_block<T, IT, VEC, LPG, RAGGED>(p, lr, blockIdx.x, blockIdx.y, blockIdx.z, red);
}

template <typename T, typename IT, int LPG, bool RAGGED>
int launch_long_rows_one(const SpmmParams& p, int batch, const LongRows& lr, hipStream_t stream) {
  constexpr int kMax = 16 / (int)sizeof(T);
  note_kernel("spmm_rows_kernel4<%s, %s, %d, %d, %s> (%d rows by four waves)", type_name<T>(), type_name<IT>(), kMax, LPG, RAGGED ? "true" : "false", lr.long_rows);
  hipLaunchKernelGGL((spmm_rows_kernel4<T, IT, kMax, LPG, RAGGED>), dim3(lr.long_rows + ceil_div(p.m - lr.long_rows, 4), ceil_div(p.n, LPG * kMax), batch),
                     dim3(4 * kWave), 0, stream, p, lr);
  return check_hip(hipGetLastError(), "spmm (long rows) launch");
}

template <typename T, typename IT>
int launch_long_rows(const SpmmParams& p, int batch, int lpg, bool ragged, const int* hist, int log2_chunks, hipStream_t stream) {
  const LongRows lr{std::min(p.m, std::max(0, hist[log2_chunks])), kWave << log2_chunks};
  if (ragged) return launch_long_rows_one<T, IT, kWave, true>(p, batch, lr, stream);
  switch (lpg) {
    case 8: return launch_long_rows_one<T, IT, 8, false>(p, batch, lr, stream);
    case 16: return launch_long_rows_one<T, IT, 16, false>(p, batch, lr, stream);
    case 32: return launch_long_rows_one<T, IT, 32, false>(p, batch, lr, stream);
    default: return launch_long_rows_one<T, IT, kWave, false>(p, batch, lr, stream);
  }
}

// How the wavefronts go to the rows of a pattern whose row lengths are known: log2(limit / 64) of the kernel above, or one of the names below
// (kRowsAsBefore: by the mean alone, or by 16).  Even = no row longer than two to four times the mean.  MI355X, us, four wavefronts a row / one / the kernel above
// at its limit (* = 16 wavefronts a workgroup, one chunk each):
//  several nonzeros per gather, even: a row to a wavefront from 2000 rows up; long rows only where the workgroups fill whole rounds of the CUs (level)
//   11008 x 4096 at 97 %, n = 64 fp16 20.8 / 11.6 / 11.9, fp32 18.2 / 17.7 / 15.9, at 90 % n = 128 fp32 82 / 79 / 78;  6000 x 3000 at 90 %, n = 128 41 / 34 / 36
//   1024 x 2000 at 90 %, n = 128 fp32 7.3 / 8.9 / 8.3, 8.3*;  n = 256 fp16 8.0 / 9.1 / 8.6, 9.7*;  not level: 4552 x 3880 at 80 %, n = 80 fp16 39 / 44 / -
//  ... uneven (geometric lengths)
//   11008 x 4096 at 97 %, n = 64 fp16 20.8 / 14.5 / 12.0;  6000 x 3000 at 90 %, n = 32 fp16 16.4 / 31 / 12.9;  4096 x 4096 at 97 %, n = 128 fp32 16.2 / 32.5 / 14.3, 18.4*
//   1024 x 2000 at 90 %, n = 128 fp32 16.3 / 45 / 15.3, 12.3*;  4096 x 4096 at 90 %, n = 64 fp32 21.6 / 53 / 22 - 24;  3752 x 416, 11 a row, n = 24 fp16 - / 5.2 / 5.4
//  one nonzero per gather, even
//   4096 x 4096 at 90 %, n = 256 fp32 61 / 60 / 60;  2000 x 4096 at 97 %, n = 512 26 / 24 / -;  4096 x 1000 at 97 %, n = 512 fp16 12.7 / 9.0 / -;  512 x 8192 at 95 %, n = 1024
//   fp32 65 / 43 / -;  424 x 1104 at 93 %, n = 1540 15.3 / 16.1 / -;  not level: 4872 x 5176 at 97 %, n = 176 29 / 32 / -
//  ... uneven
//   4096 x 4096 at 95 %, n = 512 fp32 68 / 154 / 66, n = 2048 247 / 396 / 239;  98 %, n = 512 34 / 65 / 33, fp16 n = 2048 74 / 87 / 66;  10000 x 600 at 90 %, n = 256 25 / 30 / 23
//   4096 x 4096 at 90 %, n = 256 fp32 68 / 168 / 67 - 75;  256 x 4096 at 90 %, n = 1024 136 / - / -, 57*;  512 x 1024 at 90 %, n = 512 16.2 / - / -, 11.7*;
//   2048 x 1024 at 90 %, n = 256 15.6 / - / -, 18.1*;  1024 x 1024 at 90 %, n = 1024 fp16 19.4 / - / -, 21.6*
// The limit grows with the rows, which are what a long row's chain hides behind.
constexpr int kRowsAsBefore = -1, kRowsOneWave = -2, kRowsFourWaves = -3, kRowsSixteenWaves = -4;
inline int rows_by_histogram(const SpmmParams& p, int batch, const int* hist, int elem_size, int lpg, int wpr) {
  const double mean = (double)p.nnz / std::max(p.m, 1), rows = (double)p.m * batch;
  int twice = 0;
  while (twice < 15 && (kWave << twice) < 2 * mean) ++twice;
  const bool even = hist[twice] <= 0;
  const int tiles = ceil_div(p.n, lpg * 16 / elem_size);
  const double groups = rows * tiles / (4 * 256);
  const bool level = groups >= 0.96 * std::ceil(groups);
  double ratio = 0.8 + rows / 4500;
  if (lpg == kWave) {
    if (even) return wpr == 4 && groups >= 1.9 && level && (rows >= 1900 || mean >= 250) ? kRowsOneWave : kRowsAsBefore;
    if (mean < 24) return kRowsAsBefore;
    if (wpr != 1 && !(elem_size == 2 && rows >= 4000 && mean <= 128)) {
      if (rows < 256) return kRowsAsBefore;   // (not measured below)
      if (mean >= 250 ? rows <= 1500 : mean >= 80 && tiles >= 2 && rows * tiles <= (elem_size == 4 ? 2100 : 1100)) return kRowsSixteenWaves;
      return kRowsAsBefore;
    }
    if (elem_size == 4) ratio = std::max(hist[twice] < 0.01 * p.m ? 2.0 : 0.65, rows / 5500);
  } else {
    if (even) return wpr == 1 ? kRowsAsBefore : rows < 2000 || (mean > 250 && !level) || (mean > 500 && rows < 6000) ? kRowsFourWaves : elem_size == 4 ? twice : kRowsOneWave;
    if (mean < 16 || (rows < 2000 && mean >= 100) || (rows < 5500 && mean > 250)) return kRowsAsBefore;
  }
  return std::min(15, std::max(0, (int)std::lround(std::log2(std::min(ratio, 4.0) * mean / kWave))));
}

// Wavefronts per row of the kernel for narrow ragged rows (spmm_ragged.hip), 0 = a single nonzero per gather stays ahead: rows with few nonzeros leave it nothing to
// share out, few rows nothing to fill the chip with.  Even rows by one wavefront each where there are many (the histogram tells: none longer than two to four
// times the mean), rows of several hundred nonzeros and uneven ones by four.  MI355X, us, one nonzero per gather / one wavefront a row / four:
//   even     9904 x 1000 at 97 %, n = 138 fp16, 31 a row 20.6 / 12.0 / 26.3;  5137 x 1040, n = 52, 97 a row 10.6 / 7.1 / 11.5;  10704 x 2846, n = 14, 302 43 / 20 / 27;
//            fp32 8616 x 1800, n = 67, 365 84 / 57 / 60;  1064 x 3912, n = 177, 223 11.9 / 21.4 / 14.0;  752 x 792, n = 95, 82 4.8 / 5.7 / 5.0;  2558 x 1400, n = 31, 137 8.1 / 8.7 / 8.0
//   uneven   1632 x 3347, n = 68, 418 29 / 41 / 16.5;  4248 x 800, n = 67, 89 15.8 / 21.9 / 12.7;  8768 x 3344, n = 12, 1000 87 / 64 / 50;  690 x 392, n = 246 fp32, 46 6.3 / 14.8 / 6.3
inline int ragged_narrow_waves(const SpmmParams& p, int batch, const int* hist, int elem_size) {
  const double mean = (double)p.nnz / std::max(p.m, 1), rows = (double)p.m * batch;
  bool even = false;
  if (hist) {
    int j = 0;
    while (j < 15 && (kWave << j) < 2 * mean) ++j;
    even = hist[j] == 0;
  }
  if (elem_size == 2 && p.n % 2 != 0 && mean > 1000) return 0;   // (16-byte gathers at odd addresses: 4086 x 8048 at 71 %, n = 9 118 / - / 189)
  const double groups = rows / (4 * 256);
  if (even && mean >= 24 && rows >= 2700 && (mean <= 150 || groups >= 0.96 * std::ceil(groups))) return 1;
  if (p.n > 256 / elem_size) return 0;   // (two nonzeros per gather: 568 x 2832 at 71 %, n = 137 fp16 21 / - / 31)
  const bool odd = elem_size == 2 && p.n % 2 != 0;
  if (mean >= 250) return odd && even && rows >= 2700 ? 0 : 4;
  return hist && !even && mean >= (odd ? 150 : 80) ? 4 : 0;
}

// ---- LDS-staged variant -----------------------------------------------------------------
template <typename T, typename IT, int VEC, int RPW>
__global__ __launch_bounds__(kLdsThreads, 4) void spmm_lds_kernel(SpmmParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  spmm_lds_block<T, IT, VEC, RPW>(p, blockIdx.x, blockIdx.y, blockIdx.z, smem);
}

template <typename T, typename IT, int VEC, int RPW>
int launch_lds_one(const SpmmParams& p, int batch, hipStream_t stream) {
  dim3 grid(ceil_div(p.m, kLdsWaves * RPW), ceil_div(p.n, kWave * VEC), batch);
  note_kernel("spmm_lds_kernel<%s, %s, %d, %d>", type_name<T>(), type_name<IT>(), VEC, RPW);
  hipLaunchKernelGGL((spmm_lds_kernel<T, IT, VEC, RPW>), grid, dim3(kLdsThreads), kLdsTileBytes, stream, p);
  return check_hip(hipGetLastError(), "spmm (LDS-staged) launch");
}

template <typename T, typename IT, int VEC>
int launch_lds_rpw(const SpmmParams& p, int batch, int rpw, hipStream_t stream) {
  switch (rpw) {
    case 2: return launch_lds_one<T, IT, VEC, 2>(p, batch, stream);
    case 4: return launch_lds_one<T, IT, VEC, 4>(p, batch, stream);
    case 8:
      // 8 rows x 8 accumulators per lane would spill at 4 waves per SIMD: 4 rows per wave then
      if constexpr (VEC < 8) return launch_lds_one<T, IT, VEC, 8>(p, batch, stream);
      else return launch_lds_one<T, IT, VEC, 4>(p, batch, stream);
  }
  return fail(IEX_ERR_BAD_ARGUMENT, "spmm: rows-per-wave of the LDS-staged variant must be 2, 4 or 8 (got %d)", rpw);
}

// ---- matrix-core variant (fp16 / bf16) ----------------------------------------------------
template <bool BF16, typename IT, int LPR>
__global__ __launch_bounds__(kMfmaThreads, 2) void spmm_mfma_kernel(SpmmParams p, int tiles_m) {
  extern __shared__ __align__(16) unsigned char smem[];
  // consecutive workgroups walk the row blocks of one column panel of the dense operand
  spmm_mfma_block<BF16, IT, LPR>(p, blockIdx.x % tiles_m, blockIdx.x / tiles_m, blockIdx.y, smem);
}

template <typename T, typename IT, int LPR>
int launch_mfma_one(const SpmmParams& p, int batch, hipStream_t stream) {
  constexpr bool kBf16 = std::is_same<T, __hip_bfloat16>::value;
  const int tiles_m = ceil_div(p.m, kMfmaBM), tiles_n = ceil_div(p.n, kMfmaBN);
  auto kernel = spmm_mfma_kernel<kBf16, IT, LPR>;
  static thread_local bool raised = false;  // more than 64 KB of dynamic LDS needs the attribute (per instantiation)
  if (!raised) {
    if (int rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, kMfmaLdsBytes),
                           "hipFuncSetAttribute(LDS size)"))
      return rc;
    raised = true;
  }
  note_kernel("spmm_mfma_kernel<%s, %s, %d>", kBf16 ? "true" : "false", type_name<IT>(), LPR);
  hipLaunchKernelGGL(kernel, dim3(tiles_m * tiles_n, batch), dim3(kMfmaThreads), kMfmaLdsBytes, stream, p, tiles_m);
  return check_hip(hipGetLastError(), "spmm (matrix-core) launch");
}

template <typename T, typename IT>
int launch_mfma(const SpmmParams& p, int batch, int lpr, hipStream_t stream) {
  if constexpr (sizeof(T) == 2) {
    switch (lpr) {
      case 8: return launch_mfma_one<T, IT, 8>(p, batch, stream);
      case 16: return launch_mfma_one<T, IT, 16>(p, batch, stream);
    }
    return fail(IEX_ERR_BAD_ARGUMENT, "spmm: lanes-per-row of the matrix-core variant must be 8 or 16 (got %d)", lpr);
  } else {
    return fail(IEX_ERR_UNSUPPORTED, "spmm: the matrix-core variant handles fp16 and bf16 only");
  }
}

template <bool BF16, typename IT, int W, int BKA>
__global__ __launch_bounds__(kMfma2Threads, 2) void spmm_mfma2_kernel(SpmmParams p, int tiles_m) {
  extern __shared__ __align__(16) unsigned char smem[];
  spmm_mfma2_block<BF16, IT, W, BKA>(p, blockIdx.x % tiles_m, blockIdx.x / tiles_m, blockIdx.y, smem);
}

template <typename T, typename IT, int W, int BKA = 128>
int launch_mfma2_one(const SpmmParams& p, int batch, hipStream_t stream) {
  constexpr bool kBf16 = std::is_same<T, __hip_bfloat16>::value;
  constexpr int kMfma2LdsBytes = spmm_mfma2_lds_bytes<BKA>();
  const int tiles_m = ceil_div(p.m, kMfmaBM), tiles_n = ceil_div(p.n, kMfma2BN);
  auto kernel = spmm_mfma2_kernel<kBf16, IT, W, BKA>;
  static thread_local bool raised = false;
  if (!raised) {
    if (int rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, kMfma2LdsBytes),
                           "hipFuncSetAttribute(LDS size)"))
      return rc;
    raised = true;
  }
  note_kernel("spmm_mfma2_kernel<%s, %s, %d, %d>", kBf16 ? "true" : "false", type_name<IT>(), W, BKA);
  hipLaunchKernelGGL(kernel, dim3(tiles_m * tiles_n, batch), dim3(kMfma2Threads), kMfma2LdsBytes, stream, p, tiles_m);
  return check_hip(hipGetLastError(), "spmm (matrix-core, 8 waves) launch");
}

template <typename T, typename IT>
int launch_mfma2(const SpmmParams& p, int batch, int windows, hipStream_t stream) {
  if constexpr (sizeof(T) == 2) {
    switch (windows) {
      case 1: return launch_mfma2_one<T, IT, 1>(p, batch, stream);
      case 2: return launch_mfma2_one<T, IT, 2>(p, batch, stream);
      case 4: return launch_mfma2_one<T, IT, 4>(p, batch, stream);
      case 5: return launch_mfma2_one<T, IT, 5>(p, batch, stream);
    }
    return fail(IEX_ERR_BAD_ARGUMENT, "spmm: windows of the matrix-core variant must be 1, 2, 4 or 5 (got %d)", windows);
  } else {
    return fail(IEX_ERR_UNSUPPORTED, "spmm: the matrix-core variant handles fp16 and bf16 only");
  }
}

template <bool BF16, typename IT, int W>
__global__ __launch_bounds__(kMfma3Threads, 2) void spmm_mfma3_kernel(SpmmParams p, int tiles_m) {
  extern __shared__ __align__(16) unsigned char smem[];
  spmm_mfma3_block<BF16, IT, W>(p, blockIdx.x % tiles_m, blockIdx.x / tiles_m, blockIdx.y, smem);
}

template <typename T, typename IT, int W>
int launch_mfma3_one(const SpmmParams& p, int batch, hipStream_t stream) {
  constexpr bool kBf16 = std::is_same<T, __hip_bfloat16>::value;
  const int tiles_m = ceil_div(p.m, kMfmaBM), tiles_n = ceil_div(p.n, kMfma3BN);
  auto kernel = spmm_mfma3_kernel<kBf16, IT, W>;
  static thread_local bool raised = false;
  if (!raised) {
    if (int rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, spmm_mfma3_lds_bytes()),
                           "hipFuncSetAttribute(LDS size)"))
      return rc;
    raised = true;
  }
  note_kernel("spmm_mfma3_kernel<%s, %s, %d>", kBf16 ? "true" : "false", type_name<IT>(), W);
  hipLaunchKernelGGL(kernel, dim3(tiles_m * tiles_n, batch), dim3(kMfma3Threads), spmm_mfma3_lds_bytes(), stream, p, tiles_m);
  return check_hip(hipGetLastError(), "spmm (matrix-core, direct loads) launch");
}

template <typename T, typename IT>
int launch_mfma3(const SpmmParams& p, int batch, int windows, hipStream_t stream) {
  if constexpr (sizeof(T) == 2) {
    if (windows == 1) return launch_mfma3_one<T, IT, 1>(p, batch, stream);
    if (windows == 2) return launch_mfma3_one<T, IT, 2>(p, batch, stream);
    if (windows == 4) return launch_mfma3_one<T, IT, 4>(p, batch, stream);
    return fail(IEX_ERR_BAD_ARGUMENT, "spmm: windows of the direct-load matrix-core variant must be 1, 2 or 4 (got %d)", windows);
  } else {
    return fail(IEX_ERR_UNSUPPORTED, "spmm: the matrix-core variant handles fp16 and bf16 only");
  }
}

// ---- matrix-core variant, fp32 ---------------------------------------------------------------
// arrangement code = MFMA tile height and how the 4 multiplying waves split the C tile:
//   1 = 32 x 64 (4 k slices)    2 = 32 x 128 as 2 x 64 columns (2 k slices)    4 = 32 x 128 (4 k slices)
//   5 = 16 x 64 (4 k slices)    6 = 16 x 128 as 2 x 64 columns (2 k slices)
template <int MT, int NJ, int WAVES_N, bool SPLIT, bool FAR>
__global__ __launch_bounds__(kF32Threads + (SPLIT ? MT * 8 : 0), 2) void spmm_mfma_f32_kernel(SpmmParams p, int tiles_m) {
  extern __shared__ __align__(16) unsigned char smem[];
  spmm_mfma_f32_block<MT, NJ, WAVES_N, SPLIT, FAR>(p, blockIdx.x % tiles_m, blockIdx.x / tiles_m, blockIdx.y, smem);
}

template <int MT, int NJ, int WAVES_N, bool SPLIT, bool FAR>
int launch_mfma_f32_one(const SpmmParams& p, int batch, hipStream_t stream) {
  constexpr int kBN = MT * NJ * WAVES_N;
  const int tiles_m = ceil_div(p.m, MT), tiles_n = ceil_div(p.n, kBN);
  constexpr int kLds = spmm_mfma_f32_lds_bytes<MT, NJ, WAVES_N>();
  note_kernel("spmm_mfma_f32_kernel<%d, %d, %d, %s, %s>", MT, NJ, WAVES_N, SPLIT ? "true" : "false", FAR ? "true" : "false");
  hipLaunchKernelGGL((spmm_mfma_f32_kernel<MT, NJ, WAVES_N, SPLIT, FAR>), dim3(tiles_m * tiles_n, batch),
                     dim3(kF32Threads + (SPLIT ? MT * 8 : 0)), kLds, stream, p, tiles_m);
  return check_hip(hipGetLastError(), "spmm (matrix-core, fp32) launch");
}

template <int MT, int NJ, int WAVES_N>
int launch_mfma_f32_roles(const SpmmParams& p, int batch, bool split, hipStream_t stream) {
  // what the kernel's 32-bit byte offsets reach (the dense operand's: up to a few chunks past its end)
  if (p.nnz >= 1 << 30 || ((long long)p.k + 1024) * p.n >= 1 << 30) return launch_mfma_f32_one<MT, NJ, WAVES_N, true, true>(p, batch, stream);
  return split ? launch_mfma_f32_one<MT, NJ, WAVES_N, true, false>(p, batch, stream) : launch_mfma_f32_one<MT, NJ, WAVES_N, false, false>(p, batch, stream);
}

inline int launch_mfma_f32(const SpmmParams& p, int batch, int arrangement, bool split, hipStream_t stream) {
  switch (arrangement) {
    case 1: return launch_mfma_f32_roles<32, 2, 1>(p, batch, split, stream);
    case 2: return launch_mfma_f32_roles<32, 2, 2>(p, batch, split, stream);
    case 4: return launch_mfma_f32_roles<32, 4, 1>(p, batch, split, stream);
    case 5: return launch_mfma_f32_roles<16, 4, 1>(p, batch, split, stream);
    case 6: return launch_mfma_f32_roles<16, 4, 2>(p, batch, split, stream);
  }
  return fail(IEX_ERR_BAD_ARGUMENT, "spmm: arrangement of the fp32 matrix-core variant must be 1, 2, 4, 5 or 6 (got %d)", arrangement);
}

// out = out + aux, or out * silu(aux), over n 16-bit elements: the epilogue of the products that have none of their own.
template <bool BF16>
__global__ __launch_bounds__(256) void combine_kernel(size_t n, const uint16_t* aux, int mode, uint16_t* out) {
  struct alignas(2) Any { uint16_t v[8]; };
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 8;
  auto one = [&](uint16_t o, uint16_t a) {
    const float x = f16_to_32(o, BF16), y = f16_to_32(a, BF16);
    return f32_to_16(mode == kGemmAdd ? x + y : x * (y / (1.f + __expf(-y))), BF16);
  };
  if (i + 8 <= n) {
    Any o = *reinterpret_cast<const Any*>(out + i);
    const Any a = *reinterpret_cast<const Any*>(aux + i);
#pragma unroll
    for (int e = 0; e < 8; ++e) o.v[e] = one(o.v[e], a.v[e]);
    *reinterpret_cast<Any*>(out + i) = o;
  } else {
    for (size_t j = i; j < n; ++j) out[j] = one(out[j], aux[j]);
  }
}

struct Choice {
  int wpr = 0;      // wavefronts per row of the row kernel
  bool wpr_forced = false;
  int variant = 0;  // 0 = choose, 1 = row kernel, 2 = LDS-staged kernel, 3 / 4 = matrix-core kernels (16-bit), 5 = (fp32)
  int rpw = 0;      // rows per wavefront of the LDS-staged kernel (0 = choose)
  int nt = 0;       // adjacent column tiles per wavefront of the row kernel (0 = choose)
  int lpg = 0;      // lanes per nonzero of the row kernel: 8, 16, 32 or 64 (0 = choose)
  void* ws = nullptr;   // caller's workspace for the dense form of A (variant 7), may be null
  size_t ws_bytes = 0;
  bool any_order = false;   // columns of a row in any order, possibly repeated: families 1 and 8 only
  const int* hist = nullptr;   // host: rows with more than 64 << j nonzeros, j = 0 .. 15 (iex_spmm_sched), may be null
  bool* aux_done = nullptr;    // set by a path whose own epilogue takes the auxiliary operand
  bool beside_gather = false;  // the launch shares the chip with a gather-bound one (IEX_SPMM_BESIDE_GATHER_KERNEL)
};

// The LDS-staged kernel needs a full-width tile (64 lanes x VEC, VEC the full or half 128-bit
// vector) and pays off when the rows of a workgroup share dense rows often enough:
// gathers saved per dense row staged = density * rows per workgroup.
template <typename T>
bool lds_variant(const SpmmParams& p, int batch, const Choice& ch, int& vec, int& rpw) {
  constexpr int kMax = 16 / (int)sizeof(T);
  vec = kMax;
  auto fits = [&](int v) {
    return p.n % v == 0 && kWave * v <= p.n && aligned(p.dense, sizeof(T) * v) && aligned(p.out, sizeof(T) * v);
  };
  if (!fits(vec)) vec = kMax / 2;
  if (!fits(vec)) return false;
  const long long tiles = (long long)ceil_div(p.n, kWave * vec) * batch;
  rpw = ch.rpw;
  if (rpw == 0) {
    rpw = 8;  // largest rows-per-wave that still gives every CU two workgroups
    while (rpw > 2 && (long long)ceil_div(p.m, kLdsWaves * rpw) * tiles < 512) rpw >>= 1;
  }
  if (ch.variant == 2) return true;
  if (ch.variant == 1) return false;
  // Measured on MI355X: the staged kernel wins when the rows of a workgroup reuse a staged
  // dense row a dozen times or more (2:4 weights: 4.5 -> 3.6 ms at 4096x4096, n = 8192), and
  // from a reuse of 4 when the slice of the dense operand one column tile touches (k rows of
  // a 64-lane tile) outgrows an XCD's 4 MB L2 (k = 11008: 10.8 -> 4.9 ms).  It loses on small
  // problems (fewer than two workgroups per CU: per-stage barriers expose row-length imbalance)
  // and at low reuse (90 % sparsity: 0.67 -> 0.90 ms).
  const double density = (p.m > 0 && p.k > 0) ? (double)p.nnz / ((double)p.m * p.k) : 0.0;
  const int eff_rpw = (vec * (int)sizeof(T) == 16 && sizeof(T) == 2 && rpw == 8) ? 4 : rpw;
  const double reuse = density * kLdsWaves * eff_rpw;
  const long long groups = (long long)ceil_div(p.m, kLdsWaves * eff_rpw) * tiles;
  const double slice_bytes = (double)p.k * kWave * vec * sizeof(T);
  if (groups < 512) return false;
  return reuse >= 12.0 || (slice_bytes > 6.0 * 1024 * 1024 && reuse >= 4.0);
}

// The matrix-core kernels: 16-bit types, n a multiple of 8, 16-byte aligned dense operands,
// k < 65535 for the 8-wave arrangement (packed columns).  Sets kind = 3 (4 waves, 128 x 256
// tiles; param = lanes per row) or 4 (8 waves, 128 x 512 tiles; param = windows per row);
// kind 0 = use a gather kernel.
// nothing about the row kernel's waves per row was asked for
inline bool flags_wpr_free(const Choice& ch) { return !ch.wpr_forced && (ch.variant == 0 || ch.variant == 1); }

struct MfmaChoice {
  int kind = 0, param = 0;
};

template <typename T>
MfmaChoice mfma_variant(const SpmmParams& p, int batch, const Choice& ch) {
  MfmaChoice mc;
  if (sizeof(T) != 2 || (ch.variant != 0 && ch.variant != 3 && ch.variant != 4)) return mc;
  if (!(p.nnz > 0 && p.n % 8 == 0 && aligned(p.dense, 16) && aligned(p.out, 16))) return mc;  // (also when forced)
  const double density = (p.m > 0 && p.k > 0) ? (double)p.nnz / ((double)p.m * p.k) : 0.0;
  const double run = density * kMfmaBKA;  // nonzeros of a row per 128-column chunk
  const bool wide_ok = p.k < 65535;
  const long long tiles_m = ceil_div(p.m, kMfmaBM);
  const long long wgs_wide = tiles_m * ceil_div(p.n, kMfma2BN) * batch;
  const long long wgs_narrow = tiles_m * ceil_div(p.n, kMfmaBN) * batch;
  int kind = ch.variant;
  if (kind == 0) {
    // Measured on MI355X (fp16, m x k = 11008 x 4096, n = 2048): the gather kernels and the
    // matrix-core kernels meet at about 5 % density (0.34 vs 0.32 ms); at 10 % the matrix cores
    // are 1.7x faster, at 50 % (4096 x 4096, n = 8192) 7x; at 2 % the gather kernel is 2x faster.
    // Small outputs (a handful of tiles) leave most CUs idle and stay with the gather kernels.
    // A tile computes all of its 256 / 512 columns: an n that fills less than three quarters of
    // its tiles wastes the difference (n = 64 on 512-column tiles measured 3.5x slower than the
    // gather kernel).
    if (density < 0.05) return mc;
    const double fill_wide = (double)p.n / ((double)ceil_div(p.n, kMfma2BN) * kMfma2BN);
    const double fill_narrow = (double)p.n / ((double)ceil_div(p.n, kMfmaBN) * kMfmaBN);
    if (wide_ok && wgs_wide >= 128 && fill_wide >= 0.75) kind = 4;
    else if (wgs_narrow >= 128 && fill_narrow >= 0.75) kind = 3;
    else return mc;
  }
  if (kind == 4 && !wide_ok) kind = 3;
  mc.kind = kind;
  if (kind == 3) mc.param = ch.lpg ? ch.lpg : (run > 24.0 ? 16 : 8);
  // windows of 16 nonzeros per row: enough for the run of a chunk (2:4 rows have exactly 64 per
  // chunk and need the fifth, or every row-visit would make one exposed pass to find nothing)
  else mc.param = ch.rpw ? ch.rpw : (run > 56.0 ? 5 : run > 20.0 ? 4 : run > 8.0 ? 2 : 1);
  return mc;
}

template <typename T>
bool matrix_core_kernel_applies(const SpmmParams& p, int batch) { return mfma_variant<T>(p, batch, Choice{}).kind != 0; }

// fp32 on the matrix cores: int32 indices, n a multiple of 4, 16-byte aligned dense operands.
// Returns the arrangement code (0 = use a gather kernel).
template <typename T, typename IT>
int mfma_f32_variant(const SpmmParams& p, int batch, const Choice& ch) {
  if (!std::is_same<T, float>::value || !std::is_same<IT, int>::value) return 0;
  if (ch.variant != 0 && ch.variant != 5) return 0;
  if (!(p.nnz > 0 && p.n % 4 == 0 && aligned(p.dense, 16) && aligned(p.out, 16))) return 0;  // (also when forced)
  const double density = (p.m > 0 && p.k > 0) ? (double)p.nnz / ((double)p.m * p.k) : 0.0;
  // 32-row tiles with 128 columns per wave when that still gives most CUs a workgroup; else
  // 16-row tiles (twice the workgroups, twice the reads of the dense operand)
  const long long tiles_m = ceil_div(p.m, 32);
  int arrangement = tiles_m * ceil_div(p.n, 128) * batch >= 200 ? 4 : (p.n <= 64 ? 5 : 6);
  if (ch.nt) arrangement = ch.nt;
  if (ch.variant == 5) return arrangement;
  // MI355X, us, matrix cores / the faster gather kernel, 4096 x 4096:
  //   rows of geometric lengths  n = 128       n = 256       n = 512       n = 1024      n = 2048     of one length  n = 128   n = 256   n = 1024   n = 2048
  //   10 %                       73 / 42       105 / 69      188 / 307     373 / 460     724 / 778                   53 / 33   86 / 60   340 / 227  677 / 415
  //   20 %                       72 / 61       113 / 114     195 / 325     386 / 638     747 / 1225                  52 / 61   86 / 117  340 / 388  677 / 668
  //   25 %                       74 / 77       113 / 140     200 / 341     386 / 768     750 / 1440                  53 / 72   87 / 140  340 / 451  677 / 790
  //   30 %                       75 / 93       112 / 165     201 / 363     388 / 829     753 / 1623                  53 / 87   88 / 171  341 / 518  677 / 921
  //   (11008 x 4096, n = 1024: 10 % 951 / 711, 20 % 991 / 1207, 30 % 1023 / 1750; of one length 931 / 611, 934 / 1016, 933 / 1380)
  // The limit is that of an expansion that took 6 - 20 % longer and tied at 20 %; today's is ahead from there on, and with rows of
  // geometric lengths and 512 columns from 10 %.  What a lower limit costs beside that: explicit zeros, which carry non-finite entries of rows of the dense
  // operand that no nonzero references into the output.  The 16-row arrangements (n = 128 here) stay on request.
  const double fill = (double)p.n / ((double)ceil_div(p.n, 128) * 128);  // share of the computed columns that exist
  if (density >= 0.27 && arrangement == 4 && fill >= 0.75) return arrangement;
  // Beside a kernel that is bound by gathers the tie at 20 % goes to the matrix cores, also with the 16-row tiles of
  // n = 128: alone 124 against 118 us (4096 x 4096 at 20 %, n = 256) and 90 against 84 us (30 %, n = 128), but the
  // neighbour then has the L2 -> CU path to itself (the 15 cells of that sweep on two branches of a graph: 654 -> 600 us).  (The
  // expansion of today: 112 and 74.)
  if (ch.beside_gather && density >= 0.195 && p.n >= 128 && fill >= 0.75) return arrangement;
  return 0;
}

// Windows of 16 nonzeros per row and half chunk of 64 columns for the direct-load matrix-core
// kernel.  One window holds a row's share with a margin of three standard deviations up to 13 %
// density (mean 8.3 of 64), two up to 33 % (mean 21) and exactly at 2:4 sparsity (32 of every 64,
// recognised by nnz being exactly half of m * k); four always do.  A half chunk the windows do not
// hold is multiplied twice, so a wrong guess costs time, not correctness.
inline int mfma3_windows(const SpmmParams& p) {
  const double cells = (double)p.m * p.k;
  const double density = cells > 0 ? (double)p.nnz / cells : 0.0;
  if (density <= 0.13) return 1;
  return (density <= 0.33 || 2.0 * p.nnz == cells) ? 2 : 4;
}

// Dense form of A in the caller's workspace, then the dense GEMM (16-bit types, values shared by the batch).  The GEMM
// wants rows of whole 16-byte chunks: the dense form gets them by zero columns up to a multiple of 8, a dense operand that
// has none (n or its address) is copied into the workspace first.
inline bool dense_path_fits(int elem_size, const SpmmParams& p, bool flagged) {
  return elem_size == 2 && !flagged && p.nnz > 0 && (p.pad || (p.k % 8 == 0 && p.n % 8 == 0 && aligned(p.dense, 16) && aligned(p.out, 16))) && (long long)p.m * round8(p.k) < (1ll << 31) && (long long)round8(p.k) * round8(p.n) < (1ll << 31);
}

inline bool dense_path_pads(const SpmmParams& p) { return p.n % 8 != 0 || !aligned(p.dense, 16); }
inline size_t dense_path_pad_offset(const SpmmParams& p) { return round256((size_t)p.m * round8(p.k) * 2); }
inline size_t dense_path_bytes(const SpmmParams& p, int batch) {
  return dense_path_pads(p) ? dense_path_pad_offset(p) + (size_t)batch * round8(p.k) * round8(p.n) * 2 : (size_t)p.m * round8(p.k) * 2;
}

// Whether the dense-form path is the faster one, from a time model fitted on MI355X (fp16):
//   dense form + GEMM: two launches (8 us), m * k * 2 bytes written at 4 TB/s, the product at
//     1000 TFLOP/s or, when the tiles are few, one round of 128 x 128 tiles per 512 tiles at 0.23 us
//     per K step of 32 (4096^2, n <= 512: 40-45 us whatever the sparsity; 1024^2, n = 2048: 21 us);
//   matrix-core SpMM kernels: 720 dense-equivalent TFLOP/s (2:4 4096^2, n = 8192: 0.40 against 0.27 ms
//     for the dense form; 80 % 11008 x 4096: 0.93 / 0.69; 90 %, n = 2048: 0.27 / 0.23), or with few tiles a
//     workgroup's chain of chunks of 128 columns, per chunk 3.5 us + 7 us * density for 128 x 512 tiles and
//     4.5 + 21 for 128 x 256 tiles by four wavefronts (2:4 4096^2, n = 928: 482 us; 2760 x 2231 at 13 %, n = 1336: 126);
//   gather kernels: nnz * n * 2 bytes through the L2 -> CU path at 26 TB/s (4096^2 at 70 %, n = 256:
//     110 against 58 us; at 90 %, n = 256: 40 against 58; 11008 x 4096 at 95 %, n = 2048: 0.35 / 0.21 ms).
//   a short K makes the GEMM a writer of its output at 3 TB/s (16 x 4096 x 4096, k = 64: 0.18 ms) and the
//     matrix-core SpMM kernels at 1.2 TB/s (8 x 4096 x 4096, k = 128: 0.24 ms), the gather kernels write it at 4 TB/s, the few-columns kernel at 4.5 TB/s plus 10 clocks of a CU's LDS
//     per nonzero and tile (same shape at 93 % sparsity: 0.15 ms; 8 x 4096 x 4096, k = 128 at 50 %: 0.58
//     against 0.17 for the dense form).
// The dense form has to win by 15 % to be taken, by 20 % with a copy of B, 40 % if k is short too (10440 x 664 at 97 %, n = 1422: 47 against 39 us).  `few_columns`: the alternative is the few-columns kernel.
// split_room: the workspace has room for the GEMM to take k in parts where it would (few tiles, long k: the K loop of a
// tile then runs on several CUs; 4096^2 at 70-90 %, n = 128 / 256: 40 / 41 -> 27 / 32 us).
//   Wide rows are gathered in tiles of 512 columns, the last one as slow as the others (3449 x 8696 at 94 %, n = 552: 185
//     against 72 us).
inline double other_families_seconds(const SpmmParams& p, int batch, int matrix_core_kind, bool few_columns) {
  const double cells = (double)p.m * p.k, flops = 2.0 * cells * p.n * batch, density = p.nnz / std::max(cells, 1.0), out_bytes = (double)p.m * p.n * batch * 2;
  double other;
  if (few_columns) {
    other = 8e-6 + out_bytes / 4.5e12 + (double)p.nnz * batch * ceil_div(p.n, 512) * 10.0 / (256 * 2.1e9);
  } else if (matrix_core_kind) {
    const bool wide = matrix_core_kind == 4;
    const double rounds = std::ceil((double)ceil_div(p.m, kMfmaBM) * ceil_div(p.n, wide ? kMfma2BN : kMfmaBN) * batch / (wide ? 256.0 : 512.0));
    const double chain = rounds * (p.k / 128.0) * (wide ? 3.5e-6 + 7e-6 * density : 4.5e-6 + 21e-6 * density);
    other = 8e-6 + std::max({flops / 720e12, chain, out_bytes / 1.2e12});
  } else {
    const double columns = p.n <= 256 ? p.n : ceil_div(p.n, 512) * 512;   // (whole tiles: a last tile of few columns costs like a full one)
    double per_nonzero = columns * 2 / 26e12;
    // Rows of no whole vectors: 16-byte gathers that start at multiples of 2, 4 or 8 bytes.  Us, gathers / dense form: 800 x 9672 at 91 %, n = 859 114 / 50;
    // 1747 x 752 at 81 %, n = 406 13 / 16; 2783 x 3163 at 98 %, n = 1028 30 / 44; few rows of B stay in L1: 2472 x 389 at 84 %, n = 286 11 / 18.
    const int vec = p.n % 4 == 0 ? 4 : p.n % 2 == 0 ? 2 : 1;
    if (p.n % 8 != 0 && p.n >= 256) {
      per_nonzero = columns * 2 / (p.k <= 512 || vec == 4 ? 26e12 : vec == 2 ? 22e12 : 13e12);
    } else if (p.n % 8 != 0) {
      // one nonzero per gather, 90 G of them a second (10680 x 3436 at 89 %, n = 179: 134 / 55), or several (ragged_narrow_waves; 9903 x 2825 at 88 %, n = 79:
      // 94 / 37; 5043 x 4044 at 80 %, n = 26 24 / 38)
      const double mean = (double)p.nnz / std::max(p.m, 1);
      per_nonzero = std::max(ceil_div(p.n, kWave * vec) / 90e9, columns * 2 / 26e12);
      if ((p.n <= 128 || (double)p.m * batch >= 2700) && (vec > 1 || mean <= 1000))
        per_nonzero = std::min(per_nonzero, std::max(1 / (vec > 1 ? 150e9 : 80e9), columns * 2 / ((vec == 4 ? 18e12 : vec == 2 ? 12e12 : 6.5e12) * (p.k <= 512 ? 2 : 1))));
    }
    other = 8e-6 + (double)p.nnz * batch * per_nonzero + out_bytes / 4e12;
  }
  return other;
}
inline bool dense_path_wins(const SpmmParams& p, int batch, int matrix_core_kind, bool few_columns, bool split_room = true) {
  const double cells = (double)p.m * p.k, flops = 2.0 * cells * p.n * batch;
  const double out_bytes = (double)p.m * p.n * batch * 2;
  const double tiles = (double)ceil_div(p.m, 128) * ceil_div(p.n, 128) * batch;
  const int parts = split_room && !p.accumulate ? gemm_auto_split_parts(p.m, p.n, round8(p.k), batch) : 1;
  const double product = std::max({flops / 1000e12, std::ceil(tiles / 512.0) * (p.k / 32.0) * 0.23e-6 / parts, out_bytes / 3e12});
  const double pad = dense_path_pads(p) ? 4e-6 + 4.0 * p.k * p.n * batch / 4e12 : 0.0;
  const double dense_form = 8e-6 + cells * 2 / 4e12 + pad + product;
  return (!dense_path_pads(p) ? 1.15 : p.k < 1024 ? 1.4 : 1.2) * dense_form < other_families_seconds(p, batch, matrix_core_kind, few_columns);
}

// Behind dense form and copy (rounded up to 256 bytes) the workspace may hold what the GEMM wants for splitting K over two
// workgroups per tile (few tiles, long k: gemm_auto_split_bytes); the words it wants zero are zeroed by the kernel
// that writes the dense form.
inline size_t dense_path_split_offset(const SpmmParams& p, int batch) { return round256(dense_path_bytes(p, batch)); }
inline size_t dense_path_split_bytes(const SpmmParams& p, int batch) { return p.accumulate ? 0 : gemm_auto_split_bytes(p.m, p.n, round8(p.k), batch); }

inline bool dense_path_has_split_room(const SpmmParams& p, int batch, const Choice& ch) {
  const size_t split = dense_path_split_bytes(p, batch);
  return split > 0 && ch.ws && aligned(ch.ws, 256) && ch.ws_bytes >= dense_path_split_offset(p, batch) + split;
}

template <typename IT>
int launch_dense_form(int m, int ld, const int* row_offsets, const void* cols, const void* values, void* out, int* zero_words, int n_zero_words,
                      hipStream_t stream) {
  note_kernel("csr_to_dense_kernel<%s>", type_name<IT>());
  launch_csr_to_dense<IT>(m, ld, row_offsets, cols, values, out, zero_words, n_zero_words, stream);
  return check_hip(hipGetLastError(), "spmm dense-form launch");
}

template <typename T, typename IT>
int launch_dense_path(const SpmmParams& p, int batch, const Choice& ch, hipStream_t stream) {
  const int kp = round8(p.k), np = round8(p.n);
  const size_t split = dense_path_split_bytes(p, batch), offset = dense_path_split_offset(p, batch);
  const bool with_split = dense_path_has_split_room(p, batch, ch);
  unsigned char* ws = static_cast<unsigned char*>(ch.ws);
  unsigned char* split_ws = with_split ? ws + offset : nullptr;
  size_t flags_at = 0;
  int flag_words = 0;
  if (with_split) gemm_auto_split_flags(p.m, p.n, kp, batch, &flags_at, &flag_words);
  if (int rc = launch_dense_form<IT>(p.m, kp, p.row_offsets, p.cols, p.values, ws, with_split ? reinterpret_cast<int*>(split_ws + flags_at) : nullptr,
                                     flag_words, stream))
    return rc;
  GemmParams g{p.m, p.n, kp, ws, p.dense, p.out, 0, (long long)p.k * p.n, (long long)p.m * p.n, 0, 0};
  g.row_bias = p.bias;
  g.relu = p.relu;
  g.aux = p.accumulate ? p.out : p.aux;
  g.aux_mode = p.accumulate ? kGemmAdd : p.aux_mode;
  if (p.aux && ch.aux_done) *ch.aux_done = true;
  g.kb = p.k;
  if (dense_path_pads(p)) {
    unsigned char* padded = ws + dense_path_pad_offset(p);
    if (int rc = launch_pad_rows(p.k, p.n, p.dense, kp, np, padded, batch, (long long)p.k * p.n, stream)) return rc;
    g.B = padded;
    g.ldb = np;
    g.kb = kp;
    g.stride_b = (long long)kp * np;
  }
  const int dtype = std::is_same<T, __half>::value ? IEX_F16 : IEX_BF16;
  return gemm_dispatch(dtype, 0, g, batch, stream, split_ws, with_split ? split : 0, with_split);
}

// ---- fp32 by parts: the dense form of A and B as three bf16 planes each, then their product on the bf16 matrix cores (gemm_split_device.cuh) ----
struct SplitPlan {
  int kp, np, group, parts, ld;   // group: batch entries at a time; ld: rows of the parts' sums
  size_t a_at, b_at, sums_at, bytes;
};
// Batch entries' planes at a time, all that they hold together: enough to fill the chip many times over, and a call's memory does not grow with its batch.  (64 of
// 4096 x 4096 at 80 % by 4096 x 4096: 6.5 GB of workspace, 0.6 this way.)
constexpr size_t kSplitGroupBytes = (size_t)512 << 20;
// the workspace: the ranges of the operands' entries, planes of A, planes of B, sums of the parts of K
inline SplitPlan split_plan(const SpmmParams& p, int batch) {
  SplitPlan s;
  s.kp = round32(p.k);
  s.np = round8(p.n);
  s.group = (int)std::min<size_t>(batch, std::max<size_t>(1, kSplitGroupBytes / ((size_t)s.kp * s.np * 6)));
  s.parts = gemm_split_parts(p.m, p.n, s.kp, s.group);
  s.ld = (p.n + 3) & ~3;
  s.a_at = kSplitRanges * 4;
  s.b_at = s.a_at + round256((size_t)p.m * s.kp * 6);
  s.sums_at = s.b_at + round256((size_t)s.group * s.kp * s.np * 6);
  s.bytes = s.sums_at + (s.parts > 1 ? (size_t)s.parts * s.group * p.m * s.ld * 4 : 0);
  return s;
}
// (canonical CSR; an operand's copies in the workspace, which is the caller's to allow; planes within a buffer's 4 GB; a vector of four columns for
// the kernel behind it)
inline bool split_path_fits(const SpmmParams& p) {
  return p.pad && p.nnz > 0 && p.k > 0 && p.n >= 4 && !p.accumulate && !p.per_batch_values && (long long)p.m * round32(p.k) * 6 < (1ll << 32) &&
         (long long)round32(p.k) * round8(p.n) * 6 < (1ll << 32);
}

// Whether that is the faster way, from a time model fitted on MI355X: three launches, the planes' bytes at 4.4 TB/s, the product
// (gemm_split_seconds), the parts' sums at 4 TB/s; the row kernel gathers whole tiles of 256 columns at up to 30 TB/s, the fp32 matrix-core kernel
// multiplies at 92 TFLOP/s.
inline double split_path_seconds(const SpmmParams& p, int batch) {
  const SplitPlan s = split_plan(p, batch);
  const double planes = 3.5e-6 + (6.0 * p.m * s.kp + 10.0 * batch * p.k * p.n) / 4.4e12;
  const double group = gemm_split_seconds(p.m, p.n, s.kp, s.group) + 4e-6 + (s.parts > 1 ? 4.0 * (s.parts + 1) * p.m * p.n * s.group / 4e12 : 0.0);
  return planes + group * batch / s.group + 3.5e-6 * (ceil_div(batch, s.group) - 1);
}
inline bool split_path_wins(const SpmmParams& p, int batch) {
  // Row kernel: whole tiles of 256 columns (narrow ones to the next power of two) at 30 TB/s, 25 where a tile's slice of B outgrows an XCD's L2.
  // Few rows of geometric lengths run at a third of that, which the shape does not tell: the limit is that of even rows.  A last tile of 208 columns or fewer
  // costs less than a whole one (2779 x 1144 at 71 %, n = 153 31 / 37; 5305 x 7241 at 93 %, n = 358 209 / 231).
  // MI355X, us, the kernels before / this way, at either side of the line: 4096 x 4096, even rows, n = 512, 80 % 218 / 112, 90 % 115 / 108, 95 % 62 / 104;
  // n = 256, geometric, 80 % 114 / 80, 90 % 66 / 75; n = 128, 70 % 98 / 70, 80 % 60 / 65; 1656 x 1504, n = 640, 82 % 44 / 42; 2071 x 1694, n = 216,
  // 72 % 36 / 47; 1408 x 10744, n = 513, 92 % 243 / 131; 11008 x 4096 and most of 200 drawn shapes in profiles/spmm_fp32_by_parts.txt.
  int narrow = 32;
  while (narrow < p.n) narrow *= 2;
  const int last = p.n % 256;
  const double columns = p.n <= 128 ? narrow : p.n - last + (last == 0 ? 0 : last <= 208 ? 216 : 256);
  const double gather = 5e-6 + (double)p.nnz * columns * batch * 4 / ((double)p.k * std::min(p.n, 256) > 1.1e6 ? 25e12 : 30e12);
  if (gather < 30e-6) return false;   // (what three launches and a short product take)
  // One tile of 128 columns is what the fp32 matrix-core kernel is good at, and it makes no copies: up to there it keeps the calls that its density rule gives it; from
  // two tiles on they are shorter this way.  Us, that kernel / this way, n = 128 and n = 256: 8000 x 1000 at 60 % 30.8 / 41.8, 59 / 49; 11008 x 4096 at 72 %
  // 171 / 164, 255 / 225; 4096 x 4096 at 72 % (n = 256, its 32-row tiles) 86 / 75, at 30 % 109 / 85; 4096 x 11008 at 72 % 220 / 214.
  if (p.n <= 128 && mfma_f32_variant<float, int>(p, batch, Choice{})) return false;
  return 1.1 * split_path_seconds(p, batch) < gather;
}

// What a call that goes this way wants of workspace; 0: it does not.
inline size_t split_path_bytes(const SpmmParams& p, int batch, bool forced) {
  if (!split_path_fits(p) || (!forced && !split_path_wins(p, batch))) return 0;
  const size_t bytes = split_plan(p, batch).bytes;
  return bytes <= kSplitWorkspaceMost ? bytes : 0;
}

// Behind the product: adds the parts of K up (bias, ReLU), or where an operand holds an infinity or a NaN, which a product of parts (and of the
// dense form's zeros) spreads, or entries outside the range in which parts hold all 24 bits, computes it as the row kernel does, in as many workgroups as the
// chip holds: results there are the row kernel's.  Rows of up to kFewNonzeros are a chain of multiply-adds: three of nine products of parts are left out, which the roundings of
// a longer chain outweigh (2-norm against 64 bits, nonzeros far apart, by parts / by the row kernel: one 2.59e-8 / 2.53e-8, two 3.6e-8 / 3.1e-8, four 4.5e-8 / 4.0e-8, seven
// 5.1e-8 / 5.1e-8, eight 5.3e-8 / 5.4e-8, 32 6.2e-8 / 6.7e-8).  16 x 2048 rows, n = 512, half of them of seven nonzeros: 197 -> 219 us.
// With K in one part it ends at once else (2 us).  Us a call, 4096 x 4096 at 80 %, n = 256 / at 90 %, n = 1024: row
// kernel 122 / 238, by parts 77 / 178, one infinity 159 / 394 (with the product computed all the same, and this kernel in 256 workgroups where K is in one part, 204 / 556).
constexpr int kFinishBlocks = 1024, kFewNonzeros = 7;
__global__ __launch_bounds__(256) void spmm_split_finish_kernel(SpmmParams p, const unsigned* ranges, const float* sums, int parts, int ld, int tiles, int batch) {
  __shared__ float red[spmm_lds_floats<4, 4, 1>()];
  if (ranges[kSplitVerdict] == 0) {
    const long long total = (long long)p.m * tiles * batch;
    for (long long i = blockIdx.x; i < total; i += gridDim.x) {
      const int row = (int)(i % p.m), rest = (int)(i / p.m);
      spmm_block<float, int, 4, kWave, 4, kSpmmUnroll, 1, true>(p, row, rest % tiles, rest / tiles, red);
      __syncthreads();
    }
  } else {
    typedef float four __attribute__((ext_vector_type(4)));
    typedef four any4 __attribute__((aligned(4)));
    const int chunks = ld / 4;
    const size_t rows = (size_t)p.m * batch, part = rows * ld;
    const int* cols = static_cast<const int*>(p.cols);
    auto finish = [&](size_t zr, int row, int c, four x) {
      if (p.bias) x += p.bias[row];
      if (p.relu) {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = fmaxf(x[e], 0.f);
      }
      float* out = static_cast<float*>(p.out) + zr * p.n + c;
      if (c + 4 <= p.n) {
        *reinterpret_cast<any4*>(out) = x;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (c + e < p.n) out[e] = x[e];
      }
    };
    // (a short row: n >= 4, so the last chunk is read a few columns early)
    auto chain = [&](size_t zr, int start, int end, int c) {
      const int at = min(c, p.n - 4), shift = c - at;
      const float* dense = static_cast<const float*>(p.dense) + (zr / p.m) * p.k * p.n + at;
      four x = {0.f, 0.f, 0.f, 0.f};
      for (int j0 = start; j0 < end; j0 += 4) {   // (four gathers in flight; past the end the last one's row, which is not added)
        four b[4];
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int j = min(j0 + u, end - 1);
          b[u] = *reinterpret_cast<const any4*>(dense + (size_t)cols[j] * p.n);
          v[u] = static_cast<const float*>(p.values)[j];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
#pragma unroll
          for (int e = 0; e < 4; ++e) x[e] = j0 + u < end ? fmaf(v[u], b[u][e], x[e]) : x[e];
        }
      }
      const four y = x;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = shift == 0 ? y[e] : shift == 1 ? y[min(e + 1, 3)] : shift == 2 ? y[min(e + 2, 3)] : y[3];
      return x;
    };
    auto few = [](int start, int end) { return start < end && end - start <= kFewNonzeros; };
    if (parts > 1) {
      for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < rows * chunks; i += (size_t)gridDim.x * 256) {
        const size_t zr = i / chunks;
        const int c = (int)(i - zr * chunks) * 4, row = (int)(zr % p.m), start = p.row_offsets[row], end = p.row_offsets[row + 1];
        const float* from = sums + zr * ld + c;
        four x = *reinterpret_cast<const four*>(from);
        for (int s = 1; s < parts; ++s) x += *reinterpret_cast<const four*>(from + s * part);
        if (few(start, end)) x = chain(zr, start, end, c);
        finish(zr, row, c, x);
      }
    } else {   // (the product has written all rows; short ones once more.  A wavefront looks at rows far apart, 64 at a time: short ones may stand side by side)
      const size_t waves = (size_t)gridDim.x * 4;
      for (size_t first = (size_t)blockIdx.x * 4 + uniform(threadIdx.x >> 6); first < rows; first += waves * kWave) {
        const size_t mine = first + lane_id() * waves;
        const int row = (int)(min(mine, rows - 1) % p.m), start = p.row_offsets[row], end = p.row_offsets[row + 1];
        for (unsigned long long them = __ballot(mine < rows && few(start, end)); them; them &= them - 1) {
          const int src = __ffsll(them) - 1, r = bcast_i(row, src), from = bcast_i(start, src), to = bcast_i(end, src);
          const size_t zr = first + src * waves;
          for (int c = lane_id() * 4; c < p.n; c += kWave * 4) finish(zr, r, c, chain(zr, from, to, c));
        }
      }
    }
  }
}

inline int launch_split_path(const SpmmParams& whole, int batch, void* workspace, hipStream_t stream) {
  const SplitPlan s = split_plan(whole, batch);
  unsigned char* ws = static_cast<unsigned char*>(workspace);
  unsigned* ranges = reinterpret_cast<unsigned*>(ws);
  float* sums = reinterpret_cast<float*>(ws + s.sums_at);
  const long long plane_a = (long long)whole.m * s.kp, plane_b = (long long)s.kp * s.np;
  const SplitSparse a{whole.m, s.kp, whole.row_offsets, static_cast<const int*>(whole.cols), static_cast<const float*>(whole.values), plane_a, ws + s.a_at};
  for (int first = 0; first < batch; first += s.group) {   // (A's planes stay; the other room is each group's in turn)
    const int entries = std::min(s.group, batch - first);
    SpmmParams p = whole;
    p.dense = static_cast<const float*>(whole.dense) + (size_t)first * p.k * p.n;
    p.out = static_cast<float*>(whole.out) + (size_t)first * p.m * p.n;
    const SplitDense b{entries, p.k, p.n, static_cast<const float*>(p.dense), s.kp, s.np, s.np, 3 * plane_b, plane_b, ws + s.b_at};
    if (int rc = first == 0 ? launch_split_operands(a, b, ranges, stream) : launch_split_operand(b, ranges, stream)) return rc;
    SplitParams g{};
    g.M = p.m, g.N = p.n, g.K = s.kp;
    g.A = ws + s.a_at, g.B = ws + s.b_at;
    g.lda = s.kp, g.ldb = s.np;
    g.plane_a = (unsigned)(plane_a * 2), g.plane_b = (unsigned)(plane_b * 2);
    g.stride_b = 3 * plane_b;
    g.parts = s.parts;
    if (s.parts > 1) {
      g.C = sums, g.ldc = s.ld, g.stride_c = (long long)p.m * s.ld, g.stride_part = g.stride_c * entries;
    } else {
      g.C = static_cast<float*>(p.out), g.ldc = p.n, g.stride_c = (long long)p.m * p.n;
      g.row_bias = p.bias, g.relu = p.relu;
    }
    g.ranges = ranges, g.slots_a = split_sparse_blocks(a), g.slots_b = split_dense_blocks(b), g.finite = 1;
    if (int rc = gemm_split(g, false, entries, stream)) return rc;
    note_kernel("spmm_split_finish_kernel");
    const int tiles = ceil_div(p.n, kWave * 4);
    hipLaunchKernelGGL(spmm_split_finish_kernel, dim3((unsigned)std::min<long long>(kFinishBlocks, (long long)p.m * tiles * entries)), dim3(256), 0, stream, p, ranges, sums,
                       s.parts, s.ld, tiles, entries);
    if (int rc = check_hip(hipGetLastError(), "spmm (fp32 by parts) launch")) return rc;
  }
  return 0;
}

template <typename T, typename IT>
int launch_typed(const SpmmParams& p, int batch, const Choice& given, hipStream_t stream) {
  constexpr int kMax = 16 / (int)sizeof(T);
  Choice ch = given;
  // Columns in any order: the few-columns kernel where it applies (it takes nonzeros as they come), else the row kernel.
  if (ch.any_order && ch.variant == 0) {
    if (smallk_wanted<T>(p, batch)) return launch_smallk<T, IT>(p, batch, stream);
    ch.variant = 1;
  }
  // A with few columns and rows that gather, wide output: the tile of the dense operand in LDS, rows
  // streamed (spmm_smallk_device.cuh; smallk_wanted has the measurements).  16-bit products that are
  // dense enough go to the dense-form path first (time model above).
  if (ch.variant == 0 && smallk_wanted<T>(p, batch)) {
    if constexpr (sizeof(T) == 2) {
      const bool room = ch.ws && aligned(ch.ws, 16) && ch.ws_bytes >= dense_path_bytes(p, batch);
      if (room && dense_path_fits(2, p, p.per_batch_values) && dense_path_wins(p, batch, 0, true, dense_path_has_split_room(p, batch, ch)))
        return launch_dense_path<T, IT>(p, batch, ch, stream);
    }
    return launch_smallk<T, IT>(p, batch, stream);
  }
  if constexpr (std::is_same<T, float>::value && std::is_same<IT, int>::value) {
    if ((ch.variant == 12 || (ch.variant == 0 && !ch.beside_gather)) && ch.ws && aligned(ch.ws, 256)) {
      const size_t need = split_path_bytes(p, batch, ch.variant == 12);
      if (need && ch.ws_bytes >= need) return launch_split_path(p, batch, ch.ws, stream);
    }
    if (const int arr = mfma_f32_variant<T, IT>(p, batch, ch)) {
      const bool split = ch.lpg != 8;   // (lanes-per-group code 8 = no role split, for tuning)
      // (a row's windows are the kernel's own affair; numbers that it never had are refused)
      IEX_REQUIRE(split || ch.rpw == 0 || ch.rpw == 2 || ch.rpw == 4 || ch.rpw == 8, IEX_ERR_BAD_ARGUMENT, "spmm: windows of the fp32 matrix-core variant must be 2, 4 or 8 (got %d)", ch.rpw);
      return launch_mfma_f32(p, batch, arr, split, stream);
    }
  }
  if (ch.variant == 6 && sizeof(T) == 2 && p.nnz > 0 && p.n % 8 == 0 && aligned(p.dense, 16) && aligned(p.out, 16))
    return launch_mfma3<T, IT>(p, batch, ch.rpw ? ch.rpw : mfma3_windows(p), stream);
  const MfmaChoice mc = mfma_variant<T>(p, batch, ch);
  if constexpr (sizeof(T) == 2) {
    const bool fits = dense_path_fits(2, p, p.per_batch_values);
    const bool room = ch.ws && aligned(ch.ws, 16) && ch.ws_bytes >= dense_path_bytes(p, batch);
    if (ch.variant == 7) {
      IEX_REQUIRE(fits, IEX_ERR_UNSUPPORTED, "spmm: the dense-form path needs 16-bit values shared by the batch and, without IEX_SPMM_PAD_OPERANDS, k and n multiples of 8 and 16-byte aligned operands");
      IEX_REQUIRE(room, IEX_ERR_BAD_ARGUMENT, "spmm: the dense-form path needs a 16-byte aligned workspace of %zu bytes (iex_spmm_ws)", dense_path_bytes(p, batch));
      return launch_dense_path<T, IT>(p, batch, ch, stream);
    }
    if (ch.variant == 0 && fits && room && dense_path_wins(p, batch, mc.kind, false, dense_path_has_split_room(p, batch, ch))) return launch_dense_path<T, IT>(p, batch, ch, stream);
  }
  // Where the 8-wave kernel would run: the direct-load kernel wins on 2:4 weights (4096 x 4096,
  // n = 8192: 0.37 against 0.40-0.46 ms with five windows), ties at 80 % sparsity (11008 x 4096:
  // 0.94 against 0.93; 4096 x 11008: 0.82 both) and loses at 90 % (n = 2048: 0.29 against 0.26);
  // with four windows (denser than 33 %, not 2:4) it spills registers.
  if (mc.kind == 4 && ch.variant == 0 && 2.0 * p.nnz == (double)p.m * p.k) return launch_mfma3<T, IT>(p, batch, 2, stream);
  if (mc.kind == 4) return launch_mfma2<T, IT>(p, batch, mc.param, stream);
  if (mc.kind == 3) return launch_mfma<T, IT>(p, batch, mc.param, stream);
  if (ch.variant == 8) {
    IEX_REQUIRE(smallk_fits<T>(p), IEX_ERR_UNSUPPORTED, "spmm: the few-columns kernel needs k <= %d and an output at least %d columns wide", kSmallKMax, sizeof(T) == 2 ? kWave : kWave * kMax);
    return launch_smallk<T, IT>(p, batch, stream);
  }
  int lvec = 0, rpw = 0;
  if (ch.variant != 11 && lds_variant<T>(p, batch, ch, lvec, rpw)) {
    if (lvec == kMax) return launch_lds_rpw<T, IT, kMax>(p, batch, rpw, stream);
    return launch_lds_rpw<T, IT, kMax / 2>(p, batch, rpw, stream);
  }
  int wpr = ch.wpr;
  bool by_length = true;   // (the rule for few chunks below)
  SpmmShape sh = spmm_pick_shape<T>(p.n, p.dense, p.out);
  if (ch.lpg && sh.vec == kMax && ch.lpg <= sh.lpg) sh.lpg = ch.lpg;  // narrower tiles on request
  // The caller knows the pattern's row lengths: wavefronts per row by the row's own length instead of one number for
  // the whole matrix.  Measured on MI355X (fp32, 4096 x 4096, geometric row lengths, us, four waves for every row /
  // this kernel at its best chunks-per-wave): 98 % sparse n = 64 9.0 / 7.6, n = 128 12.5 / 11.2, n = 256 17.2 / 20.0;
  // 95 % 12.7 / 13.9, 19.7 / 22.3, 36.9 / 39.2; 90 % 19.1 / 22.0, 36.7 / 38.6, 69.4 / 67.0; 80 % 33 / 42, 59 / 73,
  // 119 / 122.  The row kernel is bound by the gathers' way from L2 into the CUs (20-26 TB/s on every n = 256
  // cell), not by its longest rows: four waves on every row keep more gathers in flight than a schedule that gives short
  // rows one wave, and that wins wherever the chip is full.  So this kernel is taken where it is not: fewer chunks
  // of 64 nonzeros than the chip holds wavefronts, and narrow tiles (several nonzeros per gather instruction).
  const bool ragged = p.n % kMax != 0 && p.n >= kWave * kMax / 2 && ch.lpg == 0;
  if (ch.variant == 11) IEX_REQUIRE(ch.hist && (sh.vec == kMax || (ragged && ch.wpr_forced && wpr == 4)), IEX_ERR_BAD_ARGUMENT, "spmm: the rows-by-length kernel needs the row-length histogram (iex_spmm_sched) and full 128-bit vectors");
  const double chunk_count = (double)p.nnz / kWave * ceil_div(p.n, sh.lpg * sh.vec) * batch;
  if (ch.hist && ch.nt <= 1 && (sh.vec == kMax || ragged) && ((ch.variant == 11 && ch.wpr_forced && wpr == 4) || (ch.variant != 11 && flags_wpr_free(ch)))) {
    const int way = ch.variant == 11 ? (ch.rpw ? ch.rpw - 1 : 0) : rows_by_histogram(p, batch, ch.hist, sizeof(T), sh.lpg, wpr);
    if (way >= 0) return launch_long_rows<T, IT>(p, batch, sh.lpg, ragged, ch.hist, way, stream);
    if (way == kRowsSixteenWaves && !ragged) return launch_rows<T, IT>(p, batch, kWave, ch.hist, 1, stream);
    wpr = way == kRowsOneWave ? 1 : wpr;
    by_length = way == kRowsAsBefore;
  }
  if (by_length && ch.hist && sh.vec == kMax && ch.nt <= 1 &&
      (ch.variant == 11 || (flags_wpr_free(ch) && ch.hist[0] > 0 && wpr != 1 && sh.lpg <= 32 && chunk_count <= 8192.0)))
    return launch_rows<T, IT>(p, batch, sh.lpg, ch.hist, ch.variant == 11 ? ch.rpw : 0, stream);
  // Two tiles per wave double the slice of the dense operand that the waves of an XCD share in
  // its L2 and measured slower (2x at k = 4096, n = 8192): only on request.
  const int nt = ch.nt ? ch.nt : 1;
  if (sh.vec == kMax) {
    switch (sh.lpg) {
      case 8: return launch_wpr<T, IT, kMax, 8>(p, batch, wpr, nt, stream);
      case 16: return launch_wpr<T, IT, kMax, 16>(p, batch, wpr, nt, stream);
      case 32: return launch_wpr<T, IT, kMax, 32>(p, batch, wpr, nt, stream);
      default: return launch_wpr<T, IT, kMax, 64>(p, batch, wpr, nt, stream);
    }
  }
  // Rows whose length is not a multiple of the 128-bit vector (n = 785, 197 of the ViT shapes), at least
  // half a tile wide: 128-bit accesses at element alignment instead of narrower vectors.  Measured on
  // the reference's ViT sweep shapes (fp32, batch 384, 97 % sparse): 785 x 785 outputs 865 -> 516 us,
  // 197 x 197 outputs 64 -> 33 us.
  if (ragged) return launch_ragged<T, IT, kMax>(p, batch, wpr, stream);
  // ... and narrower ones, several nonzeros per gather
  if (p.n >= kMax && p.n < kWave * kMax / 2 && ch.lpg == 0 && nt == 1 && !ch.wpr_forced) {
    if (const int waves = ragged_narrow_waves(p, batch, ch.hist, sizeof(T)))
      return launch_spmm_ragged(std::is_same<T, float>::value ? IEX_F32 : std::is_same<T, __half>::value ? IEX_F16 : IEX_BF16, sizeof(IT) == 2 ? IEX_I16 : IEX_I32, p, batch, waves, stream);
  }
  if constexpr (kMax == 8) {
    if (sh.vec == 4) return launch_wpr<T, IT, 4, 64>(p, batch, wpr, nt, stream);
  }
  if (sh.vec == 2) return launch_wpr<T, IT, 2, 64>(p, batch, wpr, nt, stream);
  return launch_wpr<T, IT, 1, 64>(p, batch, wpr, nt, stream);
}

}  // namespace

// The estimate of the time model above for a 16-bit product by a family that reads the CSR arrays (no dense form).
double spmm_seconds(int m, int k, int n, int nonzeros) {
  void* const some_aligned = reinterpret_cast<void*>(size_t(256));
  SpmmParams p{m, k, n, nonzeros, nullptr, nullptr, nullptr, nullptr, some_aligned, nullptr, some_aligned, 0, 0, 0};
  const bool few = smallk_wanted<__half>(p, 1);
  return other_families_seconds(p, 1, few ? 0 : mfma_variant<__half>(p, 1, Choice{}).kind, few);
}

// For the fused launcher: the number of register windows if the dispatcher would run this
// fp16 SpMM (one batch entry, nothing forced) on the 8-wave matrix-core kernel, else 0.
int spmm_matrix_core_windows(const SpmmParams& p) {
  const MfmaChoice mc = mfma_variant<__half>(p, 1, Choice{});
  return mc.kind == 4 ? mc.param : 0;
}

int spmm_dispatch(int dtype, int itype, int flags, int m, int k, int n, int nonzeros,
                  const int* row_indices, const void* values, const int* row_offsets,
                  const void* column_indices, const void* dense, const float* bias, void* out,
                  void* stream, int batch, void* workspace, size_t workspace_bytes, const int* row_histogram = nullptr,
                  const void* aux = nullptr, int aux_mode = 0, bool* aux_done = nullptr) {
  IEX_REQUIRE(m >= 0 && k >= 0 && n >= 0 && nonzeros >= 0 && batch >= 0, IEX_ERR_BAD_ARGUMENT,
              "spmm: negative dimension (m=%d k=%d n=%d nnz=%d batch=%d)", m, k, n, nonzeros, batch);
  trail_reset();
  if (m == 0 || n == 0 || batch == 0) return 0;  // empty output: nothing to launch
  IEX_REQUIRE(row_indices && row_offsets && dense && out, IEX_ERR_BAD_ARGUMENT,
              "spmm: null pointer argument");
  IEX_REQUIRE(nonzeros == 0 || (values && column_indices), IEX_ERR_BAD_ARGUMENT,
              "spmm: null values / column_indices with nnz=%d", nonzeros);
  IEX_REQUIRE(batch <= 65535, IEX_ERR_TOO_LARGE, "spmm: batch %d exceeds 65535", batch);
  IEX_REQUIRE((long long)k * n < (1ll << 31) && (long long)m * n < (1ll << 31), IEX_ERR_TOO_LARGE,
              "spmm: a dense operand exceeds 2^31 elements per batch entry");
  IEX_REQUIRE(itype == IEX_I32 || (itype == IEX_I16 && k <= 32768), IEX_ERR_BAD_ARGUMENT,
              "spmm: int16 column indices need k <= 32768 (k=%d)", k);
  Choice ch;
  ch.wpr = (flags >> 8) & 0xff;
  ch.wpr_forced = ch.wpr != 0;
  if (ch.wpr == 0) ch.wpr = spmm_pick_wpr(m, nonzeros, dtype == IEX_F32 ? 4 : 2, n, batch);
  ch.hist = row_histogram;
  ch.variant = (flags >> 16) & 0xf;
  ch.rpw = (flags >> 20) & 0xf;
  ch.nt = (flags >> 24) & 0xf;
  ch.lpg = ((flags >> 28) & 0x7) ? (4 << ((flags >> 28) & 0x7)) : 0;
  ch.ws = workspace;
  ch.ws_bytes = workspace ? workspace_bytes : 0;
  ch.any_order = (flags & IEX_SPMM_ANY_COLUMN_ORDER) != 0;
  ch.beside_gather = (flags & IEX_SPMM_BESIDE_GATHER_KERNEL) != 0 && !ch.any_order;
  SpmmParams p{m, k, n, nonzeros, row_indices, values, row_offsets, column_indices, dense, bias, out,
               (flags & IEX_SPMM_PER_BATCH_VALUES) != 0, (flags & IEX_SPMM_ACCUMULATE) != 0,
               (flags & IEX_SPMM_RELU) != 0};
  p.pad = (flags & IEX_SPMM_PAD_OPERANDS) != 0;
  p.aux = aux;
  p.aux_mode = aux_mode;
  ch.aux_done = aux_done;
  // beyond the 256 MB last-level cache an output can only stream; the hint is worth 15-25 % of the write rate
  p.stream_out = (double)m * n * batch * (dtype == IEX_F32 ? 4 : 2) >= 128e6;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (ch.variant == 10 && nonzeros < 8) {   // (its loads of eight values at a time need eight to exist: the row kernel instead)
    ch.variant = 1;
    ch.wpr = spmm_pick_wpr(m, nonzeros, dtype == IEX_F32 ? 4 : 2, n, batch);   // (bits 8..15 meant the dense-block threshold)
    ch.wpr_forced = false;
  }
  const int blocks_ready = ((flags & IEX_SPMM_TABLES_READY) ? 1 : 0) | ((flags & IEX_SPMM_LISTS_READY) ? 2 : 0);
  if (ch.variant == 0 && !ch.any_order && ch.ws && aligned(ch.ws, 16) && spmm_blocks_fits(dtype, itype, p) && spmm_blocks_wins(p, batch) &&
      ch.ws_bytes >= spmm_blocks_bytes(p))
    return launch_spmm_blocks(dtype, p, batch, ch.ws, 0, blocks_ready, s);
  if (ch.variant == 10) {
    IEX_REQUIRE(spmm_blocks_fits(dtype, itype, p), IEX_ERR_UNSUPPORTED,
                "spmm: the dense-blocks kernel needs fp16 / bf16, int32 indices, n a multiple of 64 up to 1024, plain store without bias or ReLU, k <= 65536 and 16-byte aligned dense operands");
    IEX_REQUIRE(ch.ws && aligned(ch.ws, 16) && ch.ws_bytes >= spmm_blocks_bytes(p), IEX_ERR_BAD_ARGUMENT,
                "spmm: the dense-blocks kernel needs a 16-byte aligned workspace of %zu bytes (iex_spmm_ws)", spmm_blocks_bytes(p));
    return launch_spmm_blocks(dtype, p, batch, ch.ws, (flags >> 8) & 0xff, blocks_ready, s);
  }
  if (dtype == IEX_F32 && itype == IEX_I32) return launch_typed<float, int>(p, batch, ch, s);
  if (dtype == IEX_F16 && itype == IEX_I32) return launch_typed<__half, int>(p, batch, ch, s);
  if (dtype == IEX_F16 && itype == IEX_I16) return launch_typed<__half, short>(p, batch, ch, s);
  if (dtype == IEX_BF16 && itype == IEX_I32) return launch_typed<__hip_bfloat16, int>(p, batch, ch, s);
  return fail(IEX_ERR_UNSUPPORTED, "spmm: no kernel for dtype=%d itype=%d", dtype, itype);
}

// Bytes of workspace with which iex_spmm_ws would take the dense-form path for this call (0: it
// would not, whatever the workspace).  Pointers are taken to be 16-byte aligned.
// kind: which family the workspace would serve (0 = none, 7 = dense form, 9 = partial sums of the k split, 10 = the
// tables and lists of the dense-blocks kernel, 12 = the planes and sums of the fp32 product by parts).
static size_t workspace_plan(int dtype, int itype, int flags, int m, int k, int n, int nonzeros, int batch, int* kind) {
  *kind = 0;
  if (m <= 0 || k <= 0 || n <= 0 || nonzeros <= 0 || batch <= 0) return 0;
  const int variant = (flags >> 16) & 0xf;
  if (variant == 0 && (flags & IEX_SPMM_ANY_COLUMN_ORDER)) return 0;   // families 1 and 8 use no workspace
  void* const some_aligned = reinterpret_cast<void*>(size_t(256));
  if (dtype == IEX_F32 && itype == IEX_I32 && (variant == 0 || variant == 12)) {
    const SpmmParams p{m, k, n, nonzeros, nullptr, nullptr, nullptr, nullptr, some_aligned, nullptr, some_aligned,
                       (flags & IEX_SPMM_PER_BATCH_VALUES) != 0, (flags & IEX_SPMM_ACCUMULATE) != 0, (flags & IEX_SPMM_RELU) != 0, (flags & IEX_SPMM_PAD_OPERANDS) != 0};
    const size_t bytes = variant == 0 && (flags & IEX_SPMM_BESIDE_GATHER_KERNEL) ? 0 : split_path_bytes(p, batch, variant == 12);
    if (bytes) *kind = 12;
    return bytes;
  }
  if (!(dtype == IEX_F16 || dtype == IEX_BF16) || !(itype == IEX_I32 || itype == IEX_I16)) return 0;
  if (variant != 0 && variant != 7 && variant != 10) return 0;
  SpmmParams p{m, k, n, nonzeros, nullptr, nullptr, nullptr, nullptr, some_aligned, nullptr, some_aligned,
               (flags & IEX_SPMM_PER_BATCH_VALUES) != 0, (flags & IEX_SPMM_ACCUMULATE) != 0, (flags & IEX_SPMM_RELU) != 0};
  p.pad = (flags & IEX_SPMM_PAD_OPERANDS) != 0;
  if (variant != 7 && nonzeros >= 8 && spmm_blocks_fits(dtype, itype, p) && (variant == 10 || spmm_blocks_wins(p, batch))) {
    *kind = 10;
    return spmm_blocks_bytes(p);
  }
  if (variant == 10) return 0;
  if (!dense_path_fits(2, p, (flags & IEX_SPMM_PER_BATCH_VALUES) != 0)) return 0;
  if (variant == 0) {
    Choice ch;
    ch.rpw = (flags >> 20) & 0xf;
    ch.lpg = ((flags >> 28) & 0x7) ? (4 << ((flags >> 28) & 0x7)) : 0;
    const bool few = smallk_wanted<__half>(p, batch);
    if (!dense_path_wins(p, batch, few ? 0 : mfma_variant<__half>(p, batch, ch).kind, few)) return 0;
  }
  *kind = 7;
  const size_t split = dense_path_split_bytes(p, batch);
  return split ? dense_path_split_offset(p, batch) + split : dense_path_bytes(p, batch);
}

size_t spmm_workspace_bytes(int dtype, int itype, int flags, int m, int k, int n, int nonzeros, int batch) {
  int kind;
  return workspace_plan(dtype, itype, flags, m, k, n, nonzeros, batch, &kind);
}

int spmm_workspace_kind(int dtype, int itype, int flags, int m, int k, int n, int nonzeros, int batch) {
  int kind;
  workspace_plan(dtype, itype, flags, m, k, n, nonzeros, batch, &kind);
  return kind;
}

// ---- A^T * G (the gradient of a sparse layer's input) from the CSR form of A, where the dense-form path would run it:
// the dense form of A is its transpose's, read as a (K,M) operand, so neither the values nor the pattern of the
// transposed matrix are needed.  ws = dense form (m x round8(k)), copy of G where its rows are no whole chunks, GEMM's room.
struct TransposedPlan {
  bool wanted;
  bool pads;
  size_t pad_at, split_at, split_bytes, bytes;
};
static TransposedPlan transposed_plan(int dtype, int m, int k, int n, int nonzeros, const void* dense) {
  TransposedPlan t{};
  if (!(dtype == IEX_F16 || dtype == IEX_BF16) || m <= 0 || k <= 0 || n <= 0 || nonzeros <= 0) return t;
  void* const some_aligned = reinterpret_cast<void*>(size_t(256));
  SpmmParams p{k, m, n, nonzeros, nullptr, nullptr, nullptr, nullptr, dense, nullptr, some_aligned, 0, 0, 0};   // (the product as the SpMM it replaces)
  p.pad = 1;
  if (!dense_path_fits(2, p, false) || (long long)m * round8(k) >= (1ll << 31) || (long long)m * round8(n) >= (1ll << 31)) return t;
  const bool few = smallk_wanted<__half>(p, 1);
  t.wanted = dense_path_wins(p, 1, few ? 0 : mfma_variant<__half>(p, 1, Choice{}).kind, few);
  t.pads = dense_path_pads(p);
  t.pad_at = round256((size_t)m * round8(k) * 2);
  t.split_at = t.pads ? round256(t.pad_at + (size_t)m * round8(n) * 2) : t.pad_at;
  t.split_bytes = gemm_auto_split_bytes(k, n, m, 1);
  t.bytes = t.split_at + t.split_bytes;
  return t;
}

size_t spmm_transposed_workspace_bytes(int dtype, int m, int k, int n, int nonzeros) {
  const TransposedPlan t = transposed_plan(dtype, m, k, n, nonzeros, reinterpret_cast<void*>(size_t(256)));
  return t.wanted ? t.bytes : 0;
}

int spmm_transposed(int dtype, int itype, int m, int k, int n, int nonzeros, const void* values, const int* row_offsets, const void* cols, const void* dense,
                    void* out, hipStream_t stream, void* workspace, size_t workspace_bytes) {
  trail_reset();
  const TransposedPlan t = transposed_plan(dtype, m, k, n, nonzeros, dense);
  IEX_REQUIRE(t.bytes > 0, IEX_ERR_UNSUPPORTED, "spmm (transposed): needs fp16 / bf16 operands, at least one nonzero and fewer than 2^31 elements");
  IEX_REQUIRE(itype == IEX_I32 || itype == IEX_I16, IEX_ERR_UNSUPPORTED, "spmm (transposed): column indices must be int32 or int16");
  IEX_REQUIRE(values && row_offsets && cols && dense && out, IEX_ERR_BAD_ARGUMENT, "spmm (transposed): null pointer argument");
  IEX_REQUIRE(workspace && aligned(workspace, 256) && workspace_bytes >= t.bytes, IEX_ERR_BAD_ARGUMENT,
              "spmm (transposed): needs a 256-byte aligned workspace of %zu bytes", t.bytes);
  unsigned char* ws = static_cast<unsigned char*>(workspace);
  size_t flags_at = 0;
  int flag_words = 0;
  if (t.split_bytes) gemm_auto_split_flags(k, n, m, 1, &flags_at, &flag_words);
  int* flags = t.split_bytes ? reinterpret_cast<int*>(ws + t.split_at + flags_at) : nullptr;
  if (int rc = itype == IEX_I16 ? launch_dense_form<short>(m, round8(k), row_offsets, cols, values, ws, flags, flag_words, stream)
                                : launch_dense_form<int>(m, round8(k), row_offsets, cols, values, ws, flags, flag_words, stream))
    return rc;
  GemmParams g{k, n, m, ws, dense, out, 0, 0, 0, 0, 0};
  g.lda = round8(k);
  if (t.pads) {
    if (int rc = launch_pad_rows(m, n, dense, m, round8(n), ws + t.pad_at, 1, 0, stream)) return rc;
    g.B = ws + t.pad_at;
    g.ldb = round8(n);
  }
  return gemm_dispatch(dtype, 2, g, 1, stream, t.split_bytes ? ws + t.split_at : nullptr, t.split_bytes, t.split_bytes > 0);
}

// ---- the library's own scratch memory, for callers that cannot allocate ---------------------------------
// One array per GPU, placed when the code object is loaded on it and held until the process ends.  In host
// code the array's name is only a handle for hipGetSymbolAddress: every use of the memory below goes through
// the per-device pointer that call returned.
constexpr size_t kStaticScratchBytes = IEX_SPMM_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex scratch_mutex;
void* scratch_ptr[kMaxDevices] = {};   // per device: each GPU holds its own copy of the array at its own address

// The calling thread's current device's copy of `scratch` (looked up once per device, with that device current).
int static_scratch(void** ptr) {
  int device = -1;
  if (int rc = check_hip(hipGetDevice(&device), "hipGetDevice")) return rc;
  IEX_REQUIRE(device >= 0 && device < kMaxDevices, IEX_ERR_UNSUPPORTED, "spmm: device ordinal %d beyond %d", device, kMaxDevices - 1);
  std::lock_guard<std::mutex> lock(scratch_mutex);
  if (!scratch_ptr[device]) {
    void* p = nullptr;
    if (int rc = check_hip(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)")) return rc;
    IEX_REQUIRE(p != nullptr && aligned(p, 256), IEX_ERR_STATE, "spmm: the library's scratch array has no usable device address");
    scratch_ptr[device] = p;
  }
  *ptr = scratch_ptr[device];
  return 0;
}
}  // namespace

}  // namespace iex

extern "C" {

int iex_spmm_static(int dtype, int itype, int flags, int m, int k, int n, int nonzeros,
                    const int* row_indices, const void* values, const int* row_offsets,
                    const void* column_indices, const void* dense, const float* bias, void* out,
                    void* stream, int batch) {
  using namespace iex;
  // every call shares the array with whatever ran before it: nothing in it counts as "still there"
  flags &= ~(IEX_SPMM_TABLES_READY | IEX_SPMM_LISTS_READY);
  const size_t need = spmm_workspace_bytes(dtype, itype, flags, m, k, n, nonzeros, batch);
  // a call that would not touch a workspace runs as iex_spmm_ex does (a forced family 7 fails there), and so does an fp32 one that does not ask for
  // the product by parts: programs run such calls side by side, which the shared array would make a race
  if (need == 0 || (dtype == IEX_F32 && ((flags >> 16) & 0xf) == 0))
    return spmm_dispatch(dtype, itype, flags, m, k, n, nonzeros, row_indices, values, row_offsets, column_indices, dense,
                         bias, out, stream, batch, nullptr, 0);
  IEX_REQUIRE(need <= kStaticScratchBytes, IEX_ERR_TOO_LARGE,
              "spmm (static scratch): this call needs %zu bytes of scratch memory, the library's array holds %zu "
              "(pass a workspace of your own to iex_spmm_ws, or call iex_spmm_ex)", need, kStaticScratchBytes);
  void* ws = nullptr;
  if (int rc = static_scratch(&ws)) return rc;
  return spmm_dispatch(dtype, itype, flags, m, k, n, nonzeros, row_indices, values, row_offsets, column_indices, dense,
                       bias, out, stream, batch, ws, kStaticScratchBytes);
}

size_t iex_spmm_static_scratch_bytes(void) { return iex::kStaticScratchBytes; }

int iex_spmm_ex(int dtype, int itype, int flags, int m, int k, int n, int nonzeros,
                const int* row_indices, const void* values, const int* row_offsets,
                const void* column_indices, const void* dense, const float* bias, void* out,
                void* stream, int batch) {
  return iex::spmm_dispatch(dtype, itype, flags, m, k, n, nonzeros, row_indices, values, row_offsets,
                            column_indices, dense, bias, out, stream, batch, nullptr, 0);
}

int iex_spmm_ws(int dtype, int itype, int flags, int m, int k, int n, int nonzeros,
                const int* row_indices, const void* values, const int* row_offsets,
                const void* column_indices, const void* dense, const float* bias, void* out,
                void* stream, int batch, void* workspace, size_t workspace_bytes) {
  return iex::spmm_dispatch(dtype, itype, flags, m, k, n, nonzeros, row_indices, values, row_offsets,
                            column_indices, dense, bias, out, stream, batch, workspace, workspace_bytes);
}

int iex_spmm_aux(int dtype, int itype, int flags, int m, int k, int n, int nonzeros, const int* row_indices, const void* values,
                 const int* row_offsets, const void* column_indices, const void* dense, const void* aux, int aux_mode, void* out,
                 void* stream, int batch, void* workspace, size_t workspace_bytes, const int* row_histogram) {
  using namespace iex;
  IEX_REQUIRE(dtype == IEX_F16 || dtype == IEX_BF16, IEX_ERR_UNSUPPORTED, "spmm: an auxiliary operand goes with fp16 / bf16");
  IEX_REQUIRE(!(flags & (IEX_SPMM_PER_BATCH_VALUES | IEX_SPMM_ACCUMULATE | IEX_SPMM_RELU)), IEX_ERR_UNSUPPORTED,
              "spmm: an auxiliary operand goes with shared values, a plain store and no ReLU");
  IEX_REQUIRE(aux && (aux_mode == kGemmAdd || aux_mode == kGemmTimesSilu), IEX_ERR_BAD_ARGUMENT, "spmm: null auxiliary operand or unknown mode %d", aux_mode);
  bool done = false;
  if (int rc = spmm_dispatch(dtype, itype, flags, m, k, n, nonzeros, row_indices, values, row_offsets, column_indices, dense, nullptr, out, stream, batch,
                             workspace, workspace_bytes, row_histogram, aux, aux_mode, &done))
    return rc;
  const size_t total = (size_t)m * n * batch;
  if (done || total == 0) return 0;
  note_kernel("combine_kernel");
  auto kernel = dtype == IEX_BF16 ? combine_kernel<true> : combine_kernel<false>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)((total + 2047) / 2048)), dim3(256), 0, static_cast<hipStream_t>(stream), total,
                     static_cast<const uint16_t*>(aux), aux_mode, static_cast<uint16_t*>(out));
  return check_hip(hipGetLastError(), "spmm combine launch");
}

int iex_spmm_sched(int dtype, int itype, int flags, int m, int k, int n, int nonzeros,
                   const int* row_indices, const void* values, const int* row_offsets,
                   const void* column_indices, const void* dense, const float* bias, void* out,
                   void* stream, int batch, void* workspace, size_t workspace_bytes, const int* row_histogram) {
  return iex::spmm_dispatch(dtype, itype, flags, m, k, n, nonzeros, row_indices, values, row_offsets,
                            column_indices, dense, bias, out, stream, batch, workspace, workspace_bytes, row_histogram);
}

size_t iex_spmm_workspace_bytes(int dtype, int itype, int flags, int m, int k, int n, int nonzeros, int batch) {
  return iex::spmm_workspace_bytes(dtype, itype, flags, m, k, n, nonzeros, batch);
}

int iex_spmm_workspace_kind(int dtype, int itype, int flags, int m, int k, int n, int nonzeros, int batch) {
  return iex::spmm_workspace_kind(dtype, itype, flags, m, k, n, nonzeros, batch);
}

size_t iex_spmm_transposed_workspace_bytes(int dtype, int m, int k, int n, int nonzeros) {
  return iex::spmm_transposed_workspace_bytes(dtype, m, k, n, nonzeros);
}

int iex_spmm_transposed(int dtype, int itype, int m, int k, int n, int nonzeros, const void* values, const int* row_offsets, const void* column_indices,
                        const void* dense, void* out, void* stream, void* workspace, size_t workspace_bytes) {
  return iex::spmm_transposed(dtype, itype, m, k, n, nonzeros, values, row_offsets, column_indices, dense, out, static_cast<hipStream_t>(stream), workspace,
                              workspace_bytes);
}

int iex_CudaSpmm2(int m, int k, int n, int nonzeros, const int* row_indices, const float* values,
                  const int* row_offsets, const int* column_indices, const float* dense_matrix,
                  float* output_matrix, void* stream, int batch_size) {
  return iex::spmm_dispatch(IEX_F32, IEX_I32, IEX_SPMM_PER_BATCH_VALUES | IEX_SPMM_ACCUMULATE | IEX_SPMM_ANY_COLUMN_ORDER, m, k, n,
                            nonzeros, row_indices, values, row_offsets, column_indices, dense_matrix,
                            nullptr, output_matrix, stream, batch_size, nullptr, 0);
}

int iex_CudaSpmm3(int m, int k, int n, int nonzeros, const int* row_indices, const float* values,
                  const int* row_offsets, const int* column_indices, const float* dense_matrix,
                  float* output_matrix, void* stream, int batch_size) {
  return iex::spmm_dispatch(IEX_F32, IEX_I32, IEX_SPMM_ANY_COLUMN_ORDER, m, k, n, nonzeros, row_indices, values, row_offsets,
                            column_indices, dense_matrix, nullptr, output_matrix, stream, batch_size, nullptr, 0);
}

int iex_CudaSpmm5(int m, int k, int n, int nonzeros, const int* row_indices, const uint16_t* values,
                  const int* row_offsets, const int16_t* column_indices, const uint16_t* dense_matrix,
                  uint16_t* output_matrix, void* stream, int batch_size) {
  return iex::spmm_dispatch(IEX_F16, IEX_I16, IEX_SPMM_ANY_COLUMN_ORDER, m, k, n, nonzeros, row_indices, values, row_offsets,
                            column_indices, dense_matrix, nullptr, output_matrix, stream, batch_size, nullptr, 0);
}

}  // extern "C"
