// fp32 product on the bf16 matrix cores (gfx950): every fp32 entry is the sum of three bf16 parts (high, middle, low: 8 significant bits
// each, rounded to nearest, so that the three hold all 24), and C = A * B is taken as the six products of parts that reach into
// an fp32 result: high * high, high * middle, middle * high, middle * middle, high * low, low * high.  What is left out (middle *
// low, low * low) is below 2^-26 of a product.  bf16 MFMAs run at 16 times the rate of fp32 ones, so six of them per product are
// 2.7 times faster, and a fragment that is in registers serves three of them: LDS and L2 move half of what six
// separate products would.
// MI355X, us (and TFLOP/s of bf16 MFMAs): 4096 x 2048 x 4096 297 (1390), B as (N, K) 285 (1448); 4096 x 1024 x 4096 149 (1388): the rates
// of this library's 16-bit tiles, under the same power limit.  fp32 MFMAs at their peak would take 440 and 220.
//
// Accuracy (2-norm against 64 bits, normal entries, 20 % of A nonzero, k = 4096): 8.8e-8; a chain of fp32 multiply-adds over the nonzeros alone 3.6e-7.  Three sets of
// sums: high * high, which is flushed into a total every FLUSH steps (its roundings are relative to a stretch's sum), and the other five
// products, 2^-8 of it and less, in a set of their own.
//
// Tile: 128 x 128 by four wavefronts (2 x 2 of 64 x 64), one workgroup per CU, steps of 32 k, three stages of 48 KB.  Operand layout
// in LDS, chunk permutations, direct loads and hand-written waits follow gemm_dma_device.cuh.  A step is 96 MFMAs a wavefront; what
// else there is stands between them, one at a time: four fragments per product are read for the next step into registers
// that the products before have freed (high of A and low of B, which are needed to the end, have two sets), and from the barrier on, in the
// middle of the first product, the direct loads of tile t + STAGES go into the stage of tile t, whose last fragments everybody has
// then read.  (Fragments read a whole product ahead in blocks: 1100 TFLOP/s; all fragments in two sets, which the
// compiler moves between register files: 1290 - 1350.)
// Few tiles: K in parts, every part's sums in a matrix of their own; the kernel that comes next anyway (the check of the operands' range, or the
// sampling) adds them up in their order.  (4096 x 256 x 4096 in four parts, us: the workgroup that draws a tile's last ticket reading
// the others' sums, as in gemm_dma_device.cuh, 54; this way 47, and 3.5 in the next kernel.)
// Every workgroup looks at the range of the operands' entries (10 KB, a word per workgroup that made parts) while its first tiles are on their way, and ends where
// the product would not stand for the fp32 one: 4096 x 256 x 4096 47.7 -> 48.8 us, 5 where it ends, and the kernel behind it reads one word (7.6 -> 4.2).
// Requirements (the caller's, who makes the planes): K a multiple of 32, planes zero where the operands end, row strides
// multiples of 8, 16-byte aligned planes, three of them within 4 GB.
#pragma once
#include "gemm_split.h"
#include "gemm_dma_device.cuh"
#include "gemm_pp_device.cuh"

namespace iex {

template <int WM, int WN, int STAGES>
constexpr int gemm_split_lds_bytes() { return STAGES * 3 * (2 * WM * 32 + 2 * WN * 32) * 64 + kSplitVerdict * 4 + 32; }

// Whether the product of the parts stands for the fp32 one, by all 256 threads from the ranges' words in LDS, eight words of room behind them.  (An array of this
// function's own would come first in LDS and shift the stages off the 128 bytes that direct loads write at a time: 4096 x 1024 x 4096 147 -> 154 us.)
__device__ __forceinline__ bool split_stands(const SplitParams& p, unsigned* words) {
  SplitRange a, b;
#pragma unroll
  for (int i = 0; i < kSplitVerdict; i += 256) {
    const int at = (i < kSplitSlots ? i : i - kSplitSlots) + threadIdx.x;
    if (at < (i < kSplitSlots ? p.slots_b : p.slots_a)) (i < kSplitSlots ? b : a).add_word(words[i + threadIdx.x]);
  }
  a.over_wave(), b.over_wave();
  unsigned* of = words + kSplitVerdict;
  if (lane_id() == 0) of[threadIdx.x >> 6] = a.word(), of[4 + (threadIdx.x >> 6)] = b.word();
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 4; ++w) a.add_word(of[w]), b.add_word(of[4 + w]);
  return split_range_ok(a, b) && !(p.finite && (a.odd || b.odd));
}

// One tile's stretch `part` of K.  TRANS_B: B is (N, K), else (K, N).
template <bool TRANS_B, int WM, int WN, int STAGES, int FLUSH>
__device__ __forceinline__ void gemm_split_tile(const SplitParams& p, int tile_m, int tile_n, int z, int part, unsigned char* smem) {
  constexpr int BM = 2 * WM * 32, BN = 2 * WN * 32, WAVES = 4;
  constexpr int A_PLANE = BM * 64, B_PLANE = BN * 64, STAGE_BYTES = 3 * (A_PLANE + B_PLANE);
  constexpr int A_INSTR = A_PLANE / 1024 / WAVES, B_INSTR = B_PLANE / 1024 / WAVES, LOADS = 3 * (A_INSTR + B_INSTR);
  constexpr int ROWS = 2 * WM, COLS = 2 * WN;
  typedef unsigned short u16;
  typedef __attribute__((address_space(3))) unsigned char lds_u8;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / 2, wn = wave % 2;
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int steps = p.K / 32, per = (steps + p.parts - 1) / p.parts, first = part * per, KT = min(per, steps - first);
  const u16* A = static_cast<const u16*>(p.A);
  const u16* B = static_cast<const u16*>(p.B) + (size_t)z * p.stride_b;
  const unsigned lds0 = (unsigned)(size_t)(lds_u8*)smem;
  const u32x4 a_buf = buffer_of(A + (size_t)m0 * p.lda, 2 * (size_t)p.plane_a + rows_bytes(p.M - m0, p.K, p.lda));
  const u32x4 b_buf = TRANS_B ? buffer_of(B + (size_t)n0 * p.ldb, 2 * (size_t)p.plane_b + rows_bytes(p.N - n0, p.K, p.ldb))
                              : buffer_of(B, 2 * (size_t)p.plane_b + rows_bytes(p.K, p.N, p.ldb));
  unsigned a_lane[A_INSTR], b_lane[B_INSTR];
#pragma unroll
  for (int q = 0; q < A_INSTR; ++q)
    a_lane[q] = row_chunk<32>(wave * A_INSTR + q, lane, p.M - m0, p.lda).offset;
#pragma unroll
  for (int q = 0; q < B_INSTR; ++q)
    b_lane[q] = (TRANS_B ? row_chunk<32>(wave * B_INSTR + q, lane, p.N - n0, p.ldb) : column_chunk<BN>(wave * B_INSTR + q, lane, n0, p.ldb)).offset;
  const unsigned a_step = 64u, b_step = (TRANS_B ? 32u : 32u * p.ldb) * 2u;
  auto issue_one = [&](int kt, unsigned stage, int q) {
    const unsigned t = first + min(kt, KT - 1);
    if (q < 3 * A_INSTR) {
      const int plane = q / A_INSTR, i = q % A_INSTR;
      lds_dma16(a_buf, a_lane[i], t * a_step + plane * p.plane_a, __builtin_amdgcn_readfirstlane(lds0 + stage + plane * A_PLANE + (wave * A_INSTR + i) * 1024));
    } else {
      const int plane = (q - 3 * A_INSTR) / B_INSTR, i = (q - 3 * A_INSTR) % B_INSTR;
      lds_dma16(b_buf, b_lane[i], t * b_step + plane * p.plane_b, __builtin_amdgcn_readfirstlane(lds0 + stage + 3 * A_PLANE + plane * B_PLANE + (wave * B_INSTR + i) * 1024));
    }
  };
  const int frow = lane & 15, fch = lane >> 4, fsw = frow >> 2;
  const int a_off = (wm * WM * 32 + frow) * 64 + ((fch ^ fsw) * 16);
  int b_off[TRANS_B ? 1 : COLS];
  if constexpr (TRANS_B) b_off[0] = (wn * WN * 32 + frow) * 64 + ((fch ^ fsw) * 16);
  else {
#pragma unroll
    for (int j = 0; j < COLS; ++j) b_off[j] = kn16_fragment_offset<BN>(lane, wn * COLS + j);
  }
  f32x4 hi[ROWS][COLS], lo[ROWS][COLS], sum[ROWS][COLS];
#pragma unroll
  for (int i = 0; i < ROWS; ++i)
#pragma unroll
    for (int j = 0; j < COLS; ++j) hi[i][j] = lo[i][j] = sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 ah[2][ROWS], am[ROWS], al[ROWS], bh[COLS], bm[COLS], bl[2][COLS];
  constexpr int NM = ROWS * COLS;
  auto read_a = [&](const unsigned char* st, auto plane, u32x4& f, int i) {
    f = *reinterpret_cast<const u32x4*>(st + decltype(plane)::value * A_PLANE + a_off + i * 16 * 64);
  };
  auto read_b = [&](const unsigned char* st, auto plane, u32x4& f, int j) {
    if constexpr (TRANS_B) f = *reinterpret_cast<const u32x4*>(st + 3 * A_PLANE + decltype(plane)::value * B_PLANE + b_off[0] + j * 16 * 64);
    else f = kn_fragment<BN * 2>(st + 3 * A_PLANE + decltype(plane)::value * B_PLANE + b_off[j]);
  };
  const std::integral_constant<int, 0> high;
  const std::integral_constant<int, 1> middle;
  const std::integral_constant<int, 2> low;
  // the ranges' words, then the first tiles
  static_assert(kSplitVerdict * 4 % 1024 == 0, "whole direct loads");
  const u32x4 word_buf = buffer_of(p.ranges, kSplitVerdict * 4);
#pragma unroll
  for (int q = 0; q < (kSplitVerdict * 4 / 1024 + WAVES - 1) / WAVES; ++q) {
    const unsigned at = min(q * WAVES + wave, kSplitVerdict * 4 / 1024 - 1) * 1024;   // (some come twice)
    lds_dma16(word_buf, lane * 16, at, __builtin_amdgcn_readfirstlane(lds0 + STAGES * STAGE_BYTES + at));
  }
#pragma unroll
  for (int s = 0; s < STAGES; ++s)
#pragma unroll
    for (int q = 0; q < LOADS; ++q) issue_one(s, s * STAGE_BYTES, q);
  wait_vmcnt<(STAGES - 1) * LOADS>();
  __syncthreads();
  const bool stands = split_stands(p, reinterpret_cast<unsigned*>(smem + STAGES * STAGE_BYTES));
  if (blockIdx.x == 0 && blockIdx.y == 0 && tid == 0) p.ranges[kSplitVerdict] = stands;
  if (!stands) {   // (uniform)
    wait_vmcnt<0>();   // nothing may still be writing LDS when the workgroup ends
    return;
  }
#pragma unroll
  for (int i = 0; i < ROWS; ++i) read_a(smem, low, al[i], i), read_a(smem, high, ah[0][i], i), read_a(smem, middle, am[i], i);
#pragma unroll
  for (int j = 0; j < COLS; ++j) read_b(smem, high, bh[j], j), read_b(smem, low, bl[0][j], j), read_b(smem, middle, bm[j], j);
  unsigned now = 0;
  auto step = [&](int kt, auto parity) {
    constexpr int set = decltype(parity)::value;
    const unsigned next = now == (STAGES - 1) * STAGE_BYTES ? 0 : now + STAGE_BYTES;
    const unsigned char* st = smem + next;
    for_each_number<6 * NM>([&](auto number) {
      constexpr int x = decltype(number)::value, product = x / NM, y = x % NM, i = y / COLS, j = y % COLS;
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (product == 0) lo[i][j] = mfma_16x16x32<true>(bh[j], al[i], lo[i][j]);
      if constexpr (product == 1) hi[i][j] = mfma_16x16x32<true>(bh[j], ah[set][i], hi[i][j]);
      if constexpr (product == 2) lo[i][j] = mfma_16x16x32<true>(bh[j], am[i], lo[i][j]);
      if constexpr (product == 3) lo[i][j] = mfma_16x16x32<true>(bm[j], am[i], lo[i][j]);
      if constexpr (product == 4) lo[i][j] = mfma_16x16x32<true>(bm[j], ah[set][i], lo[i][j]);
      if constexpr (product == 5) lo[i][j] = mfma_16x16x32<true>(bl[set][j], ah[set][i], lo[i][j]);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (x == NM / 2 - 1) {
        wait_vmcnt<(STAGES - 2) * LOADS>();   // my loads of tile kt + 1 have landed
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
      if constexpr (product == 0 && y >= NM / 2 && (y - NM / 2) % (NM / 2 / ROWS) == 0) read_a(st, high, ah[set ^ 1][(y - NM / 2) / (NM / 2 / ROWS)], (y - NM / 2) / (NM / 2 / ROWS));
      if constexpr (product == 1 && y % (NM / ROWS) == 0) read_a(st, low, al[y / (NM / ROWS)], y / (NM / ROWS));
      if constexpr (product == 2 && y % (NM / COLS) == 0) read_b(st, low, bl[set ^ 1][y / (NM / COLS)], y / (NM / COLS));
      if constexpr (product == 3 && y % (NM / COLS) == 0) read_b(st, high, bh[y / (NM / COLS)], y / (NM / COLS));
      if constexpr (product == 4 && y % (NM / ROWS) == 0) read_a(st, middle, am[y / (NM / ROWS)], y / (NM / ROWS));
      if constexpr (product == 5 && y % (NM / COLS) == 0) read_b(st, middle, bm[y / (NM / COLS)], y / (NM / COLS));
      for_each_number<LOADS>([&](auto qn) { constexpr int q = decltype(qn)::value; if constexpr (NM + q * 5 * NM / LOADS + 2 == x) issue_one(kt + STAGES, now, q); });
    });
    now = next;
  };
  const std::integral_constant<int, 0> even;
  const std::integral_constant<int, 1> odd;
  int kt = 0;
  while (kt + 2 <= KT) {
    const int upto = min(kt + FLUSH, KT - 1);
    for (; kt < upto; kt += 2) {
      step(kt, even);
      step(kt + 1, odd);
    }
#pragma unroll
    for (int i = 0; i < ROWS; ++i)
#pragma unroll
      for (int j = 0; j < COLS; ++j) {
        sum[i][j] += hi[i][j];
        hi[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
  }
  if (kt < KT) step(kt, even);
  wait_vmcnt<0>();
#pragma unroll
  for (int i = 0; i < ROWS; ++i)
#pragma unroll
    for (int j = 0; j < COLS; ++j) hi[i][j] = sum[i][j] + hi[i][j] + lo[i][j];
  float* C = p.C + (size_t)z * p.stride_c + (size_t)part * p.stride_part;
  typedef f32x4 f32x4u __attribute__((aligned(4)));   // (rows of any length)
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    const int row = m0 + wm * WM * 32 + i * 16 + frow;
    if (row >= p.M) continue;
    const float bias = p.row_bias ? p.row_bias[row] : 0.f;
#pragma unroll
    for (int j = 0; j < COLS; ++j) {
      const int col = n0 + wn * WN * 32 + j * 16 + fch * 4;
      f32x4 x = hi[i][j];
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = p.relu ? fmaxf(x[e] + bias, 0.f) : x[e] + bias;
      float* at = C + (size_t)row * p.ldc + col;
      if (col + 4 <= p.N) {
        *reinterpret_cast<f32x4u*>(at) = x;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (col + e < p.N) at[e] = x[e];
      }
    }
  }
}

}  // namespace iex
