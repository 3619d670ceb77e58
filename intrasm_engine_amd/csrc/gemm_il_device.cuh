// Dense GEMM tile for gfx950 by eight wavefronts in phase, every instruction that is not an MFMA set between two of them.
//
// One barrier per 32 k.  A wavefront owns WM x WN blocks of 32 x 32 (WN = 2: 8 * WM MFMAs a step, four per row block of 16).
// Between the four MFMAs of a row block go one fragment of A (for AHEAD row blocks later, a ring of RING registers), in the
// second half of a step the fragments of the next step's B (two register sets), and the direct loads (global memory -> LDS) of
// a later tile, one at a time.  An MFMA of 16 cycles then covers what follows it, and no block of LDS reads has to fit behind the
// other group's MFMAs as in gemm_pp_device.cuh.  Whether that is the faster tile depends on how much there is besides the MFMAs
// (MI355X, bf16, normal operands, us alternating phases -> interleaved, the shapes of both directions of a product):
//   A as (K, M)   8192 x 8192 x 8192, 256 rows 773 -> 750;  4096 x 4096 x 2048, 256 rows 58.3 -> 54.8, 128 rows 74.0 -> 65.9;
//                 4096 x 2048 x 11008, 128 rows 165 -> 152   (fragments of A take two transposing LDS reads each)
//   192 rows      11008 x 2048 x 4096 150.0 -> 146.8, B as (N, K) 146.8 -> 144.0;  8192 x 8192 x 4096 428 -> 422
// and the other way round, so that these stay with the alternating phases:
//   256 rows      8192 x 8192 x 8192 715 -> 740, B as (N, K) 729 -> 742;  4096 x 8192 x 11008 487 -> 504
//   128 rows      4096 x 2048 x 4096 59.9 -> 60.9, B as (N, K) 57.1 -> 59.0   (with six stages of B and four of A 60.2, 60.3)
// What bounds it: the matrix cores at the clock that the card's power limit leaves them, as there; a single round of tiles also
// prologue and epilogue.
//
// Stages: A 64 k at a time (a K-contiguous row is then a whole line), three of them; B 32 k at a time, four.  The window of step
// t, from the middle of that step to the middle of the next, loads A tile t / 2 + 2 (even t) into the stage of A tile
// t / 2 - 1, whose last fragments were multiplied in step t - 1, and B tile t + 4 into the stage of B tile t, whose fragments
// were all in registers when step t began.  The barrier in the middle of step t stands between those uses, by every
// wavefront, and the loads.  What is read behind it (B tile t + 1, and the A tile of that step) was loaded in window t - 3
// or before: what may still fly at the wait before the barrier is windows t - 2 and t - 1.
// Per accumulator the MFMAs run in the same k order as in the other tiles: results are bit-equal.
#pragma once
#include "gemm_dma_device.cuh"

namespace iex {

template <int WM, int WN, int WCN>
constexpr int gemm_il_lds_bytes() { return 3 * (2 * WM * 32) * 128 + 4 * (WCN * WN * 32) * 64; }

template <bool BF16, bool TRANS_B, int WM, int WN, int WCN, bool TRANS_A>
__device__ __forceinline__ void gemm_tile_il(const GemmParams& p, int tile_m, int tile_n, int z, unsigned char* smem) {
  constexpr int BM = 2 * WM * 32, BN = WCN * WN * 32, WAVES = 2 * WCN;
  constexpr int SA = 3, SB = 4;   // stages
  constexpr int A_STAGE = BM * 128, B_STAGE = BN * 64, A_BASE = SB * B_STAGE;
  constexpr int ROWS = 2 * WM, COLS = 2 * WN;
  constexpr int RING = WM == 3 ? 3 : 4, AHEAD = WM == 4 ? 3 : 2;
  constexpr int A_INSTR = A_STAGE / 1024 / WAVES, B_INSTR = B_STAGE / 1024 / WAVES;   // per wavefront: A tile of 64 k, B tile of 32 k
  constexpr int FLY = A_INSTR + 2 * B_INSTR;   // loads of two windows
  static_assert(FLY + A_INSTR + B_INSTR < 64, "loads in flight must fit the load counter");
  static_assert(WAVES == 8 && COLS == 4, "eight wavefronts, four MFMAs a row block");
  static_assert(A_STAGE % (1024 * WAVES) == 0 && B_STAGE % (1024 * WAVES) == 0, "every wavefront fetches whole kilobytes of A and of B");
  static_assert(ROWS % RING == 0 && AHEAD < RING && AHEAD <= WM, "the next step's A is read behind the barrier, and no fragment before its last use");
  static_assert(!TRANS_A || BM == 128 || BM == 256, "(K,M) layout: chunks per k row are a power of two");
  typedef unsigned short u16;
  typedef __attribute__((address_space(3))) unsigned char lds_u8;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WCN, wn = wave % WCN;
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const u16* __restrict__ A = static_cast<const u16*>(p.A) + (size_t)z * p.stride_a;
  const u16* __restrict__ B = static_cast<const u16*>(p.B) + (size_t)z * p.stride_b;
  u16* __restrict__ C = static_cast<u16*>(p.C) + (size_t)z * p.stride_c;
  const unsigned lds0 = (unsigned)(size_t)(lds_u8*)smem;
  const int lda = p.lda ? p.lda : TRANS_A ? p.M : p.K, ldb = p.ldb ? p.ldb : TRANS_B ? p.K : p.N;
  const int kb = p.kb ? p.kb : p.K;   // the k rows of a (K,N) B
  const u32x4 a_buf = TRANS_A ? buffer_of(A, rows_bytes(p.K, p.M, lda)) : buffer_of(A + (size_t)m0 * lda, rows_bytes(p.M - m0, p.K, lda));
  const u32x4 b_buf = TRANS_B ? buffer_of(B + (size_t)n0 * ldb, rows_bytes(p.N - n0, p.K, ldb)) : buffer_of(B, rows_bytes(kb, p.N, ldb));
  unsigned a_lane[A_INSTR], b_lane[B_INSTR];
  int a_k8[A_INSTR], b_k8[B_INSTR];
#pragma unroll
  for (int q = 0; q < A_INSTR; ++q) {
    DirectChunk c;
    if constexpr (TRANS_A) c = column_chunk<BM>(wave * A_INSTR + q, lane, m0, lda);
    else c = row_chunk<64>(wave * A_INSTR + q, lane, p.M - m0, lda);
    a_lane[q] = c.offset, a_k8[q] = c.k;
  }
#pragma unroll
  for (int q = 0; q < B_INSTR; ++q) {
    DirectChunk c;
    if constexpr (TRANS_B) c = row_chunk<32>(wave * B_INSTR + q, lane, p.N - n0, ldb);
    else c = column_chunk<BN>(wave * B_INSTR + q, lane, n0, ldb);
    b_lane[q] = c.offset, b_k8[q] = c.k;
  }
  const int P = (p.K + 31) / 32, TA = (p.K + 63) / 64;
  const unsigned a_step = (TRANS_A ? 64u * lda : 64u) * 2u, b_step = (TRANS_B ? 32u : 32u * ldb) * 2u;
  auto issue_a = [&](int t, unsigned stage, int q) {
    lds_dma16(a_buf, a_lane[q], (unsigned)min(t, TA - 1) * a_step, __builtin_amdgcn_readfirstlane(lds0 + stage + (wave * A_INSTR + q) * 1024));
  };
  auto issue_b = [&](int t, unsigned stage, int q) {
    lds_dma16(b_buf, b_lane[q], (unsigned)min(t, P - 1) * b_step, __builtin_amdgcn_readfirstlane(lds0 + stage + (wave * B_INSTR + q) * 1024));
  };
  Acc16<WM, WN> acc;
  acc.clear();
  const int frow = lane & 15, fch = lane >> 4;
  int a_off[TRANS_A ? ROWS : 2];
  if constexpr (TRANS_A) {
#pragma unroll
    for (int i = 0; i < ROWS; ++i) a_off[i] = kn16_fragment_offset<BM>(lane, wm * ROWS + i);
  } else {
#pragma unroll
    for (int h = 0; h < 2; ++h) a_off[h] = (wm * WM * 32 + frow) * 128 + (((h * 4 + fch) ^ (frow >> 1)) * 16);
  }
  int b_off[TRANS_B ? 1 : COLS];
  if constexpr (TRANS_B) b_off[0] = (wn * WN * 32 + frow) * 64 + ((fch ^ (frow >> 2)) * 16);
  else {
#pragma unroll
    for (int j = 0; j < COLS; ++j) b_off[j] = kn16_fragment_offset<BN>(lane, wn * COLS + j);
  }
  u32x4 fa[RING], fb[2][COLS];
  auto read_a = [&](unsigned stage, int h, int i) {
    if constexpr (TRANS_A) fa[i % RING] = kn_fragment<BM * 2>(smem + stage + a_off[i] + h * 32 * (BM * 2));
    else fa[i % RING] = *reinterpret_cast<const u32x4*>(smem + stage + a_off[h] + i * 16 * 128);
  };
  auto read_b = [&](unsigned stage, int set, int j) {
    if constexpr (TRANS_B) fb[set][j] = *reinterpret_cast<const u32x4*>(smem + stage + b_off[0] + j * 16 * 64);
    else fb[set][j] = kn_fragment<BN * 2>(smem + stage + b_off[j]);
  };
  // entries at k >= K must be zero: what was loaded there is other data (done by the lanes that loaded it)
  auto zero_b = [&](int t, unsigned stage) {
#pragma unroll
    for (int q = 0; q < B_INSTR; ++q)
      if (t * 32 + b_k8[q] >= p.K) *reinterpret_cast<u32x4*>(smem + stage + ((wave * B_INSTR + q) * 64 + lane) * 16) = u32x4{0u, 0u, 0u, 0u};
  };
  auto zero_a = [&](int t, unsigned stage) {
#pragma unroll
    for (int q = 0; q < A_INSTR; ++q)
      if (t * 64 + a_k8[q] >= p.K) *reinterpret_cast<u32x4*>(smem + stage + ((wave * A_INSTR + q) * 64 + lane) * 16) = u32x4{0u, 0u, 0u, 0u};
  };
  const bool tail = p.K % 64 != 0;
  // of step t: the stages of A tiles t / 2 - 1, t / 2, t / 2 + 1 and of B tiles t - 1, t, t + 1
  unsigned a_prev = A_BASE + (SA - 1) * A_STAGE, a_now = A_BASE, a_next = A_BASE + A_STAGE;
  unsigned b_prev = (SB - 1) * B_STAGE, b_now = 0, b_next = B_STAGE;
  auto step = [&](int t, auto parity) {
    constexpr int set = decltype(parity)::value;   // t % 2
    for_each_number<ROWS>([&](auto row_block) {
      constexpr int i = decltype(row_block)::value, late = i >= WM;
      auto multiply = [&](auto column) {
        constexpr int j = decltype(column)::value;
        __builtin_amdgcn_sched_barrier(0);
        acc.v[i][j] = mfma_16x16x32<BF16>(fb[set][j], fa[i % RING], acc.v[i][j]);
        __builtin_amdgcn_sched_barrier(0);
      };
      multiply(std::integral_constant<int, 0>{});
      if constexpr (i == WM) {
        wait_vmcnt<FLY>();
        if (tail) {
          if (t + 2 == P) zero_b(t + 1, b_next);
          if (set == 1 && t / 2 + 2 == TA) zero_a(t / 2 + 1, a_next);
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
      if constexpr (i + AHEAD < ROWS) read_a(a_now, set, i + AHEAD);
      else read_a(set ? a_next : a_now, set ^ 1, i + AHEAD - ROWS);
      multiply(std::integral_constant<int, 1>{});
      if constexpr (late) {
#pragma unroll
        for (int j = (i - WM) * COLS / WM; j < (i - WM + 1) * COLS / WM; ++j) read_b(b_next, set ^ 1, j);
      }
      multiply(std::integral_constant<int, 2>{});
      // the second half of a step begins its window, the first half ends the one before
      {
        constexpr int slot = late ? i - WM : i + WM;
        constexpr bool a_window = late ? set == 0 : set == 1;
        constexpr int N = a_window ? A_INSTR + B_INSTR : B_INSTR;
        for_each_number<N>([&](auto number) {
          constexpr int n = decltype(number)::value;
          if constexpr (n * ROWS / N == slot) {
            if constexpr (a_window && n < A_INSTR) issue_a((late ? t : t - 1) / 2 + SA - 1, a_prev, n);
            else issue_b(late ? t + SB : t + SB - 1, late ? b_now : b_prev, n - (a_window ? A_INSTR : 0));
          }
        });
      }
      multiply(std::integral_constant<int, 3>{});
    });
    b_prev = b_now, b_now = b_next, b_next = b_next == (SB - 1) * B_STAGE ? 0 : b_next + B_STAGE;
    if constexpr (set == 1) a_prev = a_now, a_now = a_next, a_next = a_next == A_BASE + (SA - 1) * A_STAGE ? A_BASE : a_next + A_STAGE;
  };
  // prologue: what the windows before step 0 would have loaded, but for the part of the last one that step 0's first half issues
  constexpr int EARLY = (B_INSTR + 1) / 2;
#pragma unroll
  for (int q = 0; q < A_INSTR; ++q) issue_a(0, a_now, q);
#pragma unroll
  for (int q = 0; q < B_INSTR; ++q) issue_b(0, b_now, q);
#pragma unroll
  for (int w = 1; w < SB; ++w) {   // (a window's A tile goes out before its B tile)
    if (w % 2 == 0 && w / 2 < SA - 1) {
#pragma unroll
      for (int q = 0; q < A_INSTR; ++q) issue_a(w / 2, A_BASE + w / 2 * A_STAGE, q);
    }
#pragma unroll
    for (int q = 0; q < (w == SB - 1 ? EARLY : B_INSTR); ++q) issue_b(w, w * B_STAGE, q);
  }
  wait_vmcnt<(SB - 2) * B_INSTR + EARLY + (SA - 2) * A_INSTR>();   // A tile 0, B tile 0
  if (tail) {
    if (P == 1) zero_b(0, b_now);
    if (TA == 1) zero_a(0, a_now);
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < COLS; ++j) read_b(b_now, 0, j);
#pragma unroll
  for (int i = 0; i < AHEAD; ++i) read_a(a_now, 0, i);
  const std::integral_constant<int, 0> even;
  const std::integral_constant<int, 1> odd;
  int t = 0;
  for (; t + 2 <= P; t += 2) {
    step(t, even);
    step(t + 1, odd);
  }
  if (t < P) step(t, even);
  wait_vmcnt<0>();   // the re-fetched last tiles: nothing may still be writing LDS when the stages are reused
  static_assert(WAVES * gemm_store_lds_bytes<WN>() <= gemm_il_lds_bytes<WM, WN, WCN>(), "the epilogue fits the stages");
  __syncthreads();
  const u16* aux = p.aux ? static_cast<const u16*>(p.aux) + (size_t)z * p.stride_c : nullptr;
  gemm_store_tile<BF16, WM, WN>(p, acc, C, aux, m0, n0, wm, wn, lane, smem + wave * gemm_store_lds_bytes<WN>(), p.stream_out != 0);
}
}  // namespace iex
