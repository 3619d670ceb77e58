// Dense GEMM tile for gfx950 by eight wavefronts in two groups that alternate roles ("ping-pong").
//
// The direct-load tile of gemm_dma_device.cuh interleaves three things in one instruction stream: MFMAs,
// LDS reads of the next operand fragments and the direct loads of a later tile.  Every wait of that
// stream (fragments not there yet, my loads of the next tile not landed, the barrier) is a bubble in the
// matrix pipeline of its SIMD, because nothing else runs there.  Here a SIMD holds two wavefronts, one of
// each group, and the groups run half a K step apart:
//
//     interval      2p-1          2p            2p+1          2p+2
//     group 0       M(p)          C(p)          M(p+1)        C(p+1)
//     group 1       C(p-1)        M(p)          C(p)          M(p+1)
//
//   M(p)  = memory phase p: read the operand fragments of 32 k of the tile from LDS into registers,
//           issue my share of the direct loads (global memory -> LDS) of the tile STAGES - 1 ahead;
//   C(p)  = compute phase p: the 4 * WM * WN MFMAs (16 x 16 x 32) on those fragments, nothing else.
// Intervals are separated by workgroup barriers, so on every SIMD one wavefront feeds the matrix cores while
// the other one waits for LDS and issues loads, and all waits hide behind the other group's MFMAs.
// A wavefront owns WM x WN blocks of 32 x 32 (128 x 64 of a 256 x 256 tile with WM = 4, WN = 2, WCN = 4).
// What bounds it (8192^3, bf16): the matrix cores are busy 78 % of the cycles, at the 1.64 GHz that the card's power limit leaves
// them on random operands (MFMAs and nothing else: 1930 TFLOP/s); 14 % of the wavefronts' time is waiting, LDS is in use 31 %.
// One round of 128 x 256 tiles: busy 46 % at 2.25 GHz, a workgroup's only tile being mostly prologue and epilogue.
// (profiles/kernel_counters_of_the_cases.txt.)  One barrier per phase instead of strict alternation: 1315 TFLOP/s for 1440;
// loads before the fragment reads: the same; multiplying at raised priority: 1-2 % slower.
//
// Stage reuse: what phase p reads was last needed by phase p (group 1 reads it one interval after group 0), and the
// loads that overwrite it go out in later M phases.  A wavefront waits for its own loads of what phase p + 1 reads at
// the end of the interval before group 0 reads it (group 0: after C(p), group 1: after M(p)) and the barrier publishes
// them.  Chunk permutations and the hand-written load counts follow gemm_dma_device.cuh; per accumulator the MFMAs
// run in the same k order, so results are bit-equal to that kernel's.
// 192 rows, and A as (K, M), are faster with single instructions between the MFMAs: gemm_il_device.cuh, with the figures of both.
#pragma once
#include "gemm_dma_device.cuh"

namespace iex {

// Stages.  A rows are K-contiguous, and a direct load moves 16 bytes per lane: with 32 k per stage a row is
// 64 bytes, half a cache line, and every line of A crosses the L1 twice, a K step apart (counters on 8192^3: 13.0 GB
// requested from L2 for 8.6 GB of operands, the texture-data unit busy 83 % of the cycles at 20 bytes per clock).  So A is
// staged 64 k at a time (whole lines, three stages), B 32 k at a time (four stages): 3 * BM * 128 + 4 * BN * 64 bytes,
// 160 KB for 256 x 256 tiles.  Phase p reads the half p % 2 of A tile p / 2 and B tile p, and issues half of the loads
// of A tile p / 2 + 2 and all loads of B tile p + 3; every wavefront issues the same number of loads in every two
// phases, so "my loads of everything that phase p + 1 reads have landed" is vmcnt(that number) at the end of phase p.
// KP = 64: phases of 64 k, three stages of A and B tiles of 64 k, tile p + 2 loaded in phase p (one phase's loads may fly at
// its end).  For 128 x 256 tiles: half the rows leave a phase of 32 k too short for what a memory phase has to wait for.
template <int WM, int WN, int WCN, int KP>
constexpr int gemm_pp_lds_bytes() { return 3 * (2 * WM * 32) * 128 + (KP == 32 ? 4 * 64 : 3 * 128) * (WCN * WN * 32); }

template <bool BF16, bool TRANS_B, int WM, int WN, int WCN, int KP = 32>
__device__ __forceinline__ void gemm_tile_pp(const GemmParams& p, int tile_m, int tile_n, int z, unsigned char* smem) {
  constexpr int BM = 2 * WM * 32, BN = WCN * WN * 32, WAVES = 2 * WCN;
  constexpr int SA = 3, SB = KP == 32 ? 4 : 3;        // stages of A (64 k each) and of B (KP each)
  constexpr int A_STAGE = BM * 128, B_STAGE = BN * KP * 2;
  constexpr int B_BASE = SA * A_STAGE;
  constexpr int HALVES = 64 / KP, SUB = KP / 32;      // phases per A tile, MFMA sub-steps per phase
  constexpr int A_INSTR = A_STAGE / 1024 / WAVES;     // direct loads per wavefront and A tile
  constexpr int B_INSTR = B_STAGE / 1024 / WAVES;     // ... and B tile
  // Loads per wavefront that may be in flight where a phase ends: those of two phases (one, for KP = 64).
  constexpr int FLY = A_INSTR + HALVES * B_INSTR;
  constexpr int CPRB = BN / 8;                        // (K,N) layout: chunks per k row
  static_assert(WAVES == 8, "two wavefronts per SIMD");
  static_assert(KP == 32 || KP == 64, "k per phase");
  static_assert(A_INSTR >= HALVES && B_INSTR >= 1 && A_STAGE % (1024 * WAVES) == 0 && B_STAGE % (1024 * WAVES) == 0,
                "every wavefront fetches whole kilobytes of A (in HALVES parts) and of B");
  static_assert(TRANS_B || (CPRB >= 16 && CPRB <= 64), "(K,N) layout: 128 <= BN <= 512");
  static_assert(FLY + A_INSTR + B_INSTR < 64, "loads in flight must fit the load counter");
  typedef unsigned short u16;
  typedef __attribute__((address_space(3))) unsigned char lds_u8;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WCN, wn = wave % WCN;
  const int group = wave / 4;   // wavefronts w and w + 4 share a SIMD (measured: pairing w with w ^ 1 instead loses 15 %)
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const u16* __restrict__ A = static_cast<const u16*>(p.A) + (size_t)z * p.stride_a;
  const u16* __restrict__ B = static_cast<const u16*>(p.B) + (size_t)z * p.stride_b;
  u16* __restrict__ C = static_cast<u16*>(p.C) + (size_t)z * p.stride_c;
  const unsigned lds0 = (unsigned)(size_t)(lds_u8*)smem;
  const int lda = p.lda ? p.lda : p.K, ldb = p.ldb ? p.ldb : TRANS_B ? p.K : p.N;   // row strides
  const int kb = p.kb ? p.kb : p.K;   // the k rows of a (K,N) B

  // ---- what this lane fetches (gemm_addresses.h).  A: 8 rows of 128 bytes per instruction, LDS position (row, c) holds global chunk
  // c ^ ((row >> 1) & 7).  B as (N,K): the same, or 16 rows of 64 bytes, chunk c ^ ((row >> 2) & 3).  B as (K,N): k rows of BN
  // elements, chunk c ^ kn16_swizzle(k).
  // Rows past M (columns past N) are the last one's: they feed rows (columns) of C that are not stored.
  const u32x4 a_buf = buffer_of(A + (size_t)m0 * lda, rows_bytes(p.M - m0, p.K, lda));
  const u32x4 b_buf = TRANS_B ? buffer_of(B + (size_t)n0 * ldb, rows_bytes(p.N - n0, p.K, ldb)) : buffer_of(B, rows_bytes(kb, p.N, ldb));
  unsigned a_lane[A_INSTR], b_lane[B_INSTR];   // byte offset inside the buffer at k = 0
  int a_k8[A_INSTR], b_k8[B_INSTR];            // K-contiguous: first k of the chunk inside a tile; else k row inside a tile
#pragma unroll
  for (int q = 0; q < A_INSTR; ++q) {
    const DirectChunk c = row_chunk<64>(wave * A_INSTR + q, lane, p.M - m0, lda);
    a_lane[q] = c.offset;
    a_k8[q] = c.k;
  }
#pragma unroll
  for (int q = 0; q < B_INSTR; ++q) {
    DirectChunk c;
    if constexpr (TRANS_B) c = row_chunk<KP>(wave * B_INSTR + q, lane, p.N - n0, ldb);
    else c = column_chunk<BN>(wave * B_INSTR + q, lane, n0, ldb);
    b_lane[q] = c.offset;
    b_k8[q] = c.k;
  }
  const int P = (p.K + KP - 1) / KP;   // phases
  const int TA = (p.K + 63) / 64;      // A tiles
  const unsigned a_step = 64u * 2u, b_step = (TRANS_B ? (unsigned)KP : (unsigned)KP * ldb) * 2u;   // bytes per tile

  // part h (of HALVES; of an odd number of instructions the second has one more) of A tile t into stage `base`; past the end: the last tile again, into a
  // stage nobody reads.  (A chunk past a row's end is the next row's, or nothing: zero_tail.)
  auto issue_a = [&](int t, unsigned base, auto half) {
    constexpr int h = decltype(half)::value;
    const unsigned at = (unsigned)min(t, TA - 1) * a_step;
#pragma unroll
    for (int q = h * (A_INSTR / HALVES); q < (h == HALVES - 1 ? A_INSTR : A_INSTR / HALVES); ++q)
      lds_dma16(a_buf, a_lane[q], at, __builtin_amdgcn_readfirstlane(lds0 + base + (wave * A_INSTR + q) * 1024));
  };
  auto issue_b = [&](int t, unsigned stage) {
    const unsigned at = (unsigned)min(t, P - 1) * b_step, base = B_BASE + stage;
#pragma unroll
    for (int q = 0; q < B_INSTR; ++q) lds_dma16(b_buf, b_lane[q], at, __builtin_amdgcn_readfirstlane(lds0 + base + (wave * B_INSTR + q) * 1024));
  };
  // entries at k >= K must be zero: what was loaded there is other data.  Phase ph is the last one.
  auto zero_tail = [&](int ph) {
    const u32x4 zero = {0u, 0u, 0u, 0u};
    const int ta = ph / HALVES;
    unsigned char* sa = smem + (ta % SA) * A_STAGE;
#pragma unroll
    for (int q = 0; q < A_INSTR; ++q)
      if (ta * 64 + a_k8[q] >= p.K) *reinterpret_cast<u32x4*>(sa + ((wave * A_INSTR + q) * 64 + lane) * 16) = zero;
    unsigned char* sb = smem + B_BASE + (ph % SB) * B_STAGE;
#pragma unroll
    for (int q = 0; q < B_INSTR; ++q)
      if (ph * KP + b_k8[q] >= p.K) *reinterpret_cast<u32x4*>(sb + ((wave * B_INSTR + q) * 64 + lane) * 16) = zero;
  };

  Acc16<WM, WN> acc;
  acc.clear();

  // ---- operand read addresses inside a stage (bytes): a fragment is 16 rows (columns) x 32 k, lane l has row l % 16 and
  // the 8 k of chunk l / 16
  const int frow = lane & 15, fch = lane >> 4;
  int a_off[2];   // the two halves of an A tile
#pragma unroll
  for (int h = 0; h < 2; ++h) a_off[h] = (wm * WM * 32 + frow) * 128 + (((h * 4 + fch) ^ (frow >> 1)) * 16);
  int b_off[TRANS_B ? SUB : 2 * WN];
  if constexpr (TRANS_B) {
#pragma unroll
    for (int s = 0; s < SUB; ++s)
      b_off[s] = B_BASE + (wn * WN * 32 + frow) * (KP * 2) + (((s * 4 + fch) ^ (KP == 32 ? frow >> 2 : frow >> 1)) * 16);
  } else {
#pragma unroll
    for (int j = 0; j < 2 * WN; ++j) b_off[j] = B_BASE + kn16_fragment_offset<BN>(lane, wn * 2 * WN + j);
  }

  u32x4 fa[SUB][2 * WM], fb[SUB][2 * WN];  // the operand fragments of one phase
  const std::integral_constant<int, 0> even;
  const std::integral_constant<int, HALVES - 1> odd;
  // parity = ph % HALVES at compile time: which part of the A tile.  a_rd, a_wr: the stages of A tiles ph / HALVES and two
  // further; b_rd, b_wr: of B tiles ph and SB - 1 further (the stage before, going round)
  unsigned a_rd = 0, a_wr = 2 * A_STAGE, b_rd = 0, b_wr = (SB - 1) * B_STAGE;
  auto mem_phase = [&](int ph, auto parity) {
    constexpr int h = decltype(parity)::value;
    const unsigned char* sa = smem + a_rd;
    const unsigned char* sb = smem + b_rd;
#pragma unroll
    for (int s = 0; s < SUB; ++s) {
#pragma unroll
      for (int i = 0; i < 2 * WM; ++i) fa[s][i] = *reinterpret_cast<const u32x4*>(sa + a_off[h + s] + i * 16 * 128);
#pragma unroll
      for (int j = 0; j < 2 * WN; ++j) {
        if constexpr (TRANS_B) fb[s][j] = *reinterpret_cast<const u32x4*>(sb + b_off[s] + j * 16 * (KP * 2));
        else fb[s][j] = kn_fragment<BN * 2>(sb + b_off[j] + s * 32 * (BN * 2));
      }
    }
    issue_a(ph / HALVES + 2, a_wr, parity);
    issue_b(ph + SB - 1, b_wr);
    b_wr = b_rd;
    b_rd = b_rd == (SB - 1) * B_STAGE ? 0 : b_rd + B_STAGE;
    if constexpr (h == HALVES - 1) {
      a_wr = a_rd;
      a_rd = a_rd == 2 * A_STAGE ? 0 : a_rd + A_STAGE;
    }
  };
  auto compute_phase = [&]() {
#pragma unroll
    for (int s = 0; s < SUB; ++s)
#pragma unroll
      for (int i = 0; i < 2 * WM; ++i)
#pragma unroll
        for (int j = 0; j < 2 * WN; ++j) acc.v[i][j] = mfma_16x16x32<BF16>(fb[s][j], fa[s][i], acc.v[i][j]);
  };
  // at the end of phase ph: my loads of what phase ph + 1 reads have landed
  const bool tail = (p.K % KP) != 0;
  auto landed = [&](int ph) {
    wait_vmcnt<FLY>();
    if (tail && ph + 2 == P) zero_tail(ph + 1);
  };
  auto interval_end = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
  };

  // prologue = the loads that the phases before phase 0 would have issued
  if constexpr (KP == 32) {
    issue_a(0, 0, even);
    issue_a(0, 0, odd); issue_b(0, 0);
    issue_a(1, A_STAGE, even); issue_b(1, B_STAGE);
    issue_a(1, A_STAGE, odd); issue_b(2, 2 * B_STAGE);
  } else {
    issue_a(0, 0, even); issue_b(0, 0);
    issue_a(1, A_STAGE, even); issue_b(1, B_STAGE);
  }
  wait_vmcnt<FLY>();  // what phase 0 reads has landed
  if (tail && P == 1) zero_tail(0);
  __syncthreads();

  // (loops over pairs of phases with one exit each, the odd last phase after them: a loop with a second exit in its
  // middle makes the compiler keep two copies of the accumulators)
  int ph = 0;
  if (group == 0) {
    mem_phase(0, even);
    interval_end();
    for (; ph + 2 <= P; ph += 2) {
      compute_phase();
      landed(ph);
      interval_end();
      mem_phase(ph + 1, odd);
      interval_end();
      compute_phase();
      landed(ph + 1);
      interval_end();
      mem_phase(ph + 2, even);   // (past the last phase: read, never used)
      interval_end();
    }
    if (ph < P) {
      compute_phase();
      landed(ph);
      interval_end();
      mem_phase(ph + 1, odd);
      interval_end();
    }
  } else {
    interval_end();
    for (; ph + 2 <= P; ph += 2) {
      mem_phase(ph, even);
      landed(ph);
      interval_end();
      compute_phase();
      interval_end();
      mem_phase(ph + 1, odd);
      landed(ph + 1);
      interval_end();
      compute_phase();
      interval_end();
    }
    if (ph < P) {
      mem_phase(ph, even);
      landed(ph);
      interval_end();
      compute_phase();
      interval_end();
    }
  }
  wait_vmcnt<0>();  // the re-fetched last tiles: nothing may still be writing LDS when the stages are reused

  static_assert(WAVES * gemm_store_lds_bytes<WN>() <= SA * A_STAGE, "the epilogue fits the stages");
  __syncthreads();  // everybody has read its last fragments and nobody's loads are in flight
  const u16* aux = p.aux ? static_cast<const u16*>(p.aux) + (size_t)z * p.stride_c : nullptr;
  gemm_store_tile<BF16, WM, WN>(p, acc, C, aux, m0, n0, wm, wn, lane, smem + wave * gemm_store_lds_bytes<WN>(), p.stream_out != 0);
}

}  // namespace iex
