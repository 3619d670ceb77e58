// CSR SpMM in fp32 on the matrix cores (gfx950, v_mfma_f32_32x32x2_f32 or 16x16x4_f32).  The
// sparse operand is expanded to dense MT x 128 blocks in LDS (MT = 32 or 16 rows, the MFMA
// tile height) and multiplied at the dense fp32 MFMA rate (64 FMA-flops per clock and SIMD),
// which beats the gather kernels from roughly 25 % density up: those move n * 4 bytes from L2
// per nonzero.  (The text below says 32 rows and 8 k rows per group; with MT = 16 read 16 rows
// and 16 k rows per group: a wave then has four k slots of 16 lanes instead of two of 32.)
//
// Workgroup = 4 multiplying wavefronts, C tile = MT rows (CSR rows in swizzled order) x BN columns.
//   A   chunks of 128 columns, double-buffered [32][132] floats in LDS.  A wavefront expands 8 rows, a
//       lane a nonzero: the next 64 of every row are in registers (128 where rows are that dense), so those loads land
//       during the MFMAs of a chunk.  One barrier per chunk.
//   B   (k x n row-major) never touches LDS: with a 32-row tile every element of B feeds
//       exactly one MFMA of the workgroup, and the MFMA operand layout (lane = column, half
//       wave = k) is a coalesced global load already.  A lane loads NJ adjacent columns
//       (NJ*4 bytes) of one k row; element j feeds MFMA j, whose 32 "columns" are therefore
//       the strided set {NJ*i + j}.  At the end a lane holds NJ adjacent columns per
//       accumulator slot and stores them with one NJ*4-byte store.
//   k   a wave covers 32 x 32*NJ columns; the BN / (32*NJ) waves along n times WAVES_K waves
//       along k make up the workgroup.  The k slices interleave by groups of 8 k rows (one
//       128-bit LDS read of A per lane and group: lanes 0-31 take k .. k+3, lanes 32-63
//       k+4 .. k+7, the B loads follow the same assignment); partial tiles are added through
//       LDS at the end in a fixed order (deterministic).
// Loads of B run four groups (4 x 4 loads per lane) ahead of the MFMAs, by buffer address: their positions are scalar.
// SPLIT: the workgroup has 8 wavefronts with two roles, each with a loop of its own.  Waves 0-3 only multiply, waves 4-7
// only expand the next chunk; one of each shares a SIMD.  Without SPLIT all 4 waves do both, one after the other.
// What bounds it: the MFMAs, which hold the SIMD's vector ALU for 64 clocks each and slip into every gap between two vector
// instructions of the expanding wavefront.  That wavefront's vector instructions were the longer chain (up to 160 per
// chunk of 64 MFMAs, eight lanes to a row and windows of 8 nonzeros): with a lane per nonzero, the rows' instructions side by
// side, positions and masks in scalar registers, they are 16 - 40.  MI355X, us before -> now: 4096 x 4096, n = 256, rows of
// geometric lengths, 20 % and 30 % density 128 -> 112, rows of one length, 2 / 10 / 30 / 50 / 100 % 86 / 91 / 104 / 116 / 130 -> 90 / 91 /
// 92 / 109 / 112; n = 128 (16 rows), geometric 92 -> 74, equal 30 % 68 -> 56; 11008 x 4096, n = 1024, 30 % 1051 -> 1023.  (Expanding wavefronts
// at raised priority: 2 us more.)
// FAR: the dense operand or the nonzeros pass the 4 GiB that a buffer's offsets reach; they are read by 64-bit addresses then (1024 x 1024 at
// 50 %, n = 2^20: 32 ms, the row kernel 68).
// Requirements (checked by the host): n % 4 == 0, 16-byte aligned dense operand and output,
// strictly ascending column indices inside a row; without FAR (k + 1024) n and nnz below 2^30.
#pragma once
#include "spmm_device.cuh"

namespace iex {

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// columns of A per chunk: at most 128 nonzeros of a row fall into one, which two windows of 64 hold
template <int MT>
constexpr int spmm_mfma_f32_bka() { return 128; }
constexpr int kF32Threads = 256;       // per role

template <int MT, int NJ, int WAVES_N>
constexpr int spmm_mfma_f32_lds_bytes() {
  constexpr int a_bytes = 2 * MT * (spmm_mfma_f32_bka<MT>() + 4) * 4;
  constexpr int red_bytes = (4 / WAVES_N - 1) * WAVES_N * NJ * (MT * MT / 64) * 64 * 4;  // partial tiles of the k slices
  return a_bytes > red_bytes ? a_bytes : red_bytes;
}

template <int NJ>
struct F32Frag {
  float v[NJ];
};

template <int MT, int NJ, int WAVES_N, bool SPLIT, bool FAR>
__device__ __forceinline__ void spmm_mfma_f32_block(const SpmmParams& p, int tile_m, int tile_n, int z, unsigned char* smem) {
  constexpr int BM = MT, BKA = spmm_mfma_f32_bka<MT>();
  constexpr int LDA = BKA + 4;            // floats: 16 consecutive rows start in distinct 4-bank groups
  constexpr int KSLOTS = 64 / MT;         // k rows one MFMA consumes = lane groups of MT lanes (2 or 4)
  constexpr int GK = 4 * KSLOTS;          // k rows of a group (one 128-bit A read per lane = 4 MFMA steps)
  constexpr int ACC = MT * MT / 64;       // accumulator registers of one MFMA tile (16 or 4)
  constexpr int WAVES_K = 4 / WAVES_N;
  constexpr int WCOLS = MT * NJ;          // columns of a wave
  constexpr int BN = WCOLS * WAVES_N;     // columns of the workgroup
  constexpr int GROUPS = BKA / GK;        // groups per chunk (16 or 8)
  constexpr int GPW = GROUPS / WAVES_K;   // groups per wave and chunk
  constexpr int EXP_ROWS = 8;                       // rows an expanding wavefront owns
  constexpr int EXP_THREADS = MT / EXP_ROWS * 64;   // threads that expand (256 or 128)
  typedef float acc_t __attribute__((ext_vector_type(ACC)));
  static_assert(MT == 32 || MT == 16, "MFMA tile height");
  constexpr int AHEAD = GPW < 4 ? GPW : 4;  // groups of B loads in flight
  static_assert(NJ == 2 || NJ == 4, "a lane loads 2 or 4 adjacent columns");
  static_assert(GPW % AHEAD == 0, "the prefetch ring is unrolled over the groups of a chunk");

  float* sA = reinterpret_cast<float*>(smem);  // [2][BM][LDA]

  const int lane = threadIdx.x & 63;
  const int wave_id = uniform(threadIdx.x >> 6);
  const bool is_mma = wave_id < kF32Threads / 64;                                   // wave-uniform roles
  const bool is_exp = SPLIT ? !is_mma : wave_id < EXP_THREADS / 64;
  const int wave = wave_id % (kF32Threads / 64);
  const int wn = wave % WAVES_N, wk = wave / WAVES_N;
  const int half = lane / MT;  // k slot: which 4 of the GK k rows of a group this lane feeds
  const int l32 = lane % MT;   // row (A fragment) / column slot (B fragment) of this lane
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const float* values = static_cast<const float*>(p.values) + (p.per_batch_values ? (size_t)z * p.nnz : (size_t)0);
  const float* B = static_cast<const float*>(p.dense) + (size_t)z * p.k * p.n;
  float* __restrict__ C = static_cast<float*>(p.out) + (size_t)z * p.m * p.n;
  // Raw buffers: what lies past their end reads as zero, and the position inside costs no vector instruction.
  auto buffer = [](const void* at, size_t bytes) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(at), 0, (int)(unsigned)bytes, 4 << 15); };
  const auto vals_buf = buffer(values, (size_t)p.nnz * 4), cols_buf = buffer(p.cols, (size_t)p.nnz * 4), b_buf = buffer(B, (size_t)p.k * p.n * 4);

  // ---- expansion: wavefront w owns local rows 8 w .. 8 w + 7, a lane a nonzero.  The next 64 nonzeros of every row are in
  // registers (128 where a row of the wavefront has more than 40 in a chunk on average); a chunk takes 128 at most.
  int pos[EXP_ROWS], end[EXP_ROWS], c0[EXP_ROWS], c1[EXP_ROWS];
  float v0[EXP_ROWS], v1[EXP_ROWS];
  bool wide = false;
  // (scalar offsets never pass a buffer's end: only up to there does the range check hold)
  auto load_window = [&](int first, int skip, int& c, float& v) {
    if constexpr (FAR) {
      const int at = min(lane + skip, p.nnz - 1 - first);   // (-1 behind the last nonzero)
      c = (static_cast<const int*>(p.cols) + first)[at];
      v = (values + first)[at];
      return;
    }
    c = __builtin_amdgcn_raw_buffer_load_b32(cols_buf, (lane + skip) * 4, (unsigned)first * 4u, 0);
    v = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(vals_buf, (lane + skip) * 4, (unsigned)first * 4u, 0));
  };
  auto load_windows = [&]() {
#pragma unroll
    for (int r = 0; r < EXP_ROWS; ++r) load_window(pos[r], 0, c0[r], v0[r]);
    if (wide) {
#pragma unroll
      for (int r = 0; r < EXP_ROWS; ++r) load_window(pos[r], 64, c1[r], v1[r]);
    }
  };
  if (is_exp) {
#pragma unroll
    for (int r = 0; r < EXP_ROWS; ++r) {
      const int slot = m0 + wave * EXP_ROWS + r;
      pos[r] = end[r] = 0;
      c1[r] = 0, v1[r] = 0.f;
      if (slot < p.m) {
        const int row = uniform(p.row_indices[slot]);
        pos[r] = uniform(p.row_offsets[row]);
        end[r] = uniform(p.row_offsets[row + 1]);
      }
      wide = wide || (long long)(end[r] - pos[r]) * BKA > (long long)p.k * 40;
    }
    load_windows();
  }
  // Columns [ka0, ka0 + BKA) of the wavefront's rows -> abuf.  Zeros and nonzeros come from the same wavefront, and LDS keeps
  // the order of a wavefront's accesses.  An MFMA holds the vector ALU for 64 clocks and slips into every gap between two
  // vector instructions of this wavefront: so few of them, the rows' side by side, all else in scalar registers.
  auto first_of = [](int left) { return left >= 64 ? ~0ull : left > 0 ? (1ull << left) - 1 : 0ull; };
  auto expand = [&](int ka0, float* abuf) {
    float* mine = abuf + wave * EXP_ROWS * LDA;
    constexpr int QUADS = EXP_ROWS * LDA / 4;
#pragma unroll
    for (int q = 0; q < (QUADS + 63) / 64; ++q)
      if (q * 64 + 63 < QUADS || q * 64 + lane < QUADS) reinterpret_cast<f32x4_t*>(mine)[q * 64 + lane] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int kend = ka0 + BKA;
    unsigned long long in[EXP_ROWS];
    bool more = false;
#pragma unroll
    for (int r = 0; r < EXP_ROWS; ++r) {
      in[r] = __ballot(c0[r] < kend) & first_of(end[r] - pos[r]);
      more = more || in[r] == ~0ull;
    }
#pragma unroll
    for (int r = 0; r < EXP_ROWS; ++r)
      if (__builtin_amdgcn_inverse_ballot_w64(in[r])) mine[r * LDA + (c0[r] - ka0)] = v0[r];
#pragma unroll
    for (int r = 0; r < EXP_ROWS; ++r) pos[r] += __popcll(in[r]);
    if (more) {   // (uniform) the second half of a chunk with 64 and more
      if (!wide) {
#pragma unroll
        for (int r = 0; r < EXP_ROWS; ++r) load_window(pos[r], 0, c1[r], v1[r]);   // (of the others: what follows, none of it in the chunk)
      }
#pragma unroll
      for (int r = 0; r < EXP_ROWS; ++r) in[r] = in[r] == ~0ull ? __ballot(c1[r] < kend) & first_of(end[r] - pos[r]) : 0ull;
#pragma unroll
      for (int r = 0; r < EXP_ROWS; ++r)
        if (__builtin_amdgcn_inverse_ballot_w64(in[r])) mine[r * LDA + (c1[r] - ka0)] = v1[r];
#pragma unroll
      for (int r = 0; r < EXP_ROWS; ++r) pos[r] += __popcll(in[r]);
    }
    load_windows();
  };

  // ---- B: the 4 k rows of group g (chunk-relative) that this lane feeds ----------------------
  // A k row beyond the matrix reads as zeros and meets zeros of A; a column beyond n is computed and never stored.
  const int col = n0 + wn * WCOLS + l32 * NJ;  // first of the NJ columns of this lane
  unsigned b_lane[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) b_lane[i] = (unsigned)((half * 4 + i) * p.n + (col < p.n ? col : 0)) * 4u;   // n % 4 == 0: the NJ columns are in or out together
  auto load_b = [&](F32Frag<NJ> (&f)[4], int kbase) {  // kbase = first k row of the group
    if constexpr (FAR) {   // (past the matrix: its last row)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        typedef float vec __attribute__((ext_vector_type(NJ)));
        const vec v = *reinterpret_cast<const vec*>(B + (size_t)min(kbase + half * 4 + i, p.k - 1) * p.n + (col < p.n ? col : 0));
#pragma unroll
        for (int j = 0; j < NJ; ++j) f[i].v[j] = v[j];
      }
      return;
    }
    const unsigned at = (unsigned)min(kbase, p.k) * (unsigned)p.n * 4u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (NJ == 4) {
        typedef int i32x4_t __attribute__((ext_vector_type(4)));
        const i32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(b_buf, b_lane[i], at, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) f[i].v[j] = __int_as_float(v[j]);
      } else {
        typedef int i32x2_t __attribute__((ext_vector_type(2)));
        const i32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(b_buf, b_lane[i], at, 0);
        f[i].v[0] = __int_as_float(v[0]);
        f[i].v[1] = __int_as_float(v[1]);
      }
    }
  };

  // group index of this wave, global over chunks: gi -> k row (gi / GPW) * BKA + ((gi % GPW) * WAVES_K + wk) * 8
  auto group_k = [&](int gi) { return (gi / GPW) * BKA + ((gi % GPW) * WAVES_K + wk) * GK; };
  const int n_chunks = (p.k + BKA - 1) / BKA;
  auto buffer_of_chunk = [&](int c) { return sA + (c & 1) * BM * LDA; };

  if (SPLIT && is_exp) {   // (a loop of its own: neither role's registers are live in the other's)
    expand(0, sA);
    __syncthreads();
    for (int c = 0; c < n_chunks; ++c) {
      if (c + 1 < n_chunks) expand((c + 1) * BKA, buffer_of_chunk(c + 1));
      __syncthreads();
    }
    __syncthreads();
    if constexpr (WAVES_K > 1) __syncthreads();   // (the partial tiles)
    return;
  }

  acc_t acc[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int r = 0; r < ACC; ++r) acc[j][r] = 0.f;
  F32Frag<NJ> ring[AHEAD][4];
#pragma unroll
  for (int a = 0; a < AHEAD; ++a) load_b(ring[a], group_k(a));
  if (!SPLIT && is_exp) expand(0, sA);
  __syncthreads();

  // The scheduling barriers pin the order "MFMAs of group g, then the loads that refill its
  // ring slot": left alone, the compiler sinks all loads of a chunk behind its last MFMA and
  // the next chunk starts by waiting for them.  A's fragment of a group is read a group ahead, that of the next chunk's first
  // group behind the barrier, which stands before the last group of a chunk: everything of the chunk is in registers there.
  const float* a_lane = sA + l32 * LDA + half * 4 + wk * GK;
  f32x4_t fa = *reinterpret_cast<const f32x4_t*>(a_lane);
  for (int c = 0; c < n_chunks; ++c) {
    if (!SPLIT && is_exp && c + 1 < n_chunks) expand((c + 1) * BKA, buffer_of_chunk(c + 1));
    __builtin_amdgcn_sched_barrier(0);
    const float* a = a_lane + (c & 1) * BM * LDA;
    const float* a_next = a_lane + ((c + 1) & 1) * BM * LDA;
#pragma unroll
    for (int g = 0; g < GPW; ++g) {
      f32x4_t next;
      if (g + 1 < GPW) {
        next = *reinterpret_cast<const f32x4_t*>(a + (g + 1) * WAVES_K * GK);
      } else {
        __syncthreads();
        next = *reinterpret_cast<const f32x4_t*>(a_next);   // (past the last chunk: read, never used)
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          if constexpr (MT == 32) acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(ring[g % AHEAD][i].v[j], fa[i], acc[j], 0, 0, 0);
          else acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ring[g % AHEAD][i].v[j], fa[i], acc[j], 0, 0, 0);
        }
      __builtin_amdgcn_sched_barrier(0);
      load_b(ring[g % AHEAD], group_k(c * GPW + g + AHEAD));  // (past the end: zeros, unused)
      __builtin_amdgcn_sched_barrier(0);
      fa = next;
    }
  }
  __syncthreads();   // everybody is done with A's buffers

  if constexpr (WAVES_K > 1) {
    // partial tiles of the k slices -> LDS (the A buffers are free after the last barrier),
    // added by the wavefront of slice 0 in slice order
    constexpr int Q = ACC / 4;  // 128-bit pieces of an accumulator tile per lane
    f32x4_t* red = reinterpret_cast<f32x4_t*>(smem);  // [WAVES_K - 1][WAVES_N][NJ * Q][64]
    if (wk > 0) {
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int q = 0; q < Q; ++q)
          red[(((wk - 1) * WAVES_N + wn) * NJ * Q + j * Q + q) * 64 + lane] =
              f32x4_t{acc[j][q * 4], acc[j][q * 4 + 1], acc[j][q * 4 + 2], acc[j][q * 4 + 3]};
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll 1   // (unrolled, all the reads at once: more registers than there are)
    for (int s = 1; s < WAVES_K; ++s)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          const f32x4_t v = red[(((s - 1) * WAVES_N + wn) * NJ * Q + j * Q + q) * 64 + lane];
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[j][q * 4 + e] += v[e];
        }
  }

  // Swapped operands: lane holds row (lane % MT) of the tile; accumulator slot v of MFMA j is
  // column NJ * ((v / 4) * 4 * KSLOTS + (lane / MT) * 4 + v % 4) + j of the wave's column range.
  const int slot = m0 + l32;
  if (slot >= p.m) return;
  const int row = p.row_indices[slot];
  const float bias = p.bias ? p.bias[row] : 0.f;
#pragma unroll
  for (int v = 0; v < ACC; ++v) {
    const int gn = n0 + wn * WCOLS + NJ * ((v / 4) * 4 * KSLOTS + half * 4 + (v % 4));
    if (gn >= p.n) continue;
    float* dst = C + (size_t)row * p.n + gn;
    float x[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) x[j] = acc[j][v];
    if (p.accumulate) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) x[j] += dst[j];
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      x[j] += bias;
      if (p.relu) x[j] = fmaxf(x[j], 0.f);
    }
    if constexpr (NJ == 4) *reinterpret_cast<f32x4_t*>(dst) = f32x4_t{x[0], x[1], x[2], x[3]};
    else *reinterpret_cast<float2*>(dst) = make_float2(x[0], x[1]);
  }
}

}  // namespace iex
