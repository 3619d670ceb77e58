// CSR SpMM for 16-bit types on the matrix cores' structured-sparsity instructions (v_smfmac_f32_16x16x64): a sparse
// operand of which a row holds at most two of any four neighbouring columns costs half the multiplications of its dense
// form.  A weight of 2:4 structure is such an operand as it stands; an unstructured one of 90 % sparsity nearly is: of its
// groups of four, 0.4 % hold a third entry.  So the sparse operand is laid out in a workspace as
//   pairs    per row and group of four columns the first two entries and, two bits each, which columns they are;
//   spill    what is left, the third and fourth entries of a group, as a narrow dense operand: per block of rows the
//            columns that have such entries ("spilled" columns, ascending), 32 at a time.
// and the product walks the pairs (64 columns per phase, v_smfmac at twice the dense rate) and then the spilled columns (32
// columns per phase, plain MFMAs on the rows of B that a list names).  Any canonical CSR matrix can be laid out so: a
// group's spilled entries are at its third and fourth column, so a block has at most k / 2 spilled columns, which the
// workspace has room for.  How many phases the spill takes is what the choice of this path is about, not its correctness.
//
// Form.  Rows in panels of BM = 256, 192 or 128 (the tile height); a panel is a sequence of blocks, one per phase, that the
// product copies to LDS as they are: the operand fragments of 16 rows in the order in which the instruction wants them
// (lane l: row l % 16, columns 16 * (l / 16) .. + 15 as 8 entries; in a spill block 8 * (l / 16) .. + 7), 1 KB each, then the
// index bits, a 32-bit word per lane and pair of fragments.  Both halves of a panel have spill lists of their own: wavefronts of the
// two halves multiply different rows of B in a spill phase, and half as many rows spill into fewer columns (11008 x 4096 at 90 %:
// 10.5 phases of spill beside 64 for blocks of 128 rows, 19 % of the columns instead of 11 for 256).
#pragma once
#include "gemm_dma_device.cuh"
#include "spmm_dense_device.cuh"

namespace iex {

typedef unsigned int u32x8 __attribute__((ext_vector_type(8)));

constexpr int kTwoFourThreads = 1024;
constexpr int kTwoFourMaxK = 65536;     // (a block's bitmap of spilled columns, in LDS)

// Where the parts of a form lie.
struct TwoFourForm {
  int bm;              // rows per panel
  int panels, phases;  // phases of pairs: 64 columns each, an even number (zeros past k)
  int spill_phases;    // room for that many phases of spill
  int list_room;       // entries of a spill list
  int words;           // of a row of marks
  int block;           // bytes of a block
  size_t panel;        // bytes of a panel
  size_t counts_at, lists_at, ranks_at, bytes;
};
inline int two_four_block_bytes(int bm) { return bm == 192 ? 14 * 1024 : bm * 72; }   // (whole kilobytes per direct load for 192)
inline int two_four_spill_room(int k) { return ceil_div(2 * ceil_div(k, 4), 32); }   // phases: enough for any canonical CSR matrix
inline TwoFourForm two_four_form(int m, int k, int bm, int spill_room) {
  TwoFourForm f;
  f.bm = bm;
  f.panels = ceil_div(m, bm);
  f.phases = ceil_div(k, 128) * 2;
  f.spill_phases = spill_room;
  f.list_room = ceil_div(spill_room, 2) * 64;
  f.words = ceil_div(k, 32);
  f.block = two_four_block_bytes(bm);
  f.panel = (size_t)(f.phases + f.spill_phases) * f.block;
  f.counts_at = round256(f.panels * f.panel);
  f.lists_at = f.counts_at + round256((size_t)f.panels * 2 * sizeof(int));
  f.ranks_at = f.lists_at + round256((size_t)f.panels * 2 * f.list_room * sizeof(unsigned));
  f.bytes = f.ranks_at + round256((size_t)f.panels * 2 * f.words * sizeof(uint2));
  return f;
}

// ---------------------------------------------------------------------------------------------------- laying the form out
struct TwoFourSource {   // the CSR matrix
  int m, k;
  const int* row_offsets;
  const void* cols;
  const uint16_t* values;
};
struct TwoFourTarget {
  unsigned char* form;
  int* counts;        // per half panel: spilled columns
  unsigned* lists;    // ... which, ascending
  uint2* ranks;       // ... per 32 columns: the spilled ones' bits, how many there are before
  int bm, phases, spill_phases, list_room, words, block;
  size_t panel;
};

// Marks: per 32 rows a bit for every column that has spilled entries there.  An entry is spilled when the entry two before it in the row is of the
// same group.  One workgroup per 32 rows, two rows per wavefront, the loads of both in flight together.
template <typename IT>
__global__ __launch_bounds__(kTwoFourThreads) void two_four_marks_kernel(int m, int k, const int* __restrict__ row_offsets, const IT* __restrict__ cols,
                                                                         int words, unsigned* __restrict__ marks) {
  extern __shared__ __align__(16) unsigned bits[];   // [words]
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
  constexpr int R = 2, U = 8;
  static_assert(kTwoFourThreads / 64 * R == 32, "32 rows");
  int pos[R], end[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int row = blockIdx.x * 32 + wave * R + r;
    pos[r] = row < m ? uniform(row_offsets[row]) + 2 : 0;
    end[r] = row < m ? uniform(row_offsets[row + 1]) : 0;
  }
  for (int w = tid; w < words; w += kTwoFourThreads) bits[w] = 0u;
  __syncthreads();
  bool more = true;
  while (more) {
    more = false;
    int c[R][U], c2[R][U];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int j = max(min(pos[r] + u * 64 + lane, end[r] - 1), 2);   // (a row without such entries: never used; the host guarantees three entries)
        c[r][u] = (int)cols[j];
        c2[r][u] = (int)cols[j - 2];
      }
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (pos[r] + u * 64 + lane < end[r] && (c[r][u] >> 2) == (c2[r][u] >> 2) && (unsigned)c[r][u] < (unsigned)k) atomicOr(&bits[c[r][u] >> 5], 1u << (c[r][u] & 31));
      pos[r] += U * 64;
      more |= pos[r] < end[r];
    }
  }
  __syncthreads();
  for (int w = tid; w < words; w += kTwoFourThreads) marks[(size_t)blockIdx.x * words + w] = bits[w];
}

// phases[i] += phases of spill of all blocks of 64, 96, 128 rows (i = 0, 1, 2), phases[3 + i] = max of any of them.  Workgroup = block of 64, then of
// 96, then of 128 rows.
static __global__ __launch_bounds__(256) void two_four_measure_kernel(int m, int words, const unsigned* __restrict__ marks, int* __restrict__ phases) {
  const int n64 = (m + 63) / 64, n96 = (m + 95) / 96, rows32 = (m + 31) / 32;
  int b = blockIdx.x, which = 0;
  if (b >= n64) b -= n64, which = 1;
  if (which == 1 && b >= n96) b -= n96, which = 2;
  const int per = 2 + which;
  int count = 0;
  for (int w = threadIdx.x; w < words; w += 256) {
    unsigned all = 0;
    for (int f = 0; f < per; ++f)
      if (b * per + f < rows32) all |= marks[(size_t)(b * per + f) * words + w];
    count += __popc(all);
  }
  __shared__ int part[4];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) count += __shfl_xor(count, o);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = count;
  __syncthreads();
  if (threadIdx.x == 0) {
    const int mine = (part[0] + part[1] + part[2] + part[3] + 31) / 32;
    atomicAdd(&phases[which], mine);
    atomicMax(&phases[3 + which], mine);
  }
}

// Which columns of a half panel are spilled: the marks of its rows together, a rank for each, the list.  One workgroup per half panel.
static __global__ __launch_bounds__(256) void two_four_rank_kernel(TwoFourTarget t, const unsigned* __restrict__ marks, int marked) {
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), half_panel = blockIdx.x;
  __shared__ int total[4];
  const int f0 = half_panel * (t.bm / 64), f1 = min(f0 + t.bm / 64, marked);
  int before = 0;
  for (int w0 = 0; w0 < t.words; w0 += 256) {
    const int w = w0 + tid;
    unsigned all = 0;
    if (w < t.words)
      for (int f = f0; f < f1; ++f) all |= marks[(size_t)f * t.words + w];
    const int mine = __popc(all);
    int upto = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int x = __shfl_up(upto, o);
      if (lane >= o) upto += x;
    }
    if (lane == 63) total[wave] = upto;
    __syncthreads();
    int at = before + upto - mine;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      if (v < wave) at += total[v];
      before += total[v];
    }
    __syncthreads();
    if (w < t.words) t.ranks[(size_t)half_panel * t.words + w] = uint2{all, (unsigned)at};
    for (; all; all &= all - 1, ++at)
      if (at < t.list_room) t.lists[(size_t)half_panel * t.list_room + at] = w * 32 + __ffs(all) - 1;
  }
  if (tid == 0) t.counts[half_panel] = min(before, t.list_room);   // (canonical CSR: it is never more)
}

// The form of `rows` rows (a power of two, 8 at most), a wavefront or several per row.  Where an entry goes follows from its neighbours in the
// row alone: it is the first or the second of its group of four, or spilled.  So wavefronts take 61 entries at a time, with two
// before and one after them, in any order; the rows are put together in LDS and copied out.
//   index bits of a group: both columns of its two entries; of a group with one, it and a column without an entry, ascending.
constexpr int kTwoFourRowThreads = 512;
inline int two_four_rows(int k) {   // rows per workgroup: about 36 KB of LDS, four workgroups on a CU
  int rows = 8;
  while (rows > 1 && rows * k > 32768) rows /= 2;
  return rows;
}
inline int two_four_rows_lds_bytes(int rows, int phases) { return rows * (phases * 64 + 16) + rows * (phases * 8 + 4); }

template <typename IT>
__global__ __launch_bounds__(kTwoFourRowThreads) void two_four_form_kernel(TwoFourSource s, TwoFourTarget t, int rows) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int WAVES = kTwoFourRowThreads / 64, U = 4, STEP = 61;
  const int value_row = t.phases * 64 + 16, index_row = t.phases * 8 + 4;   // bytes; padded against bank conflicts
  unsigned char* value_rows = smem;
  unsigned char* index_rows = smem + rows * value_row;
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
  const int per_row = WAVES / rows, my_row = wave / per_row, row = blockIdx.x * rows + my_row;
  const int first = row < s.m ? uniform(s.row_offsets[row]) : 0, entries = (row < s.m ? uniform(s.row_offsets[row + 1]) : 0) - first;
  const int half_rows = t.bm / 2, half_panel = blockIdx.x * rows / half_rows;
  const int count = t.counts[half_panel];
  const int share = ((entries + per_row - 1) / per_row + STEP - 1) / STEP * STEP;
  int pos = min(wave % per_row * share, entries);   // (from the row's first entry)
  const int end = min(pos + share, entries);

  const IT* __restrict__ cols = static_cast<const IT*>(s.cols) + first;
  const uint16_t* __restrict__ values = s.values + first;
  int c[U];
  uint16_t v[U];
  auto load = [&]() {   // entries pos - 2 .. + 61 of every step
    if (entries <= 0) return;   // (uniform)
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const unsigned j = (unsigned)max(min(pos + u * STEP - 2 + lane, entries - 1), 0);
      c[u] = (int)*reinterpret_cast<const IT*>(reinterpret_cast<const char*>(cols) + j * (unsigned)sizeof(IT));
      v[u] = *reinterpret_cast<const uint16_t*>(reinterpret_cast<const char*>(values) + j * 2u);
    }
  };
  load();
  for (int i = tid * 16; i < rows * value_row; i += kTwoFourRowThreads * 16) *reinterpret_cast<u32x4*>(value_rows + i) = u32x4{0u, 0u, 0u, 0u};
  for (int i = tid * 4; i < rows * index_row; i += kTwoFourRowThreads * 4) *reinterpret_cast<unsigned*>(index_rows + i) = 0x44444444u;   // (no entry: columns 0 and 1)
  // where this workgroup's rows are in a block: lane l of their fragment has row l % 16 and columns 16 * (l / 16) ..
  unsigned char* panel = t.form + (half_panel >> 1) * t.panel;
  const int fragment = blockIdx.x * rows % t.bm / 16, row0 = blockIdx.x * rows % 16;
  unsigned char* spill_at = panel + (size_t)t.phases * t.block + fragment * 1024;
  const int spills = min((min(count, t.list_room) + 31) / 32, t.spill_phases);
  for (int i = tid; i < spills * 4 * rows; i += kTwoFourRowThreads)
    *reinterpret_cast<u32x4*>(spill_at + (size_t)(i / (4 * rows)) * t.block + (row0 + i % rows + i / rows % 4 * 16) * 16) = u32x4{0u, 0u, 0u, 0u};
  if (spills) wait_vmcnt<0>();   // the zeros are in L2 before another wavefront's entries
  __syncthreads();

  // ---- the entries to their places
  unsigned char* const my_values = value_rows + my_row * value_row;
  unsigned char* const my_index = index_rows + my_row * index_row;
  const uint2* const ranks = t.ranks + (size_t)half_panel * t.words;
  while (pos < end) {
    int c1[U];
    uint16_t v1[U];
#pragma unroll
    for (int u = 0; u < U; ++u) c1[u] = c[u], v1[u] = v[u];
    const int from = pos - 2 + lane;
    pos += U * STEP;
    if (pos < end) load();   // (the next ones are on the way meanwhile)
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = from + u * STEP;
      const int column = (unsigned)j < (unsigned)entries ? c1[u] : -8 * (lane + 1);   // (outside the row: a group of its own)
      const int group = column >> 2;
      const int g1 = __builtin_amdgcn_update_dpp(0, group, 0x138, 0xf, 0xf, false);          // lane - 1
      const int g2 = __builtin_amdgcn_update_dpp(0, g1, 0x138, 0xf, 0xf, false);             // lane - 2
      const int next = __builtin_amdgcn_update_dpp(0, column, 0x130, 0xf, 0xf, false);       // lane + 1
      if (lane >= 2 && lane <= 62 && j < end && (unsigned)column < (unsigned)s.k) {
        const int p = column & 3;
        const bool opens = g1 != group, alone = opens && (next >> 2) != group;
        if (opens || g2 != group) *reinterpret_cast<uint16_t*>(my_values + group * 4 + (!opens || (alone && p == 3) ? 2 : 0)) = v1[u];
        if (opens) {
          const unsigned two = alone ? p | 0xcu : p | (next & 3) << 2;
          atomicXor(reinterpret_cast<unsigned*>(my_index + (group >> 3) * 4), ((alone && p == 3 ? 0xcu : two) ^ 4u) << (group & 7) * 4);
        }
        if (!opens && g2 == group) {
          const uint2 rank = ranks[column >> 5];
          const unsigned bit = column & 31;
          const int e = (int)rank.y + __popc(rank.x & ((1u << bit) - 1u));
          if ((rank.x >> bit & 1u) && e / 32 < spills)
            *reinterpret_cast<uint16_t*>(spill_at + (size_t)(e / 32) * t.block + (row0 + my_row + e % 32 / 8 * 16) * 16 + e % 8 * 2) = v1[u];
        }
      }
    }
  }
  __syncthreads();
  for (int i = tid; i < t.phases * 4 * rows; i += kTwoFourRowThreads) {
    const int r = i % rows, quarter = i / rows % 4, ph = i / (4 * rows), slot = row0 + r + quarter * 16;
    unsigned char* block = panel + (size_t)ph * t.block;
    *reinterpret_cast<u32x4*>(block + fragment * 1024 + slot * 16) = *reinterpret_cast<const u32x4*>(value_rows + r * value_row + ph * 64 + quarter * 16);
    *reinterpret_cast<uint16_t*>(block + t.bm * 64 + (fragment >> 1) * 256 + slot * 4 + (fragment & 1) * 2) =
        *reinterpret_cast<const uint16_t*>(index_rows + r * index_row + ph * 8 + quarter * 2);
  }
}

// ---------------------------------------------------------------------------------------------------- the product
template <bool BF16, int HIGH>
__device__ __forceinline__ f32x4 smfmac_16x16x64(u32x4 a, u32x8 b, f32x4 c, unsigned index) {
  typedef _Float16 f16x16 __attribute__((ext_vector_type(16)));
  typedef __bf16 bf16x16 __attribute__((ext_vector_type(16)));
  if constexpr (BF16) return __builtin_amdgcn_smfmac_f32_16x16x64_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x16, b), c, (int)index, 0, HIGH);
  else return __builtin_amdgcn_smfmac_f32_16x16x64_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x16, b), c, (int)index, 0, HIGH);
}

// 4 bytes per lane, lane i's at M0 + 4 * i (cf. lds_dma16)
__device__ __forceinline__ void lds_dma4(u32x4 rsrc, unsigned lane_offset, unsigned uniform_offset, unsigned lds_base_uniform) {
  asm volatile("s_mov_b32 m0, %3\n\tbuffer_load_dword %0, %1, %2 offen lds" ::"v"(lane_offset), "s"(rsrc), "s"(uniform_offset), "s"(lds_base_uniform) : "memory", "m0");
}

// Sums of a wavefront whose MFMAs have the sparse operand first: a lane holds rows 4 * (lane / 16) .. + 3 of one column.  Handed out as
// quads of 4 adjacent columns of one row (Acc16's contract) by exchanging 4 x 4 blocks between the lanes of a quad.
template <int WM, int WN>
struct AccRows {
  f32x4 v[2 * WM][2 * WN];
  template <int CTRL>
  static __device__ __forceinline__ float from_lane(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
  }
  __device__ __forceinline__ f32x4 quad(int i, int t) const {
    const f32x4 x = v[2 * i + t / (2 * WN)][t % (2 * WN)];
    const bool odd = threadIdx.x & 1, upper = threadIdx.x & 2;
    // 2 x 2 blocks with the neighbour, then with the lane two further
    const float p0 = from_lane<0xb1>(odd ? x[0] : x[1]), p1 = from_lane<0xb1>(odd ? x[2] : x[3]);
    const float a0 = odd ? p0 : x[0], a1 = odd ? x[1] : p0, b0 = odd ? p1 : x[2], b1 = odd ? x[3] : p1;
    const float q0 = from_lane<0x4e>(upper ? a0 : b0), q1 = from_lane<0x4e>(upper ? a1 : b1);
    return f32x4{upper ? q0 : a0, upper ? q1 : a1, upper ? b0 : q0, upper ? b1 : q1};
  }
  static __device__ __forceinline__ int row(int t, int lane) { return t / (2 * WN) * 16 + (lane >> 4) * 4 + (lane & 3); }
  static __device__ __forceinline__ int col(int t, int lane) { return t % (2 * WN) * 16 + (lane & 12); }
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < 2 * WM; ++i)
#pragma unroll
      for (int j = 0; j < 2 * WN; ++j) v[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
};

struct TwoFourOperand {
  const unsigned char* form;
  const int* counts;
  const unsigned* lists;
  int phases, spill_phases, list_room;
  size_t panel;
};

constexpr int kTwoFourBN = 256;
constexpr int two_four_stage_bytes(int bm) { return (bm == 192 ? 14 * 1024 : bm * 72) + kTwoFourBN * 128; }
constexpr int two_four_lds_bytes(int bm) { return 3 * two_four_stage_bytes(bm); }

// One tile of BM = 64 * WM rows x 256 columns by eight wavefronts, 32 * WM x 64 each.  Three stages in LDS of a block of the form
// (BM * 72 bytes) and of 64 rows of B (32 KB).
//
// Step t multiplies block t with rows t of B.  B's fragments are in registers when it starts (two sets, the step's parity says which);
// the sparse operand's are read two or three row blocks ahead of their use, from LDS, through a ring of registers.  In the
// middle of the step every wavefront waits for its own loads of block t + 1 and rows t + 1 and meets the others; from then on
// the fragments of step t + 1 can be read, and what step t - 1 (block) and step t (rows of B) lived in is free for the
// direct loads of block t + 2 and of rows t + 3.  So a step has one barrier, nobody waits for an LDS read at it, B's loads have two
// steps to land and the form's one.
//
// What bounds it (2:4, 4096 x 4096 x 8192, fp16, 256 rows: 136 - 149 us by the card, 1850 - 2000 dense-equivalent TFLOP/s, where the dense
// product takes 188 - 195): the power limit and the way from L2.  MFMAs alone would take 85 us at the clock they leave the card
// (smfmac and nothing else: 3420 TFLOP/s on random operands, 4890 on zeros), the direct loads alone 75 (50 KB a step and CU, the L1's 64
// bytes a clock are 70 % busy), LDS reads alone 35; with all-zero B the product takes 124.  The schedule before this one, two
// groups of wavefronts in alternating phases as in gemm_pp_device.cuh, took 183: its memory phases are longer than 32 MFMAs, which in the
// dense product are 64 k's work and here 32's.  This one with a step's loads in one burst 186, spread over the step 176,
// with single MFMAs between the other instructions instead of four in a row 149.
template <bool BF16, int WM>
__device__ __forceinline__ void two_four_tile(const GemmParams& p, const TwoFourOperand& f, int tile_m, int tile_n, unsigned char* smem) {
  constexpr int WN = 2, WCN = 4, WAVES = 8;
  constexpr int BM = 2 * WM * 32, BN = kTwoFourBN;
  constexpr int BLOCK = BM == 192 ? 14 * 1024 : BM * 72;
  constexpr int A_STAGE = BLOCK, B_STAGE = BN * 128, A_BASE = 3 * B_STAGE;
  constexpr int ROWS = 2 * WM, COLS = 2 * WN;                  // fragments of a wavefront
  constexpr int RING = WM == 3 ? 3 : 4, AHEAD = WM == 4 ? 3 : 2;   // (a step's row blocks are whole turns of the ring)
  // direct loads per wavefront and block: 256 rows: 2 KB of entries and 256 bytes of index bits; 192: 2 KB of the block's 14 (the first two again
  // by the last wavefront); 128: 1 KB and 256 bytes (the index bits by two wavefronts each)
  constexpr int A_INSTR = BM == 128 ? 1 : 2, INDEX_INSTR = BM == 192 ? 0 : 1, B_INSTR = 4, LOADS = A_INSTR + INDEX_INSTR + B_INSTR;
  static_assert(WM >= 2 && WM <= 4 && ROWS % RING == 0 && AHEAD <= WM, "tiles of 128, 192 or 256 rows");
  typedef unsigned short u16;
  typedef __attribute__((address_space(3))) unsigned char lds_u8;
  typedef const __attribute__((address_space(4))) unsigned* scalar_list;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WCN, wn = wave % WCN;
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const u16* __restrict__ B = static_cast<const u16*>(p.B);
  u16* __restrict__ C = static_cast<u16*>(p.C);
  const unsigned lds0 = (unsigned)(size_t)(lds_u8*)smem;
  const int ldb = p.ldb, kb = p.kb;

  const u32x4 a_buf = buffer_of(f.form + tile_m * f.panel, f.panel);
  const u32x4 b_buf = buffer_of(B, rows_bytes(kb, p.N, ldb));
  const int counts[2] = {__builtin_amdgcn_readfirstlane(min(f.counts[tile_m * 2], f.list_room)),
                         __builtin_amdgcn_readfirstlane(min(f.counts[tile_m * 2 + 1], f.list_room))};
  const int P0 = f.phases, P = P0 + min((max(counts[0], counts[1]) + 31) / 32, f.spill_phases);
  const int my_count = counts[wm];
  // what this lane fetches of B: wavefront w has k rows 8 w .. 8 w + 7 of a stage (so a wavefront's rows of a spill block are those of its half panel)
  unsigned b_lane[B_INSTR];
#pragma unroll
  for (int q = 0; q < B_INSTR; ++q) b_lane[q] = column_chunk<BN>(wave * B_INSTR + q, lane, n0, ldb).offset;
  const unsigned b_step = 64u * ldb * 2u, b_row = ldb * 2u;
  const scalar_list my_list = (scalar_list)(f.lists + (size_t)(tile_m * 2 + wm) * f.list_room);
  const unsigned lane16 = lane * 16, lane4 = lane * 4;

  // load n of the LOADS of a step: block ta of the form into stage sa, then rows tb of B into stage sb (LDS offsets of the stages).  LISTED: rows of
  // B that may not be 64 in a row.
  auto issue = [&](auto number, auto listed, int ta, unsigned sa, int tb, unsigned sb) {
    constexpr int n = decltype(number)::value;
    if constexpr (n < A_INSTR + INDEX_INSTR) {
      const unsigned at = (unsigned)(decltype(listed)::value ? min(ta, P - 1) : ta) * BLOCK;
      if constexpr (n < A_INSTR) {
        int i = wave * A_INSTR + n;
        if (BM == 192 && i >= 14) i -= 14;
        lds_dma16(a_buf, lane16, at + i * 1024, __builtin_amdgcn_readfirstlane(lds0 + sa + i * 1024));
      } else {
        const int i = BM * 64 + (BM == 128 ? wave % 4 : wave) * 256;
        lds_dma4(a_buf, lane4, at + i, __builtin_amdgcn_readfirstlane(lds0 + sa + i));
      }
    } else {
      constexpr int q = n - A_INSTR - INDEX_INSTR;
      const unsigned to = __builtin_amdgcn_readfirstlane(lds0 + sb + (wave * B_INSTR + q) * 1024);
      if constexpr (!decltype(listed)::value) {
        lds_dma16(b_buf, b_lane[q], (unsigned)tb * b_step, to);
      } else {
        // The rows of pairs (past B's last: that one again, which meets zeros), or the rows that this half's list names (past its end, and past
        // the last step: row 0, not multiplied)
        const int kr = wave * 8 + q * 2;
        unsigned r0 = 0, r1 = 0;
        if (tb < P0) {
          r0 = min(tb * 64 + kr, kb - 1);
          r1 = min(tb * 64 + kr + 1, kb - 1);
        } else {
          const int e = (tb - P0) * 32 + (kr & 31);
          if (e < my_count) r0 = my_list[e];
          if (e + 1 < my_count) r1 = my_list[e + 1];
        }
        lds_dma16(b_buf, b_lane[q] + (lane < 32 ? r0 - kr : r1 - kr - 1) * b_row, 0u, to);
      }
    }
  };
  // A step's loads go out one by one over a whole step, from the middle of one to the middle of the next: in a burst they
  // fill the queue before the L1 (64 bytes a clock), and a wavefront that cannot issue a load issues no MFMA either.
  auto issue_slot = [&](auto slot, auto listed, int ta, unsigned sa, int tb, unsigned sb) {
    for_each_number<LOADS>([&](auto n) {
      if constexpr (decltype(n)::value * ROWS / LOADS == decltype(slot)::value) issue(n, listed, ta, sa, tb, sb);
    });
  };
  auto issue_all = [&](int from, int to, int ta, unsigned sa, int tb, unsigned sb) {
    for_each_number<LOADS>([&](auto n) {
      if (decltype(n)::value >= from && decltype(n)::value < to) issue(n, std::true_type{}, ta, sa, tb, sb);
    });
  };

  AccRows<WM, WN> acc;
  acc.clear();
  const int a_off = wm * WM * 2048 + lane * 16, index_off = BM * 64 + wm * WM * 256 + lane * 4;
  int b_off[COLS];
#pragma unroll
  for (int j = 0; j < COLS; ++j) b_off[j] = kn16_fragment_offset<BN>(lane, wn * COLS + j);

  u32x4 fa[RING];
  unsigned index[WM];
  u32x8 fb[2][COLS];
  auto read_a = [&](unsigned stage, int i) {
    fa[i % RING] = *reinterpret_cast<const u32x4*>(smem + stage + a_off + i * 1024);
    if (i % 2 == 0) index[i / 2] = *reinterpret_cast<const unsigned*>(smem + stage + index_off + i / 2 * 256);
  };
  // half h (32 k) of column block j.  A spill block has 32 rows of B for each half panel.
  auto read_b = [&](unsigned stage, int set, int j, int h, auto spill) {
    if (decltype(spill)::value && h) return;
    const u32x4 v = kn_fragment<BN * 2>(smem + stage + b_off[j] + (decltype(spill)::value ? wm : h) * 32 * (BN * 2));
#pragma unroll
    for (int e = 0; e < 4; ++e) fb[set][j][h * 4 + e] = v[e];
  };
  const std::integral_constant<int, 0> even;
  const std::integral_constant<int, 1> odd;
  const std::false_type no;
  const std::true_type yes;

  // LDS offsets of the stages of steps t, t + 1, t + 2 (and t + 3 goes where t was)
  unsigned a_now = A_BASE, a_next = A_BASE + A_STAGE, a_after = A_BASE + 2 * A_STAGE, b_now = 0, b_next = B_STAGE, b_after = 2 * B_STAGE;
  auto step = [&](int t, auto parity, auto this_spill, auto next_spill, auto listed) {
    constexpr int set = decltype(parity)::value;
    const bool idle = decltype(this_spill)::value && (t - P0) * 32 >= my_count;   // (uniform; the other half's list may be longer)
    for_each_number<ROWS>([&](auto row_block) {
      constexpr int i = decltype(row_block)::value, late = i >= WM;
      // One MFMA (16 clocks), then something for another unit, and so on: what a wavefront issues beside its own MFMAs costs them nothing
      auto multiply = [&](auto column) {
        constexpr int j = decltype(column)::value;
        if constexpr (j < COLS) {
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (!decltype(this_spill)::value) acc.v[i][j] = smfmac_16x16x64<BF16, i % 2>(fa[i % RING], fb[set][j], acc.v[i][j], index[i / 2]);
          else if (!idle) acc.v[i][j] = mfma_16x16x32<BF16>(fa[i % RING], u32x4{fb[set][j][0], fb[set][j][1], fb[set][j][2], fb[set][j][3]}, acc.v[i][j]);
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      multiply(std::integral_constant<int, 0>{});
      if constexpr (i == WM) {
        wait_vmcnt<B_INSTR>();   // my loads of block t + 1 and of rows t + 1 have landed; those of rows t + 2 may fly
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
      if constexpr (i + AHEAD < ROWS) read_a(a_now, i + AHEAD);
      else read_a(a_next, i + AHEAD - ROWS);
      multiply(std::integral_constant<int, 1>{});
      if constexpr (late) {
#pragma unroll
        for (int j = (i - WM) * COLS / WM; j < (i - WM + 1) * COLS / WM; ++j) read_b(b_next, set ^ 1, j, 0, next_spill);
      }
      multiply(std::integral_constant<int, 2>{});
      if constexpr (late) {
#pragma unroll
        for (int j = (i - WM) * COLS / WM; j < (i - WM + 1) * COLS / WM; ++j) read_b(b_next, set ^ 1, j, 1, next_spill);
      }
      multiply(std::integral_constant<int, 3>{});
      if constexpr (late) issue_slot(std::integral_constant<int, i - WM>{}, listed, t + 2, a_after, t + 3, b_now);
      else issue_slot(std::integral_constant<int, i + WM>{}, listed, t + 1, a_next, t + 2, b_after);
    });
    const unsigned a_was = a_now, b_was = b_now;
    a_now = a_next, a_next = a_after, a_after = a_was;
    b_now = b_next, b_next = b_after, b_after = b_was;
  };

  constexpr int EARLY = (WM * LOADS + ROWS - 1) / ROWS;   // loads before a step's end: n with n * ROWS / LOADS < WM
  issue_all(0, LOADS, 0, a_now, 0, b_now);
  issue_all(LOADS - B_INSTR, LOADS, 0, 0, 1, b_next);
  issue_all(0, EARLY, 1, a_next, 2, b_after);
  wait_vmcnt<B_INSTR + EARLY>();
  __syncthreads();
#pragma unroll
  for (int j = 0; j < COLS; ++j) read_b(b_now, 0, j, 0, no), read_b(b_now, 0, j, 1, no);
#pragma unroll
  for (int i = 0; i < AHEAD; ++i) read_a(a_now, i);

  int t = 0;   // (P0 is even)
  const int plain = min(kb / 64, P0 - 1) - 3;   // steps whose loads are whole blocks of 64 rows, and of pairs
  for (; t + 1 < plain; t += 2) {
    step(t, even, no, no, no);
    step(t + 1, odd, no, no, no);
  }
  for (; t < P0 - 2; t += 2) {
    step(t, even, no, no, yes);
    step(t + 1, odd, no, no, yes);
  }
  step(t, even, no, no, yes);
  step(t + 1, odd, no, yes, yes);
  for (t += 2; t < P; t += 2) {   // (an odd last step is followed by one that multiplies nothing)
    step(t, even, yes, yes, yes);
    step(t + 1, odd, yes, yes, yes);
  }
  wait_vmcnt<0>();   // the re-fetched last blocks: nothing may still be writing LDS when the stages are reused
  static_assert(WAVES * gemm_store_lds_bytes<WN>() <= two_four_lds_bytes(BM), "the epilogue fits the stages");
  __syncthreads();
  const u16* aux = static_cast<const u16*>(p.aux);
  gemm_store_tile<BF16, WM, WN>(p, acc, C, aux, m0, n0, wm, wn, lane, smem + wave * gemm_store_lds_bytes<WN>(), p.stream_out != 0);
}

}  // namespace iex
