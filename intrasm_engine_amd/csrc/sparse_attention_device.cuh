// Sparse attention over a CSR mask for gfx950 in one kernel: out = softmax(scale * q k^T at the mask's entries) v per head,
// operands (heads, tokens, HD), HD = 32, 64 or 128, fp16 / bf16 / fp32.  Scores and probabilities exist in registers only.
//
// By three kernels (SDDMM, softmax over CSR rows, SpMM) the scores of 16 heads over 287 entries per row of 4096 went
// through memory five times (38 MB each way), the gather kernels read 2 * HD * size bytes per entry through the L2 -> CU path,
// and a short prompt was three launches of 5 - 20 us.  Us per call before / here: 8 heads x 1000 tokens, causal band of 256,
// bf16: 37 / 6.8; 16 x 4096, band 256 + 32 scattered, fp16: 81 / 38.7; 32 x 2048 x 128, causal band of 512, fp32: 1121 / 182.
//
// The mask's tables (made once per mask by mask_tables_kernel): per block of 128 rows the 64-column tiles that hold at
// least dense_min / 4 entries for each group of 32 rows that has any there ("dense"), for each of them a 64-bit word per row, and per row the columns outside dense tiles.
// Which tiles are better off as dense ones is not the same for every launch, and the tables are made before one is known: those between two limits stand at the
// end of the list, their entries at the end of the rows' lists, and a launch takes them one way or the other.
// A wavefront owns 32 queries, a workgroup QW wavefronts (fewer where the heads are few: more workgroups, and fewer tiles
// that only some of its wavefronts want), or KW wavefronts share 32 queries, each with every KW-th tile and stages of its own
// (8 heads x 1000 tokens, fp32: 27.8 -> 16 us), with more wavefronts beside them that do nothing but the other entries: their chains run
// beside the tiles' on the SIMDs that the stages' LDS leaves empty (8 x 1500 of 128, band 64 + 32 scattered, bf16 44.9 -> 25.4 us, fp32 16 x 1214 of 128
// + 16 118 -> 66, 12 x 3280 of 64 + 32 102 -> 81; by no scattered entries but the band's corners, 8 x 1000 of 64, 8.2 -> 7.7).
//   * dense tiles as in attention_device.cuh: K and V rows of a tile straight into LDS, two stages; S^T = K Q^T on the
//     matrix cores, entries outside the mask to -infinity by the row's word, running maximum and sum per query in registers,
//     O^T += V^T P^T with the probabilities as they lie in the lanes.  fp32 goes by v_mfma_f32_32x32x2, tiles in halves.
//   * other entries: HD * size / 16 lanes per row walk the row's list, 4 or 8 entries at a time, 16 bytes of each K and V
//     row per lane, dot products across the lanes, a softmax state per row; rows' results meet the dense part's in LDS.
// What bounds it (profiles/kernel_counters_of_the_cases.txt): for 16-bit types vector instructions, 270 - 300 per wavefront and
// tile for the softmax (1100 - 1200 clocks beside 512 of MFMAs) and 4 per scattered entry, on the two wavefronts per SIMD that
// LDS leaves room for; a short prompt is the chain of a wavefront's few tiles (59 % waiting); for fp32 the MFMAs (4096 clocks
// per half tile of HD = 64; busy 60 %).
#pragma once
#include "gemm_dma_device.cuh"
#include "online_softmax_device.cuh"

namespace iex {

constexpr int kMaRows = 128, kMaCols = 64, kMaMaxTokens = 16384;
constexpr int kMaEntries = 1 << 31;
constexpr int kMaEither = 1 << 30;

// Where the parts of a mask's tables lie in their memory.  They hold all that the kernel reads of the mask: a recorded launch
// works on the mask as it was, whatever becomes of the index arrays.
struct MaskTables {
  int blocks, tiles;            // blocks of 128 rows, tiles of 64 columns
  size_t list, ends, thin, thin_cols, bits, bytes;   // byte offsets and the total
};
inline __host__ __device__ MaskTables mask_tables_layout(int m, int n, int nnz) {
  MaskTables t;
  t.blocks = (m + kMaRows - 1) / kMaRows;
  t.tiles = (n + kMaCols - 1) / kMaCols;
  t.list = 0;                                                              // int [blocks][tiles + 1]: how many; tile | wavefronts of 32 rows << 16
  t.ends = t.list + (size_t)t.blocks * (t.tiles + 1) * 4;                  // for launches that take the tiles at the list's end: int [blocks]: how many tiles; [blocks * 128]: how many entries of a row
  t.thin = (t.ends + (size_t)t.blocks * (1 + kMaRows) * 4 + 7) / 8 * 8;    // int2 [blocks * 128]: where a row's begin (kMaEntries: it has entries); how many
  t.thin_cols = t.thin + (size_t)t.blocks * kMaRows * 8;                   // int [nnz]: row r's from row_offsets[r]
  t.bits = (t.thin_cols + (size_t)nnz * 4 + 255) / 256 * 256;              // u64 [blocks][tiles][128]: by position in the list
  t.bytes = t.bits + (size_t)t.blocks * t.tiles * kMaRows * 8;
  return t;
}

// One workgroup of 16 wavefronts per block of 128 rows, a wavefront per row at a time.  Columns ascend inside a row.
constexpr int kMtWaves = 16;
inline __host__ __device__ int mask_tables_lds_bytes(int tiles) { return tiles * 3 * 4 + kMtWaves * tiles * 8; }

__global__ __launch_bounds__(kMtWaves * kWave) void mask_tables_kernel(int m, int n, int nnz, int dense_min, int either_min, const int* __restrict__ row_offsets,
                                                                       const int* __restrict__ cols, unsigned char* __restrict__ ws) {
  extern __shared__ __align__(16) int mt_smem[];
  const MaskTables t = mask_tables_layout(m, n, nnz);
  const int tiles = t.tiles, rb = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int* count = mt_smem;             // [tiles]: entries; then the tile's position in the list (| kMaEither), or -1
  int* groups = count + tiles;      // [tiles]: bit g: rows 32 g .. 32 g + 31 have entries there
  int* dense = groups + tiles;      // [tiles]: the list
  unsigned* map = reinterpret_cast<unsigned*>(dense + tiles) + wave * tiles * 2;   // [tiles * 2]: this wavefront's row, a bit per column
  int* list = reinterpret_cast<int*>(ws + t.list) + (size_t)rb * (tiles + 1);
  int* ends = reinterpret_cast<int*>(ws + t.ends);
  int2* thin_of = reinterpret_cast<int2*>(ws + t.thin) + (size_t)rb * kMaRows;
  int* thin_cols = reinterpret_cast<int*>(ws + t.thin_cols);
  unsigned long long* bits = reinterpret_cast<unsigned long long*>(ws + t.bits) + (size_t)rb * tiles * kMaRows;
  for (int i = threadIdx.x; i < 2 * tiles; i += blockDim.x) count[i] = 0;
  __syncthreads();
  for (int r = wave; r < kMaRows; r += kMtWaves) {
    const int row = rb * kMaRows + r;
    if (row >= m) break;   // (uniform)
    const int start = row_offsets[row], end = row_offsets[row + 1];
    for (int j0 = start; j0 < end; j0 += kWave) {
      const int j = j0 + lane, tile = j < end ? cols[j] >> 6 : -1;
      const int before = __shfl_up(tile, 1);
      const bool first = tile >= 0 && (lane == 0 || tile != before);   // of a run of lanes with this tile
      const unsigned long long firsts = __ballot(first), here = __ballot(tile >= 0);
      if (first) {
        const unsigned long long later = lane == 63 ? 0ull : firsts & (~0ull << (lane + 1));
        const int upto = later ? __ffsll((long long)later) - 1 : __popcll(here);
        atomicAdd(&count[tile], upto - lane);
        atomicOr(&groups[tile], 1 << (r / 32));
      }
    }
  }
  __syncthreads();
  if (wave == 0) {   // the list, in the order of the tiles
    int had = 0, certain = 0;
    for (int pass = 0; pass < 2; ++pass) {   // dense for all, for some
      for (int base = 0; base < tiles; base += kWave) {
        const int tile = base + lane;
        // (a tile costs every group of 32 rows that has entries there: a band's corner with entries of one group is worth it from a quarter on; fp32, 8 x 1544 of
        // 32, band 512 + 16 scattered, 31.5 -> 23 us, 16 x 1179 of 64, band 64, 33.8 -> 27.7)
        const int there = tile < tiles ? count[tile] : 0, of = tile < tiles ? __popc((unsigned)groups[tile]) : 0;
        const bool is = pass ? there == -2 : there > 0 && 4 * there >= dense_min * of;
        const unsigned long long them = __ballot(is);
        if (is) {
          const int at = had + __popcll(them & ((1ull << lane) - 1));
          count[tile] = at | (pass ? kMaEither : 0);
          dense[at] = tile;
          list[1 + at] = tile | (groups[tile] << 16);
        } else if (pass == 0 && tile < tiles) {
          count[tile] = there > 0 && 4 * there >= either_min * of ? -2 : -1;
        }
        had += __popcll(them);
      }
      if (pass == 0) certain = had;
    }
    if (lane == 0) {
      list[0] = certain;
      ends[rb] = had;
      groups[0] = certain | had << 16;   // (the groups are done)
    }
  }
  __syncthreads();
  const int nd = groups[0] >> 16;
  const bool either_way = nd > (groups[0] & 0xffff);
  for (int r = wave; r < kMaRows; r += kMtWaves) {
    const int row = rb * kMaRows + r;
    for (int i = lane; i < 2 * tiles; i += kWave) map[i] = 0;
    int thin = 0, both = 0, begin = 0;
    if (row < m) {
      const int start = row_offsets[row], end = row_offsets[row + 1];
      begin = start | (start < end ? kMaEntries : 0);
      for (int j0 = start; j0 < end; j0 += kWave) {
        const int j = j0 + lane, col = j < end ? cols[j] : -1;
        const bool to_thin = col >= 0 && count[col >> 6] < 0;
        if (col >= 0 && !to_thin) atomicOr(&map[col >> 5], 1u << (col & 31));
        const unsigned long long them = __ballot(to_thin);
        if (to_thin) thin_cols[start + thin + __popcll(them & ((1ull << lane) - 1))] = col;
        thin += __popcll(them);
      }
      both = thin;
      if (either_way)
        for (int j0 = start; j0 < end; j0 += kWave) {
          const int j = j0 + lane, col = j < end ? cols[j] : -1;
          const bool either = col >= 0 && count[col >> 6] >= kMaEither;
          const unsigned long long them = __ballot(either);
          if (either) thin_cols[start + both + __popcll(them & ((1ull << lane) - 1))] = col;
          both += __popcll(them);
        }
    }
    if (lane == 0) thin_of[r] = int2{begin, both}, ends[t.blocks + rb * kMaRows + r] = thin;
    __builtin_amdgcn_wave_barrier();   // (the LDS operations of one wavefront execute in order)
    for (int s = lane; s < nd; s += kWave) {
      const int tile = dense[s];
      bits[(size_t)s * kMaRows + r] = (unsigned long long)map[2 * tile] | (unsigned long long)map[2 * tile + 1] << 32;
    }
    __builtin_amdgcn_wave_barrier();
  }
}

struct SparseAttentionParams {
  int heads, tokens, nnz;
  const void* q;
  const void* k;
  const void* v;
  void* out;
  float scale_log2;        // scale * log2(e), > 0
  const unsigned char* tables;
};

template <int TYPE, int HD>   // TYPE: 0 = fp16, 1 = bf16, 2 = fp32
struct SparseAttentionShape {
  static constexpr int ES = TYPE == 2 ? 4 : 2;
  static constexpr int KEYS = TYPE == 2 ? 32 : 64;          // of a stage
  static constexpr int CPR = HD * ES / 16;                  // 16-byte chunks per row
  static constexpr int TILE = KEYS * HD * ES;               // bytes of K or V per stage
  static constexpr int TLD = HD + 4;                        // floats per row of the scattered entries' results
  static constexpr int stages(int qw, int kw) { return kw * 2 * (2 * TILE + qw * 256); }
  // by several wavefronts to 32 queries the scattered entries' results lie behind the stages, else in their place
  static constexpr int lds(int qw, int kw) {
    const int thin = qw * 32 * (TLD + 4) * 4;
    return kw > 1 ? stages(qw, kw) + thin : stages(qw, kw) > thin ? stages(qw, kw) : thin;
  }
  // wavefronts beside those KW, for the scattered entries alone
  static constexpr int extra(int kw) { return kw == 1 ? 0 : kw == 2 ? 6 : 4; }
  // Tiles that may be taken either way as dense ones: where the same wavefronts do the other entries afterwards, 16 lanes to each.  (16-bit, us as entries / as tiles: 32 heads x 533 of 128,
  // band 256 + 16 scattered 26.8 / 23.8; 32 x 677 of 128, causal, 64 + 32 35.6 / 30.7; 32 x 1000 of 128, 64 + 32 41.6 / 42.1, of 64 24.3 / 25.8, of 32 16.3 / 20.8; lists beside
  // the tiles: 4 x 1000 of 128 13.8 / 20.4, 32 x 500 of 128 19.5 / 24.0, 12 x 1266 of 128 26.7 / 29.1)
  static constexpr bool takes_either(int kw) { return kw == 1 && HD == 128; }
};

// LDS row of a key (or chunk permutation of a row): what keeps the operand reads of 16 consecutive lanes apart.
template <int CPR>
__device__ __forceinline__ int sa_key_swizzle(int row) { return CPR == 4 ? (row >> 2) & 3 : CPR == 8 ? (row >> 1) & 7 : row & 15; }
template <int TYPE, int HD>
__device__ __forceinline__ int sa_value_swizzle(int row) {
  if constexpr (TYPE == 2) return HD >= 64 ? ((row >> 2) & 1) << 3 : 0;
  return HD >= 64 ? kn_swizzle<HD>(row) : 0;
}

template <int TYPE>
__device__ __forceinline__ float sa_dot(u32x4 a, u32x4 b) {
  float acc = 0.f;
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (TYPE == 2) acc = fmaf(__uint_as_float(a[i]), __uint_as_float(b[i]), acc);
    else if constexpr (TYPE == 1) acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2, (unsigned)a[i]), __builtin_bit_cast(b2, (unsigned)b[i]), acc, false);
    else acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, (unsigned)a[i]), __builtin_bit_cast(h2, (unsigned)b[i]), acc, false);
  }
  return acc;
}

// The whole row's product out of its CPR lanes' chunks; every one of them gets it.
template <int TYPE, int CPR>
__device__ __forceinline__ float sa_row_dot(u32x4 a, u32x4 b) {
  float x = group_sum<(CPR > 16 ? 16 : CPR)>(sa_dot<TYPE>(a, b));
  if constexpr (CPR == 32) x += __shfl_xor(x, 16);
  return x;
}

// acc += w * the elements of a chunk
template <int TYPE>
__device__ __forceinline__ void sa_add_row(float* acc, float w, u32x4 chunk) {
#pragma unroll
  for (int e = 0; e < (TYPE == 2 ? 4 : 8); ++e) {
    float x;
    if constexpr (TYPE == 2) x = __uint_as_float(chunk[e]);
    else x = f16_to_32((unsigned short)(chunk[e / 2] >> (16 * (e & 1))), TYPE == 1);
    acc[e] = fmaf(w, x, acc[e]);
  }
}

template <int TYPE, int HD, int QW, int KW>
__global__ __launch_bounds__((QW * KW + SparseAttentionShape<TYPE, HD>::extra(KW)) * kWave, 2) void sparse_attention_kernel(SparseAttentionParams p) {
  typedef SparseAttentionShape<TYPE, HD> Shape;
  constexpr int ES = Shape::ES, KEYS = Shape::KEYS, CPR = Shape::CPR, TILE = Shape::TILE, TLD = Shape::TLD;
  constexpr bool F32 = TYPE == 2;
  constexpr int XW = Shape::extra(KW);              // (wavefronts KW .. KW + XW - 1)
  constexpr bool TAKE = Shape::takes_either(KW);    // tiles that are dense for some as dense ones
  constexpr int PER = kMaCols / KEYS;               // stages per tile of the mask
  constexpr int KB = KEYS / 32, DT = HD / 32;       // blocks of 32 keys, of 32 features
  constexpr int RPI = kWave / CPR;                  // rows per direct load
  constexpr int INSTR = TILE / 1024 / QW;           // direct loads per wavefront, operand and stage
  static_assert(TILE % (1024 * QW) == 0, "whole kilobytes per wavefront");
  static_assert(QW == 1 || KW == 1, "either queries or keys are shared out");
  constexpr float kNone = -1e30f;                   // the maximum of no entries (finite: differences of it are)
  typedef __attribute__((address_space(3))) unsigned char lds_u8;
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int STAGE = 2 * TILE, MASKS = 2 * STAGE;
  const int lane = threadIdx.x & 63, kw = KW > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  const int wave = KW > 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // of the queries
  const int half = lane >> 5, col = lane & 31;
  const int T = p.tokens;
  unsigned char* stages = smem + kw * (MASKS + QW * 512);
  // workgroups go to the XCDs round-robin; renumbered so that an XCD gets all queries of a head, whose K and V stay in its L2
  const int blocks = (T + QW * 32 - 1) / (QW * 32), total = gridDim.x;
  const int id = total % kXcds == 0 ? (blockIdx.x % kXcds) * (total / kXcds) + blockIdx.x / kXcds : blockIdx.x;
  const int q0 = (id % blocks) * (QW * 32), head = id / blocks;
  const int rb = q0 / kMaRows, group0 = q0 % kMaRows / 32;
  const size_t at = (size_t)head * T * HD * ES;
  const unsigned char* q = static_cast<const unsigned char*>(p.q) + at;
  const unsigned char* k = static_cast<const unsigned char*>(p.k) + at;
  const unsigned char* v = static_cast<const unsigned char*>(p.v) + at;
  const MaskTables mt = mask_tables_layout(T, T, p.nnz);
  const int* __restrict__ list = reinterpret_cast<const int*>(p.tables + mt.list) + (size_t)rb * (mt.tiles + 1);
  const int* __restrict__ ends = reinterpret_cast<const int*>(p.tables + mt.ends);
  const unsigned char* bits = p.tables + mt.bits + ((size_t)rb * mt.tiles * kMaRows + (group0 + wave) * 32) * 8;
  const unsigned lds0 = (unsigned)(size_t)(lds_u8*)stages;
  const u32x4 k_buf = buffer_of(k, (size_t)T * HD * ES), v_buf = buffer_of(v, (size_t)T * HD * ES);   // (rows past the end: zeros)

  // ---- this lane's query (fragments: features half * 8 .. + 7 of every 16; fp32: half * 4 .. + 3 of every 8)
  const int query = q0 + wave * 32 + col;
  u32x4 fq[HD * ES / 32];
#pragma unroll
  for (int s = 0; s < HD * ES / 32; ++s) fq[s] = *reinterpret_cast<const u32x4*>(q + ((size_t)min(query, T - 1) * HD * ES + (s * 2 + half) * 16));

  unsigned k_lane[INSTR], v_lane[INSTR];
#pragma unroll
  for (int i = 0; i < INSTR; ++i) {
    const int row = (wave * INSTR + i) * RPI + lane / CPR, c = lane % CPR;
    k_lane[i] = (row * CPR + (c ^ sa_key_swizzle<CPR>(row))) * 16;
    v_lane[i] = (row * CPR + (c ^ sa_value_swizzle<TYPE, HD>(row))) * 16;
  }
  auto issue = [&](int entry, int position, int part, int stage) {
    const unsigned from = ((entry & 0xffff) * PER + part) * TILE;
#pragma unroll
    for (int i = 0; i < INSTR; ++i) {
      const unsigned base = lds0 + stage * STAGE + (wave * INSTR + i) * 1024;
      lds_dma16(k_buf, k_lane[i], from, __builtin_amdgcn_readfirstlane(base));
      lds_dma16(v_buf, v_lane[i], from, __builtin_amdgcn_readfirstlane(base + TILE));
    }
    const unsigned char* words = bits + (size_t)position * kMaRows * 8 + lane * 4;
    asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dword %0, off" ::"v"(words),
                 "s"(__builtin_amdgcn_readfirstlane(lds0 + MASKS + (stage * QW + wave) * 256)) : "memory", "m0");
  };

  f32x16 o[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[d][r] = 0.f;
  float top = kNone, sum = 0.f;   // of this lane's query: the maximum so far (both lanes' keys), this lane's share of the sum

  auto tile = [&](int stage, int part) {
    const unsigned char* sk = stages + stage * STAGE;
    const unsigned char* sv = sk + TILE;
    // ---- scores: rows = keys.  16-bit: key 4..7 and 8..11 of every 16 change places, so that a lane's 8 sums of 16 keys are
    // 8 consecutive keys, the operand of the second product; fp32: sum r is key r / 4 * 8 + half * 4 + r % 4
    f32x16 s[KB];
    const int key_row = F32 ? col : (col & 19) | ((col & 4) << 1) | ((col & 8) >> 1);
#pragma unroll
    for (int b = 0; b < KB; ++b) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[b][r] = 0.f;
      const int row = b * 32 + key_row;
      const unsigned char* at_row = sk + row * CPR * 16;
#pragma unroll
      for (int e = 0; e < HD * ES / 32; ++e) {
        const u32x4 fk = *reinterpret_cast<const u32x4*>(at_row + (((e * 2 + half) ^ sa_key_swizzle<CPR>(row)) * 16));
        if constexpr (F32) {
#pragma unroll
          for (int x = 0; x < 4; ++x)
            s[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(fk[x]), __uint_as_float(fq[e][x]), s[b], 0, 0, 0);
        } else {
          s[b] = mfma_32x32x16<TYPE == 1>(fk, fq[e], s[b]);
        }
      }
    }
    // ---- the mask
    u32x2 word = *reinterpret_cast<const u32x2*>(stages + MASKS + (stage * QW + wave) * 256 + col * 8);
    if constexpr (F32) word.x = word.y = part ? word.y : word.x;
    if (__ballot((word.x & word.y) != 0xffffffffu)) {   // (uniform) some entry of some query is not there
#pragma unroll
      for (int b = 0; b < KB; ++b) {
        const unsigned mine = (b ? word.y : word.x) >> (F32 ? half * 4 : half * 8);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const unsigned there = (unsigned)__builtin_amdgcn_sbfe((int)mine, F32 ? r / 4 * 8 + r % 4 : r / 8 * 16 + r % 8, 1);
          s[b][r] = __uint_as_float((__float_as_uint(s[b][r]) & there) | (0xff800000u & ~there));
        }
      }
    }
    softmax_maximum(s, o, top, sum, p.scale_log2);
#pragma unroll
    for (int b = 0; b < KB; ++b) softmax_weights<16>(s[b], 0, top, sum, p.scale_log2);
    // ---- times V: rows = features
    if constexpr (F32) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = r / 4 * 8 + half * 4 + r % 4;
#pragma unroll
        for (int d = 0; d < DT; ++d) {
          const int c = (d * 8 + col / 4) ^ sa_value_swizzle<TYPE, HD>(row);
          const float fv = *reinterpret_cast<const float*>(sv + (row * CPR + c) * 16 + col % 4 * 4);
          o[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(fv, s[0][r], o[d], 0, 0, 0);
        }
      }
    } else {
#pragma unroll
      for (int e = 0; e < KEYS / 16; ++e) {
        const u32x4 fp = probability_operand<TYPE == 1>(s[e / 2], e % 2 * 8);
        const int kr = half * 8 + ((lane & 15) >> 2);
#pragma unroll
        for (int d = 0; d < DT; ++d) {
          const int c = (d * 4 + ((lane >> 4) & 1) * 2 + ((lane & 3) >> 1)) ^ sa_value_swizzle<TYPE, HD>(kr);
          const u32x4 fv = kn_fragment<HD * 2>(sv + (e * 16 + kr) * (HD * 2) + c * 16 + (lane & 1) * 8);
          o[d] = mfma_32x32x16<TYPE == 1>(fv, fp, o[d]);
        }
      }
    }
  };

  // ---- dense tiles that any of this workgroup's rows have entries in
  if (XW == 0 || kw < KW) {
    const int count = uniform(TAKE ? ends[rb] : list[0]), mine = ((1 << QW) - 1) << group0;
    int entry = 0;   // of the tile that `next` has found
    auto next = [&](int i) {
      while (i < count && (i % KW != kw || !(((entry = uniform(list[1 + i])) >> 16) & mine))) ++i;
      return i;
    };
    int i = next(0), part = 0, stage = 0;
    if (i < count) issue(entry, i, 0, 0);
    while (i < count) {
      const int now = entry;
      int ni = i, npart = part + 1;
      if (npart == PER) ni = next(i + 1), npart = 0;
      wait_vmcnt<0>();
      if constexpr (KW == 1) __syncthreads();   // everybody's loads of this stage have landed, and everybody is done with the other one
      if (ni < count) issue(entry, ni, npart, stage ^ 1);
      if ((now >> 16) & (1 << (group0 + wave))) tile(stage, part);
      i = ni;
      part = npart;
      stage ^= 1;
    }
  }
  sum += __shfl_xor(sum, 32);
  if constexpr (KW == 1) __syncthreads();   // everybody is done with the stages

  // ---- entries outside dense tiles: CPR lanes per row, G rows side by side, U entries of each at a time.  A lane holds the
  // same 16 bytes of every row of K and V, so nothing but the dot products crosses lanes.
  float* rows = reinterpret_cast<float*>(smem + (KW > 1 ? Shape::stages(QW, KW) : 0)) + wave * 32 * (TLD + 4);   // [32][TLD]: sums over them; then [32][2]: maximum, sum
  float* state = rows + 32 * TLD;
  const int row0 = q0 + wave * 32;
  const int my_row = min(row0 + col, T - 1);
  const int2* thin_of = reinterpret_cast<const int2*>(p.tables + mt.thin);
  auto thin_count = [&](int row) { return TAKE ? ends[mt.blocks + row] : thin_of[row].y; };
  const int my_count = row0 + col < T ? thin_count(my_row) : 0;
  if (__ballot(my_count > 0)) {   // (uniform)
    constexpr int G = kWave / CPR, U = HD * ES >= 256 ? 4 : 8, E = 16 / ES;
    typedef int i32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
    const int* thin_cols = reinterpret_cast<const int*>(p.tables + mt.thin_cols);
    const int sub = lane / CPR, part = lane % CPR;
    for (int r0 = (kw + XW) % (KW + XW) * G; r0 < 32; r0 += (KW + XW) * G) {
      const int row = row0 + r0 + sub, safe = min(row, T - 1);
      const int2 thin = thin_of[safe];
      const int count = row < T ? TAKE ? thin_count(safe) : thin.y : 0;
      const int* at_cols = thin_cols + (thin.x & ~kMaEntries);   // (what follows the columns in the tables may be read, not used)
      int most = count;   // of the G rows
#pragma unroll
      for (int x = CPR; x < kWave; x <<= 1) most = max(most, __shfl_xor(most, x));
      most = uniform(most);
      const u32x4 qv = *reinterpret_cast<const u32x4*>(q + ((size_t)safe * CPR + part) * 16);
      float top_r = kNone, sum_r = 0.f, acc[E];
#pragma unroll
      for (int e = 0; e < E; ++e) acc[e] = 0.f;
      i32x4_a4 next[U / 4];
#pragma unroll
      for (int x = 0; x < U / 4; ++x) next[x] = *reinterpret_cast<const i32x4_a4*>(at_cols + x * 4);
      // Past the row's last entry: its first one again, with weight 0.  Another token's V there would turn a row that is finite
      // into NaN (and be computed once more, below).  Zeroes in the registers instead: 16 x 4096, 32 scattered, 40.3 -> 41.4 us.
      const int past = count > 0 ? next[0][0] : 0;
      for (int c0 = 0; c0 < most; c0 += U) {
        u32x4 kv[U], vv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int c = c0 + u < count ? next[u / 4][u % 4] : past;
          kv[u] = *reinterpret_cast<const u32x4*>(k + ((size_t)c * CPR + part) * 16);
          vv[u] = *reinterpret_cast<const u32x4*>(v + ((size_t)c * CPR + part) * 16);
        }
        if (c0 + U < most) {
          const int from = min(c0 + U, max(count - 1, 0));   // (a row that has ended: anything of its own)
#pragma unroll
          for (int x = 0; x < U / 4; ++x) next[x] = *reinterpret_cast<const i32x4_a4*>(at_cols + from + x * 4);
        }
        float d[U], m = -INFINITY;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const float x = sa_row_dot<TYPE, CPR>(qv, kv[u]);
          d[u] = c0 + u < count ? x : -INFINITY;
          m = fmaxf(m, d[u]);
        }
        const float now = fmaxf(top_r, m), keep = __builtin_amdgcn_exp2f((top_r - now) * p.scale_log2), shift = -now * p.scale_log2;
        top_r = now;
        sum_r *= keep;
#pragma unroll
        for (int e = 0; e < E; ++e) acc[e] *= keep;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const float w = __builtin_amdgcn_exp2f(fmaf(d[u], p.scale_log2, shift));
          sum_r += w;
          sa_add_row<TYPE>(acc, w, vv[u]);
        }
      }
#pragma unroll
      for (int e = 0; e < E; e += 4) *reinterpret_cast<f32x4*>(rows + (r0 + sub) * TLD + part * E + e) = f32x4{acc[e], acc[e + 1], acc[e + 2], acc[e + 3]};
      if (part == 0) {
        state[(r0 + sub) * 2] = top_r;
        state[(r0 + sub) * 2 + 1] = sum_r;
      }
    }
  }
  if constexpr (KW > 1) {   // the sums of the other wavefronts' tiles
    constexpr int N = 16 * DT;
    float* parts = reinterpret_cast<float*>(smem);   // [KW - 1][N + 2][64]
    static_assert((KW - 1) * (N + 2) * kWave * 4 <= Shape::stages(QW, KW), "in the place of the stages");
    __syncthreads();   // everybody is done with the stages
    if (kw > 0 && kw < KW) {
      float* mine = parts + (kw - 1) * (N + 2) * kWave + lane;
#pragma unroll
      for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) mine[(d * 16 + r) * kWave] = o[d][r];
      mine[N * kWave] = top;
      mine[(N + 1) * kWave] = sum;
    }
    __syncthreads();
    if (kw > 0) return;
    for (int w = 0; w < KW - 1; ++w) {
      const float* theirs = parts + w * (N + 2) * kWave + lane;
      const float top_w = theirs[N * kWave], now = fmaxf(top, top_w);
      const float keep = __builtin_amdgcn_exp2f((top - now) * p.scale_log2), keep_w = __builtin_amdgcn_exp2f((top_w - now) * p.scale_log2);
      top = now;
      sum = sum * keep + theirs[(N + 1) * kWave] * keep_w;
#pragma unroll
      for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[d][r] = o[d][r] * keep + theirs[(d * 16 + r) * kWave] * keep_w;
    }
  }
  float top_all = top;
  if (__ballot(my_count > 0)) {   // (uniform) the sums over entries outside dense tiles
    __builtin_amdgcn_wave_barrier();   // (the LDS operations of one wavefront execute in order)
    const float top_t = state[col * 2], sum_t = state[col * 2 + 1];
    const float now = fmaxf(top, top_t);
    const float keep = __builtin_amdgcn_exp2f((top - now) * p.scale_log2), keep_t = __builtin_amdgcn_exp2f((top_t - now) * p.scale_log2);
    top_all = now;
    sum = sum * keep + sum_t * keep_t;
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(rows + col * TLD + d * 32 + g * 8 + half * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[d][g * 4 + e] = o[d][g * 4 + e] * keep + x[e] * keep_t;
      }
  }

  // ---- rows whose result the above does not give, once more, entry by entry, by the mask's words and lists: a masked key's
  // infinity or NaN in V times its weight 0 is NaN for all 32 queries (so any row that is not finite); scores that are all at
  // or below kNone, or infinite, left nothing in the sum.  Two passes over a row, its maximum first.  Looking costs 0.1 us (12
  // heads x 424 of 128: 7.96 -> 8.07); clean V in every tile would cost every tile.
  bool again = false;
  {
    float all[4] = {sum, 0.f, 0.f, 0.f};   // not finite where anything in it is not (or where products are beyond 1e38: no harm)
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int r = 0; r < 16; r += 2) all[r / 2 % 4] = fmaf(o[d][r], o[d][r + 1], all[r / 2 % 4]);
    again = query < T && !(fabsf((all[0] + all[1]) + (all[2] + all[3])) < INFINITY && sum > 0.f && top_all > kNone);
  }
  if (__ballot(again)) {   // (uniform)
    if (again && !(thin_of[query].x & kMaEntries)) {   // a row without entries: zeros
      again = false;
      sum = 0.f;
#pragma unroll
      for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[d][r] = 0.f;
    }
    const unsigned long long lanes = __ballot(again);
    const unsigned todo = (unsigned)lanes | (unsigned)(lanes >> 32);
    constexpr int G = kWave / CPR, E = 16 / ES;
    const int* thin_cols = reinterpret_cast<const int*>(p.tables + mt.thin_cols);
    const int sub = lane / CPR, part = lane % CPR;
    for (int r0 = 0; r0 < 32; r0 += G) {
      const unsigned these = todo >> r0 & (unsigned)((1ull << G) - 1);
      if (!these) continue;   // (uniform)
      if (these >> sub & 1) {
        const int r = r0 + sub, row = row0 + r, nd = TAKE ? ends[rb] : list[0], nt = thin_count(row), first = thin_of[row].x & ~kMaEntries;
        const u32x4 qv = *reinterpret_cast<const u32x4*>(q + ((size_t)row * CPR + part) * 16);
        auto entries = [&](auto each) {   // (the same for the CPR lanes of a row)
          for (int i = 0; i < nd; ++i) {
            unsigned long long word = *reinterpret_cast<const unsigned long long*>(bits + ((size_t)i * kMaRows + r) * 8);
            const int c0 = (list[1 + i] & 0xffff) * kMaCols;
            for (; word; word &= word - 1) each(c0 + __ffsll((long long)word) - 1);
          }
          for (int i = 0; i < nt; ++i) each(thin_cols[first + i]);
        };
        auto score = [&](int c) { return sa_row_dot<TYPE, CPR>(qv, *reinterpret_cast<const u32x4*>(k + ((size_t)c * CPR + part) * 16)); };
        float m = -INFINITY, total = 0.f, acc[E];
#pragma unroll
        for (int e = 0; e < E; ++e) acc[e] = 0.f;
        entries([&](int c) { m = fmaxf(m, score(c)); });
        entries([&](int c) {
          const float w = __builtin_amdgcn_exp2f((score(c) - m) * p.scale_log2);
          total += w;
          sa_add_row<TYPE>(acc, w, *reinterpret_cast<const u32x4*>(v + ((size_t)c * CPR + part) * 16));
        });
#pragma unroll
        for (int e = 0; e < E; e += 4) *reinterpret_cast<f32x4*>(rows + r * TLD + part * E + e) = f32x4{acc[e], acc[e + 1], acc[e + 2], acc[e + 3]};
        if (part == 0) state[r * 2 + 1] = total;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (todo >> col & 1) {
      sum = state[col * 2 + 1];
#pragma unroll
      for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 x = *reinterpret_cast<const f32x4*>(rows + col * TLD + d * 32 + g * 8 + half * 4);
#pragma unroll
          for (int e = 0; e < 4; ++e) o[d][g * 4 + e] = x[e];
        }
    }
  }

  const float inv = sum != 0.f ? 1.f / sum : 0.f;   // (a row without entries: zeros)
  if (query < T) {
    unsigned char* to = static_cast<unsigned char*>(p.out) + at + (size_t)query * HD * ES;
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float x0 = o[d][g * 4] * inv, x1 = o[d][g * 4 + 1] * inv, x2 = o[d][g * 4 + 2] * inv, x3 = o[d][g * 4 + 3] * inv;
        unsigned char* there = to + (d * 32 + g * 8 + half * 4) * ES;
        if constexpr (F32) *reinterpret_cast<f32x4*>(there) = f32x4{x0, x1, x2, x3};
        else *reinterpret_cast<u32x2*>(there) = u32x2{pack_pair<TYPE == 1>(x0, x1), pack_pair<TYPE == 1>(x2, x3)};
      }
  }
}

}  // namespace iex
