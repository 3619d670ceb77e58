// Walks, on the host, every 16-byte chunk that the direct-load GEMM tiles ask for (the same functions that the device code
// calls) and reports the first one that
//   * lies inside its buffer and outside the operand's allocation -- a read the hardware would perform --, or
//   * holds k < K of an existing row or column and does not come whole from where that element lies.
// A buffer load performs the 4-byte words that end inside the buffer (scalar offset included) and delivers zeros for others.
//   gemm_addresses_check M N K lda ldb layout(0 = B (K,N), 1 = B (N,K), 2 = A (K,M)) kb split(0 = none, -2 = halves, -3 = operands in three planes, n = parts) [1: sizes as rows * stride]
#include <algorithm>
#include <cstdio>
#include <cstdlib>

#include "../intrasm_engine_amd/csrc/gemm_addresses.h"

using namespace iex;
typedef long long ll;

static bool sizes_from_strides = false;
static ll checked = 0;

// One operand of one tile.  base: elements from the allocation's start to the buffer's; extent: elements of the allocation.
struct Walk {
  const char* what;
  ll base, extent;
  ll bytes;              // of the buffer
  bool rows_along_k;     // element (row, k) at row * ld + k, else (k, column) at k * ld + column
  int first, count;      // the tile's first row or column, and how many exist
  int K, ld, step_k;     // of this part; k per step
  ll k_base;             // of the part's first k, in elements from the allocation's start (of row / column 0)
  ll plane = 0;          // elements before the plane that is read (an operand in three planes)

  int chunk(DirectChunk c, int step, int lds_row, int lds_pos_first) const {
    const ll soffset = plane * 2 + (rows_along_k ? (ll)step * step_k * 2 : (ll)step * step_k * ld * 2);
    const int k = step * step_k + c.k;
    const bool wanted = k < K && (rows_along_k ? first + lds_row < count : lds_pos_first < count);
    int words = 0;
    for (int w = 0; w < 4; ++w) {
      const ll from = c.offset + w * 4;
      if (from + 4 > bytes - soffset) continue;
      ++words;
      const ll last = (base * 2 + soffset + from + 4 + 1) / 2;   // elements needed of the allocation
      if (last > extent) {
        std::printf("%s: step %d reads up to element %lld of %lld\n", what, step, last, extent);
        return 1;
      }
    }
    ++checked;
    if (!wanted) return 0;
    const ll at = base + (soffset + c.offset) / 2;
    const ll want = plane + (rows_along_k ? (ll)(first + lds_row) * ld + k_base + k : k_base + (ll)k * ld + lds_pos_first);
    if (words != 4 || at != want) {
      std::printf("%s: step %d, row or column %d, k %d: element %lld (%d words) instead of %lld\n", what, step, rows_along_k ? first + lds_row : lds_pos_first, k,
                  at, words, want);
      return 1;
    }
    return 0;
  }
};

template <int STAGE_K, int ROWS>
static int walk_rows(const Walk& w) {
  for (int step = 0; step * STAGE_K < w.K; ++step)
    for (int instr = 0; instr < ROWS * STAGE_K * 2 / 1024; ++instr)
      for (int lane = 0; lane < 64; ++lane)
        if (w.chunk(row_chunk<STAGE_K>(instr, lane, w.count - w.first, w.ld), step, instr * (512 / STAGE_K) + lane / (STAGE_K / 8), 0)) return 1;
  return 0;
}

template <int COLS, int STAGE_K>
static int walk_columns(const Walk& w) {
  for (int step = 0; step * STAGE_K < w.K; ++step)
    for (int instr = 0; instr < COLS * STAGE_K * 2 / 1024; ++instr)
      for (int lane = 0; lane < 64; ++lane) {
        const DirectChunk c = column_chunk<COLS>(instr, lane, w.first, w.ld);
        if (w.chunk(c, step, 0, w.first + ((lane % (COLS / 8)) ^ kn16_swizzle<COLS>(c.k)) * 8)) return 1;
      }
  return 0;
}

// A tile shape: BM x BN, A staged KA at a time, B KB at a time, K dealt out in steps of BK.
template <int BM, int BN, int KA, int KB, int BK>
static int walk(int M, int N, int K, int lda, int ldb, int layout, int kb, int split) {
  const int parts = split == -2 ? 2 : std::max(split, 1);
  const bool ta = layout == 2, tb = layout == 1;
  const ll a_extent = ta ? (ll)(K - 1) * lda + (M + 7) / 8 * 8 : (ll)(M - 1) * lda + K;
  const ll b_extent = tb ? (ll)(N - 1) * ldb + K : (ll)(kb - 1) * ldb + (N + 7) / 8 * 8;
  for (int part = 0; part < parts; ++part) {
    const KPart p = split == -2 ? k_in_halves(K, kb, BK, part) : k_in_parts(K, kb, BK, parts, part);
    if (p.K <= 0 || p.kb <= 0) {
      std::printf("part %d of %d is empty\n", part, parts);
      return 1;
    }
    auto size = [&](int rows, int width, int ld) { return sizes_from_strides ? (ll)rows * ld * 2 : (ll)rows_bytes(rows, width, ld); };
    for (int m0 = 0; m0 < M; m0 += BM) {
      Walk w{"A", ta ? (ll)p.k0 * lda : (ll)p.k0 + (ll)m0 * lda, a_extent, ta ? size(p.K, M, lda) : size(M - m0, p.K, lda), !ta, m0, M, p.K, lda, KA,
             ta ? (ll)p.k0 * lda : (ll)p.k0};
      if (ta ? walk_columns<BM, KA>(w) : walk_rows<KA, BM>(w)) return 1;
    }
    for (int n0 = 0; n0 < N; n0 += BN) {
      Walk w{"B", tb ? (ll)p.k0 + (ll)n0 * ldb : (ll)p.k0 * ldb, b_extent, tb ? size(N - n0, p.K, ldb) : size(p.kb, N, ldb), tb, n0, N, tb ? p.K : p.kb, ldb, KB,
             tb ? (ll)p.k0 : (ll)p.k0 * ldb};
      if (tb ? walk_rows<KB, BN>(w) : walk_columns<BN, KB>(w)) return 1;
    }
  }
  return 0;
}

// The fp32 product by parts: 128 x 128 tiles, steps of 32 k, both operands in three planes; K a multiple of 32 (zeros where the operands end).
static int walk_planes(int M, int N, int K, int lda, int ldb, int layout) {
  const bool tb = layout == 1;
  const ll plane_a = (ll)M * lda, plane_b = (ll)(tb ? N : K) * ldb;
  for (int plane = 0; plane < 3; ++plane) {
    for (int m0 = 0; m0 < M; m0 += 128)
      if (walk_rows<32, 128>(Walk{"A", (ll)m0 * lda, 3 * plane_a, 4 * plane_a + (ll)rows_bytes(M - m0, K, lda), true, m0, M, K, lda, 32, 0, plane * plane_a})) return 1;
    for (int n0 = 0; n0 < N; n0 += 128) {
      const Walk w{"B", tb ? (ll)n0 * ldb : 0, 3 * plane_b, 4 * plane_b + (ll)(tb ? rows_bytes(N - n0, K, ldb) : rows_bytes(K, N, ldb)), tb, n0, N, K, ldb, 32, 0, plane * plane_b};
      if (tb ? walk_rows<32, 128>(w) : walk_columns<128, 32>(w)) return 1;
    }
  }
  return 0;
}

int main(int argc, char** argv) {
  if (argc < 9) return 2;
  int v[8];
  for (int i = 0; i < 8; ++i) v[i] = std::atoi(argv[1 + i]);
  sizes_from_strides = argc > 9 && std::atoi(argv[9]);
  const int M = v[0], N = v[1], K = v[2], lda = v[3], ldb = v[4], layout = v[5], kb = v[6], split = v[7];
  int bad = 0;
  if (split == -3) bad = walk_planes(M, N, K, lda, ldb, layout);                                       // fp32 by parts
  else if (split > 0) bad = walk<64, 128, 64, 64, 64>(M, N, K, lda, ldb, layout, kb, split);              // K in parts
  else if (split == -2) bad = walk<256, 256, 32, 32, 32>(M, N, K, lda, ldb, layout, kb, split);      // K in halves
  else
    bad = walk<128, 128, 32, 32, 32>(M, N, K, lda, ldb, layout, kb, 0) || walk<64, 128, 64, 64, 64>(M, N, K, lda, ldb, layout, kb, 0) ||
          walk<256, 256, 64, 32, 32>(M, N, K, lda, ldb, layout, kb, 0) || walk<128, 256, 64, 64, 64>(M, N, K, lda, ldb, layout, kb, 0) ||
          (layout != 2 && walk<192, 256, 64, 32, 32>(M, N, K, lda, ldb, layout, kb, 0));
  if (!bad) std::printf("%lld chunks\n", checked);
  return bad;
}
