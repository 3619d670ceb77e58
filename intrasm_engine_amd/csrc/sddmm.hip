// CSR SDDMM for gfx950 (wave64): out[j] = <lhs[row(j), :], rhs[col(j), :]>.
//
// Work decomposition
//   * a wavefront owns one CSR row (swizzled order) or, for long rows, every WPR-th
//     chunk of 64 nonzeros of it; outputs are independent, so no reduction crosses
//     wavefronts and nothing is atomic;
//   * a group of LPN adjacent lanes handles one nonzero: the LPN lanes read one rhs row
//     as a single contiguous LPN*VEC*sizeof(T) segment (128-bit per lane when the shape
//     allows), so G = 64/LPN nonzeros are in flight per instruction;
//   * the lhs row fragment that a lane needs is the same for every nonzero of the row
//     and is held in registers when k <= 2*LPN*VEC (the attention shapes); otherwise it
//     is re-read (it hits L1: every group reads the same bytes);
//   * column indices are read 64 at a time (one per lane, the next 64 prefetched) and a
//     full chunk issues all its gathers before the first reduction;
//   * the LPN partial dot products are summed with DPP row operations (quad_perm,
//     row_half_mirror, row_mirror): no LDS, no bpermute in the reduction.
// Accumulation is fp32; with SUM_OVER_BATCH the batch loop runs inside the kernel so
// the (nnz) output is a deterministic sum.
#include <algorithm>
#include <cmath>
#include "gemm_split.h"
#include "iex_common.h"
#include "sddmm_mfma_device.cuh"
#include "spmm_dense_device.cuh"

namespace iex {
namespace {

struct SddmmParams {
  int m, k, n, nnz, batch;
  const int* row_indices;
  const int* row_offsets;
  const int* cols;
  const void* lhs;
  const void* rhs;
  void* out;
  int sum_over_batch, accumulate;
  int pad = 0;   // the dense product may copy operands into the workspace (IEX_SDDMM_PAD_OPERANDS)
};

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

template <typename T, int VEC>
__device__ __forceinline__ float dot_vec(const vec_t<T, VEC>& a, const vec_t<T, VEC>& b, float acc) {
  if constexpr (sizeof(T) == 2 && VEC >= 2 && __is_same(T, __half)) {
#pragma unroll
    for (int i = 0; i < VEC / 2; ++i) {
      f16x2 x = __builtin_bit_cast(f16x2, *reinterpret_cast<const uint32_t*>(&a.v[2 * i]));
      f16x2 y = __builtin_bit_cast(f16x2, *reinterpret_cast<const uint32_t*>(&b.v[2 * i]));
      acc = __builtin_amdgcn_fdot2(x, y, acc, false);
    }
    return acc;
  } else {
#pragma unroll
    for (int i = 0; i < VEC; ++i)
      acc = fmaf(elem<T>::to_float(a.v[i]), elem<T>::to_float(b.v[i]), acc);
    return acc;
  }
}

// VEC elements of a row of k from element kk on.  TAIL: the vector may reach past the row's end: the VEC elements that
// end there are read instead (k >= VEC, checked by the host) and `keep` clears those that are not kk .. kk + VEC - 1, in
// both operands (a zero in one alone would turn an infinity of the other into a NaN).
template <typename T, int VEC>
struct tail_mask {
  static constexpr int kWords = (int)sizeof(T) * VEC / 4;
  uint32_t keep[kWords > 0 ? kWords : 1];
  __device__ __forceinline__ explicit tail_mask(int valid) {   // the last `valid` elements of the vector stay
    constexpr int per_word = 4 / (int)sizeof(T);
#pragma unroll
    for (int w = 0; w < kWords; ++w) {
      const int dead = VEC - valid - w * per_word;   // elements of this word to clear
      keep[w] = dead <= 0 ? 0xffffffffu : dead >= per_word ? 0u : 0xffff0000u;
    }
  }
  __device__ __forceinline__ void apply(vec_t<T, VEC>& v) const {
    uint32_t* w = reinterpret_cast<uint32_t*>(&v);
#pragma unroll
    for (int i = 0; i < kWords; ++i) w[i] &= keep[i];
  }
};

// PASSES > 0: k <= PASSES*LPN*VEC (EXACT: k equals it, so no load needs a predicate): the lhs
//             fragment of a (row, batch entry) is one register load per pass; a chunk of 64
//             nonzeros takes LPN steps of G nonzeros: all column indices are shuffled out and
//             all gathers issued first, then step s reduces and leaves its result in lane s of
//             every group, so each lane ends up with exactly one output (nonzero lane%LPN*G +
//             lane/LPN) and the chunk is written with ONE store instruction that covers 64
//             consecutive outputs.  Plain stores only (no accumulate mode).
// PASSES == 0: generic k, accumulate mode and sums over a batch: operands streamed in LPN*VEC slices, a slice of lhs
//             serving kSddmmSteps nonzeros per lane group at a time, two slices in flight.
// RAGGED: k is no multiple of VEC (or the operands are not aligned to it): vectors at element alignment, the one past
//         the row's end masked.  (By single elements: 631 x 3656 at 96 %, k = 1189, fp16 267 us.)
// A block serves kSddmmZb batch entries (grid.z = ceil(batch / kSddmmZb)) in per-entry output
// mode, so the row's column indices are fetched once and reused.
constexpr int kSddmmZb = 4;
constexpr int kSddmmSteps = 4;

template <typename T, int VEC, int LPN, int PASSES, int WPR, bool EXACT, bool RAGGED>
__global__ __launch_bounds__(256) void sddmm_kernel(SddmmParams p) {
  constexpr int G = kWave / LPN;
  constexpr int KT = LPN * VEC;
  constexpr int kRowsPerBlock = 4 / WPR;
  // k below PASSES * KT: a predicate on each load, or loads that all lanes do.  In bf16, whose products widen both operands, the predicated loads' registers
  // spill (us, predicates / without: 9709 x 632 at 86 %, k = 184 256 / 56; 4000 x 2000 at 95 %, k = 200 109 / 27; 10773 x 1185 at 95.5 %, k = 136 75 / 25); fp16
  // and fp32 are as fast or faster with them (k = 96 13.5 / 15.5, 200 20.7 / 21.9; fp32 1200 x 3434, k = 44 11.4 / 13.6).
  constexpr bool CLAMP = RAGGED || (!EXACT && VEC > 1 && __is_same(T, __hip_bfloat16));
  const int lane = lane_id();
  const int wave = uniform(threadIdx.x >> 6);
  const int sub = lane / LPN;
  const int sl = lane % LPN;
  const int row_slot = blockIdx.x * kRowsPerBlock + wave / WPR;
  const int part = wave % WPR;
  if (row_slot >= p.m) return;

  const int row = uniform(p.row_indices[row_slot]);
  const int start = uniform(p.row_offsets[row]);
  const int end = uniform(p.row_offsets[row + 1]);
  // per-entry output: this block's slice of the batch; batch-summed output: one pass that
  // loops over the whole batch inside the dot product
  const int zbeg = p.sum_over_batch ? 0 : (int)blockIdx.z * kSddmmZb;
  const int zend = p.sum_over_batch ? 1 : min(p.batch, zbeg + kSddmmZb);
  const int zn = p.sum_over_batch ? p.batch : 1;
  const size_t lhs_zstride = (size_t)p.m * p.k;
  const size_t rhs_zstride = (size_t)p.n * p.k;
  const T* __restrict__ lhs_row = static_cast<const T*>(p.lhs) + (size_t)row * p.k;
  const T* __restrict__ rhs_all = static_cast<const T*>(p.rhs);
  T* __restrict__ out_all = static_cast<T*>(p.out);

  // column index of nonzero base+lane; the next chunk's indices are fetched while the
  // current chunk is processed
  int base = start + part * kWave;
  int c = (base + lane < end) ? p.cols[base + lane] : 0;
  for (; base < end; base += kWave * WPR) {
    const int next = base + kWave * WPR;
    const int c_next = (next + lane < end) ? p.cols[next + lane] : 0;
    const int cnt = min(kWave, end - base);
    if constexpr (PASSES > 0) {
      // slots past cnt carry column 0: they gather a valid row and their result is dropped
      int cc[LPN];
#pragma unroll
      for (int st = 0; st < LPN; ++st) cc[st] = __shfl(c, st * G + sub, kWave);
      const int my_t = sl * G + sub;  // the nonzero whose result this lane will hold
      for (int z = zbeg; z < zend; ++z) {
        const T* __restrict__ lhs = lhs_row + (size_t)z * lhs_zstride;
        const T* __restrict__ rhs = rhs_all + (size_t)z * rhs_zstride;
        vec_t<T, VEC> lfrag[PASSES];
        vec_t<T, VEC> rv[LPN][PASSES];
        // (CLAMP: every lane reads a vector, and what the last pass reads past the row's end is cleared)
        const int last_kk = (PASSES - 1) * KT + sl * VEC;
        const tail_mask<T, VEC> mask(CLAMP ? min(max(p.k - last_kk, 0), VEC) : VEC);
        auto at = [&](int ps) { return CLAMP ? min(ps * KT + sl * VEC, p.k - VEC) : ps * KT + sl * VEC; };
#pragma unroll
        for (int ps = 0; ps < PASSES; ++ps) {
          if (EXACT || CLAMP || at(ps) < p.k) lfrag[ps] = load_vec<T, VEC, !RAGGED>(lhs + at(ps));
        }
        if constexpr (CLAMP) mask.apply(lfrag[PASSES - 1]);
#pragma unroll
        for (int st = 0; st < LPN; ++st) {
          const T* r = rhs + (size_t)cc[st] * p.k;
#pragma unroll
          for (int ps = 0; ps < PASSES; ++ps) {
            if (EXACT || CLAMP || at(ps) < p.k) rv[st][ps] = load_vec<T, VEC, !RAGGED>(r + at(ps));
          }
        }
        float res = 0.f;
#pragma unroll
        for (int st = 0; st < LPN; ++st) {
          float acc = 0.f;
#pragma unroll
          for (int ps = 0; ps < PASSES; ++ps) {
            if constexpr (CLAMP) {
              if (ps == PASSES - 1) mask.apply(rv[st][ps]);
            }
            if (EXACT || CLAMP || at(ps) < p.k) acc = dot_vec<T, VEC>(lfrag[ps], rv[st][ps], acc);
          }
          acc = group_sum<LPN>(acc);
          res = (sl == st) ? acc : res;
        }
        if (my_t < cnt) out_all[(p.sum_over_batch ? (size_t)0 : (size_t)z * p.nnz) + base + my_t] = elem<T>::from_float(res);
      }
    } else {
      for (int z = zbeg; z < zend; ++z) {
        const T* __restrict__ lhs = lhs_row + (size_t)z * lhs_zstride;
        const T* __restrict__ rhs = rhs_all + (size_t)z * rhs_zstride;
        T* __restrict__ out = out_all + (p.sum_over_batch ? (size_t)0 : (size_t)z * p.nnz);
        const int steps = (cnt + G - 1) / G;
        for (int st = 0; st < steps; st += kSddmmSteps) {
          // nonzero st * G + u * G + sub of this chunk is the u-th of my lane group; slots past cnt carry column 0
          int t[kSddmmSteps];
          const T* row_of[kSddmmSteps];
          float acc[kSddmmSteps];
#pragma unroll
          for (int u = 0; u < kSddmmSteps; ++u) {
            t[u] = (st + u) * G + sub;
            row_of[u] = rhs + (size_t)__shfl(c, t[u] & (kWave - 1), kWave) * p.k;
            acc[u] = 0.f;
          }
          for (int zz = 0; zz < zn; ++zz) {
            const T* l = lhs + (size_t)zz * lhs_zstride;
            const size_t zoff = (size_t)zz * rhs_zstride;
            int kk = sl * VEC;
            // two slices of lhs and of every nonzero's rhs row in flight: the chain load -> multiply -> load is what a
            // launch with few wavefronts waits for, and a slice of lhs is read once for kSddmmSteps nonzeros
            for (; kk + KT + VEC <= p.k; kk += 2 * KT) {
              vec_t<T, VEC> lv[2], rv[2][kSddmmSteps];
#pragma unroll
              for (int h = 0; h < 2; ++h) {
                lv[h] = load_vec<T, VEC, !RAGGED>(l + kk + h * KT);
#pragma unroll
                for (int u = 0; u < kSddmmSteps; ++u) rv[h][u] = load_vec<T, VEC, !RAGGED>(row_of[u] + zoff + kk + h * KT);
              }
#pragma unroll
              for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int u = 0; u < kSddmmSteps; ++u) acc[u] = dot_vec<T, VEC>(lv[h], rv[h][u], acc[u]);
            }
            for (; kk < p.k; kk += KT) {
              const int from = RAGGED ? min(kk, p.k - VEC) : kk;
              const tail_mask<T, VEC> mask(RAGGED ? min(p.k - kk, VEC) : VEC);
              vec_t<T, VEC> lv = load_vec<T, VEC, !RAGGED>(l + from), rv[kSddmmSteps];
#pragma unroll
              for (int u = 0; u < kSddmmSteps; ++u) rv[u] = load_vec<T, VEC, !RAGGED>(row_of[u] + zoff + from);
              if constexpr (RAGGED) mask.apply(lv);
#pragma unroll
              for (int u = 0; u < kSddmmSteps; ++u) {
                if constexpr (RAGGED) mask.apply(rv[u]);
                acc[u] = dot_vec<T, VEC>(lv, rv[u], acc[u]);
              }
            }
          }
#pragma unroll
          for (int u = 0; u < kSddmmSteps; ++u) {
            acc[u] = group_sum<LPN>(acc[u]);
            if (sl == 0 && t[u] < cnt) {
              const size_t o = (size_t)base + t[u];
              if (p.accumulate) acc[u] += elem<T>::to_float(out[o]);
              out[o] = elem<T>::from_float(acc[u]);
            }
          }
        }
      }
    }
    c = c_next;
  }
}

template <typename T, int VEC, int LPN, int PASSES, int WPR, bool EXACT, bool RAGGED>
int launch_one(const SddmmParams& p, hipStream_t stream) {
  dim3 grid(ceil_div(p.m, 4 / WPR), 1, p.sum_over_batch ? 1 : ceil_div(p.batch, kSddmmZb));
  note_kernel("sddmm_kernel<%s, %d, %d, %d, %d, %s, %s>", type_name<T>(), VEC, LPN, PASSES, WPR, EXACT ? "true" : "false", RAGGED ? "true" : "false");
  hipLaunchKernelGGL((sddmm_kernel<T, VEC, LPN, PASSES, WPR, EXACT, RAGGED>), grid, dim3(256), 0, stream, p);
  return check_hip(hipGetLastError(), "sddmm launch");
}

template <typename T, int VEC, int LPN, int PASSES, bool EXACT, bool RAGGED>
int launch_wpr(const SddmmParams& p, int wpr, hipStream_t stream) {
  if (wpr == 4) return launch_one<T, VEC, LPN, PASSES, 4, EXACT, RAGGED>(p, stream);
  return launch_one<T, VEC, LPN, PASSES, 1, EXACT, RAGGED>(p, stream);
}

template <typename T, int VEC, int LPN, bool RAGGED>
int launch_passes(const SddmmParams& p, int wpr, hipStream_t stream) {
  // register-resident lhs needs one batch entry per dot product and plain stores
  const bool fast = !(p.sum_over_batch && p.batch > 1) && !p.accumulate;
  constexpr int kt = LPN * VEC;
  if constexpr (!RAGGED) {
    if (fast && p.k == kt) return launch_wpr<T, VEC, LPN, 1, true, RAGGED>(p, wpr, stream);
    if (fast && p.k == 2 * kt) return launch_wpr<T, VEC, LPN, 2, true, RAGGED>(p, wpr, stream);
  }
  if (fast && p.k <= kt) return launch_wpr<T, VEC, LPN, 1, false, RAGGED>(p, wpr, stream);
  if (fast && p.k <= 2 * kt) return launch_wpr<T, VEC, LPN, 2, false, RAGGED>(p, wpr, stream);
  return launch_wpr<T, VEC, LPN, 0, false, RAGGED>(p, wpr, stream);
}

template <typename T>
int launch_typed(const SddmmParams& p, int wpr, hipStream_t stream) {
  constexpr int kMax = 16 / (int)sizeof(T);
  if (p.k < kMax) return launch_passes<T, 1, 16, false>(p, wpr, stream);   // (no whole vector in a row)
  // lanes per nonzero: enough to cover k in one or two passes, at most 16 (one DPP row)
  const bool ragged = p.k % kMax != 0 || !aligned(p.lhs, 16) || !aligned(p.rhs, 16);
  if (p.k <= 8 * kMax) return ragged ? launch_passes<T, kMax, 8, true>(p, wpr, stream) : launch_passes<T, kMax, 8, false>(p, wpr, stream);
  return ragged ? launch_passes<T, kMax, 16, true>(p, wpr, stream) : launch_passes<T, kMax, 16, false>(p, wpr, stream);
}

// ---- dense product, then sampling (16-bit types, caller's workspace of m * n * 2 bytes) ----
// A long k makes the gather kernel read k * 2 bytes of rhs per nonzero through the L2 -> CU path;
// the dense GEMM computes all m * n dot products on the matrix cores in less time than that takes
// once the mask is not very sparse, and a small kernel then picks the nonzeros' entries.
// Same arithmetic per output (fp32 accumulation over k, one rounding to the 16-bit type).
// WIDE: a workgroup per row instead of a wavefront (rows of hundreds of nonzeros: their chain of steps is what few rows wait for).
template <bool WIDE>
__global__ __launch_bounds__(256) void sample_dense_kernel(int m, int ld, const int* __restrict__ row_offsets,
                                                           const int* __restrict__ cols,
                                                           const uint16_t* __restrict__ dense,
                                                           uint16_t* __restrict__ out) {
  const int row = WIDE ? (int)blockIdx.x : (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6);
  if (row >= m) return;
  const int start = row_offsets[row], end = row_offsets[row + 1];
  const uint16_t* drow = dense + (size_t)row * ld;
  for (int j = start + (WIDE ? (int)threadIdx.x : lane_id()); j < end; j += WIDE ? 256 : kWave) out[j] = drow[cols[j]];
}

// us of the whole product, a wavefront / a workgroup per row: 1128 x 10508 at 81 %, k = 248 45 / 33; 424 x 9043 at 88 %, k = 685 41 / 34; 696 x 2192 at 88 %, k = 248 11.8 / 10.4;
// 4680 x 2144 at 88 %, k = 112 21.8 / 22.7
inline bool sample_wide(const SddmmParams& p) { return p.nnz >= (p.m <= 2048 ? 128ll : 256ll) * p.m; }

inline bool sddmm_dense_fits(int dtype, const SddmmParams& p) {
  return (dtype == IEX_F16 || dtype == IEX_BF16) && !p.accumulate && !(p.sum_over_batch && p.batch > 1) && p.k > 0 &&
         (p.pad || (p.k % 8 == 0 && p.n % 8 == 0 && aligned(p.lhs, 16) && aligned(p.rhs, 16))) && (long long)p.m * round8(p.n) < (1ll << 31) &&
         (long long)std::max(p.m, p.n) * round8(p.k) < (1ll << 31);
}

// The workspace: the product (rows of round8(n)), then copies of lhs and rhs where k or their addresses are no whole vectors.
inline bool sddmm_dense_pads(const SddmmParams& p) { return p.k % 8 != 0 || !aligned(p.lhs, 16) || !aligned(p.rhs, 16); }
inline size_t sddmm_dense_lhs_offset(const SddmmParams& p) { return round256((size_t)p.m * round8(p.n) * 2); }
inline size_t sddmm_dense_rhs_offset(const SddmmParams& p) { return round256(sddmm_dense_lhs_offset(p) + (size_t)p.m * round8(p.k) * 2); }
inline size_t sddmm_dense_bytes(const SddmmParams& p) {
  return sddmm_dense_pads(p) ? sddmm_dense_rhs_offset(p) + (size_t)p.n * round8(p.k) * 2 : (size_t)p.m * round8(p.n) * 2;
}

// Time model fitted on MI355X (fp16).  Dense product per batch entry: two launches, the GEMM at
// 1000 TFLOP/s or, with few tiles, 0.23 us per K step of 32 per round of 512 tiles of 128 x 128,
// m * n * 2 bytes written and nnz entries picked at 4 TB/s, two more launches where the operands are copied.  Gather kernel: nnz * k * 2 bytes at
// 14 TB/s, at 9 (13 in registers) or 7 where rows start at odd multiples of 4 or 2 bytes, and half of that for k of a few dozen; with a k beyond the register-resident
// fragments no less than one wave's chain of
// loads (0.12 us per 128 elements of k and step of 4 nonzeros with four slices in flight:
// 1024 x 1024 at 95 %, k = 4096: 50 us).  Us, gather / dense product: 11008 x 4096 at 80 %, k = 8192 (weight gradient of an MLP
// projection) 16500 / 770; 4096 x 4096 at 90 %, k = 512 120 / 55; at either side of the line 1056 x 3184 at 80 %, k = 152 22.5 / 12.7; 1168 x 1248 at 81 %, k = 192 11.7 / 9.5;
// 534 x 3173 at 88 %, k = 104 7.9 / 12.1; 696 x 2192 at 88 %, k = 248 10.8 / 10.4; 3304 x 494 at 90 %, k = 563 30 / 19; 1120 x 2184 at 80 %, k = 241 27 / 18; 422 x 2632 at 95 %, k = 667 16 / 20;
// 958 x 2305 at 95 %, k = 438 12 / 23; 1529 x 6000 at 92 %, k = 242 27 / 33; 5472 x 7472 at 81 %, k = 23 109 / 47; 5043 x 4044 at 80 %, k = 26 30 / 40.  The dense product has to win by 15 %.
inline bool sddmm_dense_wins(const SddmmParams& p) {
  const double flops = 2.0 * p.m * p.n * p.k;
  const double tiles = (double)ceil_div(p.m, 128) * ceil_div(p.n, 128);
  const double product = std::max(flops / 1000e12, std::ceil(tiles / 512.0) * (p.k / 32.0) * 0.23e-6);
  const double pad = sddmm_dense_pads(p) ? 7e-6 + 4.0 * ((double)p.m + p.n) * p.k / 4e12 : 0.0;
  const double row_nnz = (double)p.nnz / p.m;
  const double sample = (p.nnz * 8.0) / 4e12 + row_nnz / (sample_wide(p) ? 256 : 64) * 0.35e-6;
  const double dense = p.batch * (8.5e-6 + pad + product + (double)p.m * p.n * 2 / 4e12 + sample);
  const double chain = p.k > 256 ? std::ceil(row_nnz / (row_nnz >= 64.0 ? 16.0 : 4.0)) * (p.k / 128.0) * 0.12e-6 : 0.0;
  const double rate = p.k % 4 == 0 ? 14e12 : p.k % 2 == 0 ? (p.k >= 64 && p.k <= 256 ? 13e12 : 9e12) : p.k < 64 ? 4e12 : 7e12;
  const double gather = std::max(4e-6 + (double)p.batch * p.nnz * p.k * 2 / rate, chain);
  return 1.15 * dense < gather;
}

int launch_sddmm_dense(int dtype, const SddmmParams& p, void* ws, hipStream_t stream) {
  const int kp = round8(p.k), ld = round8(p.n);
  unsigned char* at = static_cast<unsigned char*>(ws);
  for (int z = 0; z < p.batch; ++z) {
    const void* lhs = static_cast<const uint16_t*>(p.lhs) + (size_t)z * p.m * p.k;
    const void* rhs = static_cast<const uint16_t*>(p.rhs) + (size_t)z * p.n * p.k;
    if (sddmm_dense_pads(p)) {
      void *lhs_copy = at + sddmm_dense_lhs_offset(p), *rhs_copy = at + sddmm_dense_rhs_offset(p);
      if (int rc = launch_pad_rows(p.m, p.k, lhs, p.m, kp, lhs_copy, 1, 0, stream)) return rc;
      if (int rc = launch_pad_rows(p.n, p.k, rhs, p.n, kp, rhs_copy, 1, 0, stream)) return rc;
      lhs = lhs_copy;
      rhs = rhs_copy;
    }
    // (the dispatcher, not the public entry point: that one starts a new trail of kernel names)
    GemmParams g{p.m, p.n, kp, lhs, rhs, ws, 0, 0, 0, 0, 0};
    g.ldc = ld;
    if (int rc = gemm_dispatch(dtype, 1, g, 1, stream)) return rc;
    note_kernel("sample_dense_kernel");
    uint16_t* out = static_cast<uint16_t*>(p.out) + (size_t)z * p.nnz;
    if (sample_wide(p)) hipLaunchKernelGGL(sample_dense_kernel<true>, dim3(p.m), dim3(256), 0, stream, p.m, ld, p.row_offsets, p.cols, static_cast<const uint16_t*>(ws), out);
    else hipLaunchKernelGGL(sample_dense_kernel<false>, dim3(ceil_div(p.m, 4)), dim3(256), 0, stream, p.m, ld, p.row_offsets, p.cols, static_cast<const uint16_t*>(ws), out);
    if (int rc = check_hip(hipGetLastError(), "sddmm sampling launch")) return rc;
  }
  return 0;
}

// ---- fp32: the dense product by three bf16 parts of every entry (gemm_split_device.cuh), then sampling ----
// A sum over the batch is one product with the batch's k side by side.
struct SddmmSplit {
  int kp, K, ld, parts;   // k rounded up, of all batch entries; rows of scores; parts of K
  size_t lhs_at, rhs_at, scores_at, bytes;
};
inline SddmmSplit sddmm_split_plan(const SddmmParams& p) {
  SddmmSplit s;
  s.kp = round32(p.k);
  s.K = s.kp * p.batch;
  s.ld = (p.n + 3) & ~3;
  s.parts = gemm_split_parts(p.m, p.n, s.K, 1);
  s.lhs_at = kSplitRanges * 4;
  s.rhs_at = s.lhs_at + round256((size_t)p.m * s.K * 6);
  s.scores_at = s.rhs_at + round256((size_t)p.n * s.K * 6);
  s.bytes = s.scores_at + (size_t)s.parts * p.m * s.ld * 4;
  return s;
}
// (copies of the operands, which are the caller's to allow; planes within a buffer's 4 GB)
inline bool sddmm_split_fits(int dtype, const SddmmParams& p) {
  return dtype == IEX_F32 && p.pad && !p.accumulate && (p.sum_over_batch || p.batch == 1) && p.k > 0 && p.n > 0 &&
         (long long)std::max(p.m, p.n) * round32(p.k) * p.batch < (1ll << 32) / 6 && (long long)p.m * p.n < (1ll << 30);
}
// Time model fitted on MI355X: three launches, the planes' bytes at 4.4 TB/s, the product (gemm_split_seconds), the scores of all parts written and read
// once at 4 TB/s; the gather kernel at 18 TB/s, 13.5 where rhs outgrows an XCD's L2.  Us, gather kernel / this way, at either side of
// the line: 2160 x 1449, k = 221, 81 % 43 / 36; 3711 x 1112, k = 296, 86 % 38 / 52; 10680 x 3436, k = 179, 89 % 143 / 167; 8463 x 3904, k = 252, 88 % 229 / 191;
// 4296 x 1093, k = 997, 95 % 73 / 102; 5176 x 1344, k = 1197, 86 % 305 / 127; 1560 x 2069, k = 1517, 97 % 52 / 83; 986 x 10230, k = 1049, 85 % 603 / 176.
inline bool sddmm_split_wins(const SddmmParams& p) {
  const double bytes = (double)p.nnz * p.k * p.batch * 4, gather = 4e-6 + bytes / ((double)p.n * p.k * 4 <= 4.5e6 ? 18e12 : 13.5e12);
  if (gather < 28e-6) return false;   // (what three launches and a short product take)
  const SddmmSplit s = sddmm_split_plan(p);
  const double sample = 4.5e-6 + (4.0 * s.parts * p.m * s.ld + 8.0 * p.nnz) / 4e12;
  return 1.1 * (3.5e-6 + 10.0 * ((double)p.m + p.n) * s.K / 4.4e12 + gemm_split_seconds(p.m, p.n, s.K, 1) + sample) < gather;
}
// What a call that goes this way wants of workspace; 0: it does not.
inline size_t sddmm_split_bytes(int dtype, const SddmmParams& p, bool forced) {
  if (!sddmm_split_fits(dtype, p) || (!forced && !sddmm_split_wins(p))) return 0;
  const size_t bytes = sddmm_split_plan(p).bytes;
  return bytes <= kSplitWorkspaceMost ? bytes : 0;
}
int launch_sddmm_split(const SddmmParams& p, void* workspace, hipStream_t stream) {
  const SddmmSplit s = sddmm_split_plan(p);
  unsigned char* ws = static_cast<unsigned char*>(workspace);
  unsigned* ranges = reinterpret_cast<unsigned*>(ws);
  const long long plane_a = (long long)p.m * s.K, plane_b = (long long)p.n * s.K;
  const SplitDense a{p.batch, p.m, p.k, static_cast<const float*>(p.lhs), p.m, s.kp, s.K, s.kp, plane_a, ws + s.lhs_at};
  const SplitDense b{p.batch, p.n, p.k, static_cast<const float*>(p.rhs), p.n, s.kp, s.K, s.kp, plane_b, ws + s.rhs_at};
  if (int rc = launch_split_operands(a, b, ranges, stream)) return rc;
  SplitParams g{};
  g.M = p.m, g.N = p.n, g.K = s.K;
  g.A = a.dst, g.B = b.dst, g.C = reinterpret_cast<float*>(ws + s.scores_at);
  g.lda = g.ldb = s.K, g.ldc = s.ld;
  g.plane_a = (unsigned)(plane_a * 2), g.plane_b = (unsigned)(plane_b * 2);
  g.parts = s.parts, g.stride_part = (long long)p.m * s.ld;
  g.ranges = ranges, g.slots_a = split_dense_blocks(a), g.slots_b = split_dense_blocks(b);
  if (int rc = gemm_split(g, true, 1, stream)) return rc;
  const SplitSample q{p.m, p.k, p.n, p.batch, s.ld, s.parts, sample_wide(p), g.stride_part, p.row_offsets, p.cols, g.C, static_cast<const float*>(p.lhs), static_cast<const float*>(p.rhs),
                      static_cast<float*>(p.out), ranges};
  return launch_split_sample(q, stream);
}

// ---- score tiles on the matrix cores, sampled inside the workgroup (sddmm_mfma_device.cuh) ----
// 16-bit types, k = 32, 64 or 128, plain store, one output per batch entry, canonical CSR (columns ascending and
// distinct inside a row), n <= 128 * kSdMaxTiles; the workspace holds (6 ceil(n / 128) + 1) * m words (per row and
// column tile: a 128-bit mask, a cursor, a packed word).
inline bool sddmm_mfma_fits(int dtype, const SddmmParams& p) {
  return (dtype == IEX_F16 || dtype == IEX_BF16) && !p.accumulate && !(p.sum_over_batch && p.batch > 1) &&
         (p.k == 32 || p.k == 64 || p.k == 128) && aligned(p.lhs, 16) && aligned(p.rhs, 16) &&
         ceil_div(p.n, kSdBN) <= kSdMaxTiles && (long long)(ceil_div(p.n, kSdBN) + 1) * p.m < (1ll << 28);
}

inline size_t sddmm_mfma_bytes(const SddmmParams& p) { return sb_words(p.m, ceil_div(p.n, kSdBN), p.nnz) * sizeof(int); }

// The host does not look at the pattern, so the choice goes by the mask's overall density.  Measured on MI355X
// (fp16, 16 heads of 4096 x 4096, k = 64, microseconds, gather kernel / this kernel with its two setup kernels;
// bench.py, extras.sddmm_fp16_16heads_by_mask):
//   band of 256 + 32 scattered per row (7 %)  114 /  54      band of 512 + 32 (13 %)      213 /  70
//   band of 128 + 16 scattered (3.5 %)          73 /  45      block diagonal 256 (6 %)      98 /  34
//   causal window of 512 (12 %)                173 /  55
//   equal rows, columns at random:  1 %  29 (stays on the gather kernel)   5 %  89 / 100    10 %  155 / 177
//                                  20 % 287 / 175
// (a caller that keeps tables and lists saves 15 of these microseconds per call).  Masks with structure (what per-entry
// SDDMM is used for: attention) gain 1.6x to 3x from 3 % up; a mask without any loses 1.1x to 1.2x below 15 %.
// IEX_SDDMM_FORCE_VARIANT(1) keeps the gather kernel.
inline bool sddmm_mfma_wins(const SddmmParams& p) {
  const double density = (double)p.nnz / ((double)p.m * p.n);
  return density >= 0.03 && (double)p.batch * p.m * p.n >= 32.0 * 1024 * 1024;
}

template <bool BF16, int KS>
int launch_sddmm_mfma_ks(const SddmmMfmaParams& q, int batch, hipStream_t stream) {
  constexpr int lds = sddmm_mfma_lds_bytes<KS>();
  auto kernel = sddmm_mfma_kernel<BF16, KS>;
  static thread_local bool raised = false;   // per instantiation: more than 64 KB of dynamic LDS
  if (!raised) {
    if (int rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds),
                           "hipFuncSetAttribute(LDS size)"))
      return rc;
    raised = true;
  }
  note_kernel("sddmm_mfma_kernel<%s, %d>", BF16 ? "true" : "false", KS);
  hipLaunchKernelGGL(kernel, dim3(ceil_div(q.m, kSdBM), batch), dim3(kSdThreads), lds, stream, q);
  return check_hip(hipGetLastError(), "sddmm (matrix-core) launch");
}

// ready: bit 0 = the caller vouches that an earlier call on this pattern left the tables in the workspace, bit 1 = that the
// lists are there too, from a call with the same dense_code (this kernel's, or the SpMM's for such patterns: same lists).
int launch_sddmm_mfma(int dtype, const SddmmParams& p, void* ws, int dense_code, int ready, hipStream_t stream) {
  const int tiles_n = ceil_div(p.n, kSdBN);
  const SdTables t = sd_tables(ws, p.m, tiles_n);
  const SbLists l = sb_lists(ws, p.m, tiles_n, p.nnz);
  // dense_code (for tests and tuning): 0 = the built-in threshold, 1 = every tile on the matrix cores, 255 = none,
  // else 64 * code nonzeros per 128 x 128 block
  if (int rc = sb_setup(t, l, p.m, tiles_n, dense_code, ready, p.row_offsets, p.cols, stream)) return rc;
  SddmmMfmaParams q{p.m, p.k, p.n, p.nnz, p.cols, p.lhs, p.rhs, p.out, t.mask, t.tile_ptr, t.brief, tiles_n,
                    p.row_offsets, l.thin_ent, l.thin_cnt, l.dense_list};
  const bool bf16 = dtype == IEX_BF16;
  switch (p.k) {
    case 32: return bf16 ? launch_sddmm_mfma_ks<true, 2>(q, p.batch, stream) : launch_sddmm_mfma_ks<false, 2>(q, p.batch, stream);
    case 64: return bf16 ? launch_sddmm_mfma_ks<true, 4>(q, p.batch, stream) : launch_sddmm_mfma_ks<false, 4>(q, p.batch, stream);
    default: return bf16 ? launch_sddmm_mfma_ks<true, 8>(q, p.batch, stream) : launch_sddmm_mfma_ks<false, 8>(q, p.batch, stream);
  }
}

}  // namespace

// Bytes of workspace with which iex_sddmm_ws would compute the dense product and sample it (0: it
// would not, whatever the workspace).  Pointers are taken to be 16-byte aligned.
// What iex_sddmm_ws would do with a workspace of the size that sddmm_workspace_bytes names: 0 = not use it, 3 = keep the
// tables of the kernel for masks with structure in it, 7 = the dense product.
int sddmm_workspace_kind(int dtype, int flags, int m, int k, int n, int nonzeros, int batch) {
  if (m <= 0 || k <= 0 || n <= 0 || nonzeros <= 0 || batch <= 0) return 0;
  const int variant = (flags >> 16) & 0xf;
  if (variant != 0 && variant != 7 && variant != 3 && variant != 12) return 0;
  void* const some_aligned = reinterpret_cast<void*>(size_t(256));
  SddmmParams p{m, k, n, nonzeros, batch, nullptr, nullptr, nullptr, some_aligned, some_aligned, nullptr,
                (flags & IEX_SDDMM_SUM_OVER_BATCH) != 0, (flags & IEX_SDDMM_ACCUMULATE) != 0, (flags & IEX_SDDMM_PAD_OPERANDS) != 0};
  if (dtype == IEX_F32 && variant != 3 && variant != 7) return sddmm_split_bytes(dtype, p, variant == 12) ? 12 : 0;
  if (variant == 12) return 0;
  const bool any_order = (flags & IEX_SDDMM_ANY_COLUMN_ORDER) != 0;
  if (variant != 7 && sddmm_mfma_fits(dtype, p) && (variant == 3 || (!any_order && sddmm_mfma_wins(p)))) return 3;
  if (variant == 3 || !sddmm_dense_fits(dtype, p)) return 0;
  return (variant == 7 || sddmm_dense_wins(p)) ? 7 : 0;
}

size_t sddmm_workspace_bytes(int dtype, int flags, int m, int k, int n, int nonzeros, int batch) {
  if (m <= 0 || k <= 0 || n <= 0 || nonzeros <= 0 || batch <= 0) return 0;
  const int variant = (flags >> 16) & 0xf;
  if (variant != 0 && variant != 7 && variant != 3 && variant != 12) return 0;
  void* const some_aligned = reinterpret_cast<void*>(size_t(256));
  SddmmParams p{m, k, n, nonzeros, batch, nullptr, nullptr, nullptr, some_aligned, some_aligned, nullptr,
                (flags & IEX_SDDMM_SUM_OVER_BATCH) != 0, (flags & IEX_SDDMM_ACCUMULATE) != 0, (flags & IEX_SDDMM_PAD_OPERANDS) != 0};
  if (dtype == IEX_F32 && variant != 3 && variant != 7) return sddmm_split_bytes(dtype, p, variant == 12);
  if (variant == 12) return 0;
  const bool any_order = (flags & IEX_SDDMM_ANY_COLUMN_ORDER) != 0;
  if (variant != 7 && sddmm_mfma_fits(dtype, p) && (variant == 3 || (!any_order && sddmm_mfma_wins(p)))) return sddmm_mfma_bytes(p);
  if (variant == 3) return 0;
  if (!sddmm_dense_fits(dtype, p)) return 0;
  if (variant == 0 && !sddmm_dense_wins(p)) return 0;
  return sddmm_dense_bytes(p);
}

int sddmm_dispatch(int dtype, int flags, int m, int k, int n, int nonzeros, const int* row_indices,
                   const int* row_offsets, const int* column_indices, const void* lhs, const void* rhs,
                   void* out, void* stream, int batch, void* workspace, size_t workspace_bytes) {
  IEX_REQUIRE(m >= 0 && k >= 0 && n >= 0 && nonzeros >= 0 && batch >= 0, IEX_ERR_BAD_ARGUMENT,
              "sddmm: negative dimension (m=%d k=%d n=%d nnz=%d batch=%d)", m, k, n, nonzeros, batch);
  trail_reset();
  if (m == 0 || nonzeros == 0 || batch == 0) return 0;
  IEX_REQUIRE(row_indices && row_offsets && column_indices && out, IEX_ERR_BAD_ARGUMENT,
              "sddmm: null pointer argument");
  IEX_REQUIRE(k == 0 || (lhs && rhs), IEX_ERR_BAD_ARGUMENT, "sddmm: null dense operand");
  IEX_REQUIRE(batch <= 65535, IEX_ERR_TOO_LARGE, "sddmm: batch %d exceeds 65535", batch);
  IEX_REQUIRE((long long)m * k < (1ll << 31) && (long long)n * k < (1ll << 31), IEX_ERR_TOO_LARGE,
              "sddmm: a dense operand exceeds 2^31 elements per batch entry");
  SddmmParams p{m, k, n, nonzeros, batch, row_indices, row_offsets, column_indices, lhs, rhs, out,
                (flags & IEX_SDDMM_SUM_OVER_BATCH) != 0, (flags & IEX_SDDMM_ACCUMULATE) != 0, (flags & IEX_SDDMM_PAD_OPERANDS) != 0};
  int wpr = (flags >> 8) & 0xff;  // forced (1 or 4), else from the mean row length
  if (wpr != 1 && wpr != 4) wpr = ((double)nonzeros / m >= 64.0) ? 4 : 1;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int variant = (flags >> 16) & 0xf;  // 0 = choose, 1 = gather kernel, 3 = score tiles on the matrix cores, 7 = dense product then sampling, 12 = the same by parts
  const bool any_order = (flags & IEX_SDDMM_ANY_COLUMN_ORDER) != 0;   // (the tables of variant 3 assume ascending, distinct columns)
  if ((variant == 0 && !any_order) || variant == 3) {
    const bool fits = sddmm_mfma_fits(dtype, p);
    const bool room = workspace && aligned(workspace, 16) && workspace_bytes >= sddmm_mfma_bytes(p);
    if (variant == 3) {
      IEX_REQUIRE(fits, IEX_ERR_UNSUPPORTED, "sddmm: the matrix-core kernel needs fp16 / bf16, k = 32, 64 or 128, plain store, one output per batch entry and 16-byte aligned operands");
      IEX_REQUIRE(room, IEX_ERR_BAD_ARGUMENT, "sddmm: the matrix-core kernel needs a 16-byte aligned workspace of %zu bytes (iex_sddmm_ws)", sddmm_mfma_bytes(p));
    }
    if (fits && room && (variant == 3 || sddmm_mfma_wins(p))) return launch_sddmm_mfma(dtype, p, workspace, variant == 3 ? (flags >> 8) & 0xff : 0,
                                                                                 ((flags & IEX_SDDMM_TABLES_READY) ? 1 : 0) | ((flags & IEX_SDDMM_LISTS_READY) ? 2 : 0), s);
  }
  if (variant == 0 || variant == 7) {
    const bool fits = sddmm_dense_fits(dtype, p);
    const bool room = workspace && aligned(workspace, 16) && workspace_bytes >= sddmm_dense_bytes(p);
    if (variant == 7) {
      IEX_REQUIRE(fits, IEX_ERR_UNSUPPORTED, "sddmm: the dense-product path needs fp16 / bf16, plain store, one batch entry per output and, without IEX_SDDMM_PAD_OPERANDS, k and n multiples of 8 and 16-byte aligned operands");
      IEX_REQUIRE(room, IEX_ERR_BAD_ARGUMENT, "sddmm: the dense-product path needs a 16-byte aligned workspace of %zu bytes (iex_sddmm_ws)", sddmm_dense_bytes(p));
    }
    if (fits && room && (variant == 7 || sddmm_dense_wins(p))) return launch_sddmm_dense(dtype, p, workspace, s);
  }
  if ((variant == 0 || variant == 12) && workspace && aligned(workspace, 256)) {
    const size_t need = sddmm_split_bytes(dtype, p, variant == 12);
    if (need && workspace_bytes >= need) return launch_sddmm_split(p, workspace, s);
  }
  switch (dtype) {
    case IEX_F32: return launch_typed<float>(p, wpr, s);
    case IEX_F16: return launch_typed<__half>(p, wpr, s);
    case IEX_BF16: return launch_typed<__hip_bfloat16>(p, wpr, s);
  }
  return fail(IEX_ERR_UNSUPPORTED, "sddmm: no kernel for dtype=%d", dtype);
}

}  // namespace iex

extern "C" {

int iex_sddmm_ex(int dtype, int flags, int m, int k, int n, int nonzeros, const int* row_indices,
                 const int* row_offsets, const int* column_indices, const void* lhs_matrix,
                 const void* rhs_matrix, void* output_values, void* stream, int batch) {
  return iex::sddmm_dispatch(dtype, flags, m, k, n, nonzeros, row_indices, row_offsets, column_indices,
                             lhs_matrix, rhs_matrix, output_values, stream, batch, nullptr, 0);
}

int iex_sddmm_ws(int dtype, int flags, int m, int k, int n, int nonzeros, const int* row_indices,
                 const int* row_offsets, const int* column_indices, const void* lhs_matrix,
                 const void* rhs_matrix, void* output_values, void* stream, int batch, void* workspace,
                 size_t workspace_bytes) {
  return iex::sddmm_dispatch(dtype, flags, m, k, n, nonzeros, row_indices, row_offsets, column_indices,
                             lhs_matrix, rhs_matrix, output_values, stream, batch, workspace, workspace_bytes);
}

size_t iex_sddmm_workspace_bytes(int dtype, int flags, int m, int k, int n, int nonzeros, int batch) {
  return iex::sddmm_workspace_bytes(dtype, flags, m, k, n, nonzeros, batch);
}

size_t iex_pattern_tables_bytes(int m, int n, int nonzeros) {
  using namespace iex;
  if (m <= 0 || n <= 0 || nonzeros <= 0) return 0;
  const int tiles = ceil_div(n, kSdBN);
  if (tiles > kSdMaxTiles || (long long)(tiles + 1) * m >= (1ll << 28)) return 0;
  return sb_words(m, tiles, nonzeros) * sizeof(int);
}

int iex_pattern_tables(int m, int n, int nonzeros, const int* row_offsets, const int* column_indices, void* workspace,
                       size_t workspace_bytes, void* stream) {
  using namespace iex;
  const size_t need = iex_pattern_tables_bytes(m, n, nonzeros);
  IEX_REQUIRE(need > 0, IEX_ERR_UNSUPPORTED, "pattern tables: needs m, n, nonzeros > 0 and n <= %d", kSdMaxTiles * kSdBN);
  IEX_REQUIRE(row_offsets && column_indices && workspace && aligned(workspace, 16) && workspace_bytes >= need, IEX_ERR_BAD_ARGUMENT,
              "pattern tables: null pointer, or the workspace is not 16-byte aligned or shorter than %zu bytes", need);
  trail_reset();
  const int tiles = ceil_div(n, kSdBN);
  return sb_setup(sd_tables(workspace, m, tiles), sb_lists(workspace, m, tiles, nonzeros), m, tiles, 0, 0, row_offsets, column_indices,
                  static_cast<hipStream_t>(stream));
}

int iex_sddmm_workspace_kind(int dtype, int flags, int m, int k, int n, int nonzeros, int batch) {
  return iex::sddmm_workspace_kind(dtype, flags, m, k, n, nonzeros, batch);
}

int iex_CudaSddmm2(int m, int k, int n, int nonzeros, const int* row_indices, const int* row_offsets,
                   const int* column_indices, const float* lhs_matrix, const float* rhs_matrix,
                   float* output_values, void* stream, int batch_size) {
  return iex::sddmm_dispatch(IEX_F32, IEX_SDDMM_SUM_OVER_BATCH | IEX_SDDMM_ANY_COLUMN_ORDER, m, k, n, nonzeros, row_indices,
                             row_offsets, column_indices, lhs_matrix, rhs_matrix, output_values, stream,
                             batch_size, nullptr, 0);
}

}  // extern "C"
