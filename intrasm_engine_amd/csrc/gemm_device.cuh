// Dense companion GEMM for gfx950: C = A * B (or A * B^T), fp16 / bf16 in, fp32
// accumulate on the matrix cores, LDS double-buffered.  Here: what the GEMM kernels share (the matrix-core forms, their
// accumulators, the epilogue), and the tile whose operands travel through registers (tile codes 1 - 4, v_mfma_f32_32x32x16);
// the tiles that are chosen are those of gemm_dma_device.cuh and gemm_pp_device.cuh (v_mfma_f32_16x16x32).
//
// Tiling: a workgroup of 2 x WCN wavefronts (WCN = 2, or 4 for the 512-thread workgroups of
// the fused launch) owns a (2*WM*32) x (WCN*WN*32) tile of C; a wavefront owns WM x WN MFMA
// tiles of 32 x 32.  The K loop advances BK = 32 per step.
// Software pipeline: global loads run kGemmSets steps ahead of the MFMAs (one register set
// per step in flight, 128-bit loads), a set is written to the idle LDS buffer one step
// before it is consumed, one barrier per step:
//   step t:  MFMA on LDS[t%2] | registers(tile t+1) -> LDS[(t+1)%2] | issue loads of tile t+1+SETS
// so a global load has kGemmSets MFMA steps to complete (L2 / MALL latency is several steps).
// A (and B given as (N, K)) sit in LDS K-contiguous ([row][k], rows padded by 8 elements so
// that the 128-bit operand reads of 8 consecutive lanes fall in distinct banks).  B given as
// (K, N) is kept in LDS as it is in memory ([k][n], rows padded by 32 elements) and the MFMA
// operand is formed by the LDS transpose read of gfx950 (ds_read_b64_tr_b16): the 16 lanes
// of a group each point at 4 adjacent n of one k row, and lane i receives column n0+i of 4
// consecutive k rows, so no register transposes and full 128-bit global loads for both
// layouts.
// The MFMA is issued with the operands swapped (B fragment as the "A" operand): a lane
// then holds 4 adjacent columns of one row of C per accumulator quad and stores them
// with one 64-bit store.
#pragma once
#include <type_traits>
#include <utility>

#include "iex_common.h"

namespace iex {

// f(0), .., f(COUNT - 1), each number a type
template <typename F, int... N>
__device__ __forceinline__ void for_each_of(F&& f, std::integer_sequence<int, N...>) {
  (f(std::integral_constant<int, N>{}), ...);
}
template <int COUNT, typename F>
__device__ __forceinline__ void for_each_number(F&& f) {
  for_each_of(f, std::make_integer_sequence<int, COUNT>{});
}

struct GemmParams {
  int M, N, K;
  const void* A;
  const void* B;
  void* C;
  long long stride_a, stride_b, stride_c;
  int tiles_m, tiles_n;
  // epilogue beyond C = A * B: C = relu?(A * B + row_bias[row]), then with an auxiliary operand of C's shape and strides
  // (any alignment; it may be C itself) C = that + aux (kGemmAdd) or C = that * silu(aux) (kGemmTimesSilu)
  const float* row_bias = nullptr;
  int relu = 0;
  int aux_mode = 0;
  const void* aux = nullptr;
  int stream_out = 0;  // C is far larger than the caches: store it with the streaming hint
  // row strides in elements, 0 = the natural one (A: K, or M where it is given as (K,M); B: K, or N where it is given as
  // (K,N); C: N), and the rows of a (K,N) B that exist where K has been rounded up (0 = K; A is zero beyond them)
  int lda = 0, ldb = 0, ldc = 0, kb = 0;
  // K split over two workgroups per tile (gemm.hip): where the first workgroup to finish a tile leaves its fp32 partial
  // sums, and per tile a ticket counter and a "partial sums written" flag (both zero at launch)
  float* split_ws = nullptr;
  int* split_flags = nullptr;
  // K split over split_parts workgroups per tile, every one of which leaves its partial sums in the workspace and draws
  // a ticket (zero at launch); the one that draws the last adds all parts up in the order of the parts and stores
  int split_parts = 0, split_part = 0;
};

constexpr int kGemmAdd = 1, kGemmTimesSilu = 2;

// iex_gemm with the options above (gemm.hip).  code: bit 0 = B is (N,K), bit 1 = A is (K,M), bits 4..8 = forced kernel.
int gemm_dispatch(int dtype, int code, const GemmParams& p, int batch, hipStream_t stream, void* workspace = nullptr, size_t workspace_bytes = 0,
                  bool workspace_flags_are_zero = false);
// Bytes of workspace with which gemm_dispatch, left to choose, splits K over two workgroups per tile (0: this shape is
// not split), and where in such a workspace the words sit that must be zero at launch (gemm_dispatch zeroes them with a
// launch of its own unless the caller says it has: workspace_flags_are_zero).
size_t gemm_auto_split_bytes(int M, int N, int K, int batch);
int gemm_auto_split_parts(int M, int N, int K, int batch);   // parts of K that gemm_dispatch would use with that workspace (1: no split)
void gemm_auto_split_flags(int M, int N, int K, int batch, size_t* offset_bytes, int* words);
double gemm_seconds(int M, int N, int K);   // an estimate, for choices between a dense product and others

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

constexpr int kGemmBK = 32;
constexpr int kGemmPad = 8;
constexpr int kGemmLd = kGemmBK + kGemmPad;  // LDS row stride in elements (80 bytes)
constexpr int kGemmSets = 3;                 // register sets = K steps of global loads in flight

constexpr int kGemmLdbPad = 32;  // padding of a [k][n] row of B in LDS, elements

template <bool TRANS_B, int WM, int WN, int WCN = 2, int BK = kGemmBK>
constexpr int gemm_lds_bytes() {
  constexpr int a_elems = 2 * WM * 32 * (BK + kGemmPad);
  constexpr int b_elems = TRANS_B ? WCN * WN * 32 * (BK + kGemmPad) : BK * (WCN * WN * 32 + kGemmLdbPad);
  return 2 /*buffers*/ * (a_elems + b_elems) * 2 /*bytes*/;
}

typedef short s16x4 __attribute__((ext_vector_type(4)));

template <bool BF16>
__device__ __forceinline__ f32x16 mfma_32x32x16(u32x4 a, u32x4 b, f32x16 c) {
  if constexpr (BF16) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
  }
}

// Half the accumulator traffic per flop of the 32 x 32 form: under the power limit random operands run at 1930 instead of
// 1710 TFLOP/s, all-zero ones at 2430 / 2460 (benchmarks/mfma_rates.hip: MFMAs and nothing else on every CU).
template <bool BF16>
__device__ __forceinline__ f32x4 mfma_16x16x32(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (BF16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
}

// The accumulators of a wavefront's WM x WN blocks of 32 x 32 (operands swapped: a quad is 4 adjacent columns of one row),
// as quads: quad t of 4 * WN of row block i, with the row and the first column it has inside the block row.
template <int WM, int WN>
struct Acc32 {   // one 32 x 32 MFMA per block
  f32x16 v[WM][WN];
  __device__ __forceinline__ f32x4 quad(int i, int t) const {
    const f32x16& a = v[i][t / 4];
    return f32x4{a[t % 4 * 4], a[t % 4 * 4 + 1], a[t % 4 * 4 + 2], a[t % 4 * 4 + 3]};
  }
  static __device__ __forceinline__ int row(int, int lane) { return lane & 31; }
  static __device__ __forceinline__ int col(int t, int lane) { return t * 8 + (lane >> 5) * 4; }
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) v[i][j][r] = 0.f;
  }
};
template <int WM, int WN>
struct Acc16 {   // 2 x 2 MFMAs of 16 x 16 per block
  f32x4 v[2 * WM][2 * WN];
  __device__ __forceinline__ f32x4 quad(int i, int t) const { return v[2 * i + t / (2 * WN)][t % (2 * WN)]; }
  __device__ __forceinline__ void add(int i, int t, f32x4 x) { v[2 * i + t / (2 * WN)][t % (2 * WN)] += x; }
  static __device__ __forceinline__ int row(int t, int lane) { return t / (2 * WN) * 16 + (lane & 15); }
  static __device__ __forceinline__ int col(int t, int lane) { return t % (2 * WN) * 16 + (lane >> 4) * 4; }
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < 2 * WM; ++i)
#pragma unroll
      for (int j = 0; j < 2 * WN; ++j) v[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
};

__device__ __forceinline__ float f16_to_32(unsigned short h, bool bf16) {
  if (bf16) return __uint_as_float((unsigned)h << 16);
  return (float)__builtin_bit_cast(_Float16, h);
}

__device__ __forceinline__ unsigned short f32_to_16(float v, bool bf16) {
  if (bf16) {
    __hip_bfloat16 h = __float2bfloat16(v);
    return __builtin_bit_cast(unsigned short, h);
  }
  __half h = __float2half_rn(v);
  return __builtin_bit_cast(unsigned short, h);
}

// The slice of one K step that a thread carries from global memory to LDS.
template <bool TRANS_B, int BM, int BN, int THREADS = 256, int BK_ = kGemmBK>
struct GemmStage {
  static constexpr int BK = BK_;
  static constexpr int LD = BK_ + kGemmPad;
  static constexpr int A_CHUNKS = BM * (BK / 8) / THREADS;   // 128-bit chunks per thread (A, and B^T layout)
  static constexpr int B_CHUNKS = BN * (BK / 8) / THREADS;
  static_assert(A_CHUNKS >= 1 && B_CHUNKS >= 1, "a stage must give every thread a chunk of A and of B");
  static constexpr int LDB = BN + kGemmLdbPad;               // LDS row stride of B kept as [k][n]
  static constexpr int B_ELEMS = TRANS_B ? BN * LD : BK * LDB;  // one LDS buffer of B, elements
  typedef unsigned short u16;

  u32x4 ra[A_CHUNKS];
  u32x4 rb[B_CHUNKS];  // (N,K): chunk = 8 k of one n row; (K,N): chunk = 8 n of one k row

  // Loads are unconditional, from addresses clamped into the matrices, and nothing is computed
  // on their results here: guarded loads are branches, and behind a branch the compiler can no
  // longer count the loads in flight and waits for all of them wherever one is needed.  Rows of A
  // (columns of B) beyond the matrix only feed rows (columns) of C that are never stored; the K
  // tail is zeroed when the set is written to LDS.
  __device__ __forceinline__ void load(const GemmParams& p, const u16* __restrict__ A, const u16* __restrict__ B, int m0,
                                       int n0, int kt, int tid) {
    const int k0 = kt * BK;
    const int last_k8 = p.K - 8;  // K % 8 == 0: the last whole chunk of a row
#pragma unroll
    for (int c = 0; c < A_CHUNKS; ++c) {
      const int chunk = tid + c * THREADS;
      const int row = chunk / (BK / 8), kc = chunk % (BK / 8);
      const int gm = min(m0 + row, p.M - 1), gk = min(k0 + kc * 8, last_k8);
      ra[c] = *reinterpret_cast<const u32x4*>(A + (size_t)gm * p.K + gk);
    }
    if constexpr (TRANS_B) {
#pragma unroll
      for (int c = 0; c < B_CHUNKS; ++c) {
        const int chunk = tid + c * THREADS;
        const int row = chunk / (BK / 8), kc = chunk % (BK / 8);
        const int gn = min(n0 + row, p.N - 1), gk = min(k0 + kc * 8, last_k8);
        rb[c] = *reinterpret_cast<const u32x4*>(B + (size_t)gn * p.K + gk);
      }
    } else {
      const int last_n8 = p.N - 8;  // N % 8 == 0 in this layout
#pragma unroll
      for (int c = 0; c < B_CHUNKS; ++c) {
        const int chunk = tid + c * THREADS;
        const int kr = chunk / (BN / 8), nc = chunk % (BN / 8);
        const int gk = min(k0 + kr, p.K - 1), gn = min(n0 + nc * 8, last_n8);
        rb[c] = *reinterpret_cast<const u32x4*>(B + (size_t)gk * p.N + gn);
      }
    }
  }

  // kt = the K step the set carries (for the K tail: entries at k >= K are written as zeros)
  __device__ __forceinline__ void store(const GemmParams& p, u16* a, u16* b, int kt, int tid) const {
    const int k0 = kt * BK;
    const bool tail = k0 + BK > p.K;  // uniform
    const u32x4 zero = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int c = 0; c < A_CHUNKS; ++c) {
      const int chunk = tid + c * THREADS;
      const int row = chunk / (BK / 8), kc = chunk % (BK / 8);
      *reinterpret_cast<u32x4*>(a + row * LD + kc * 8) = (tail && k0 + kc * 8 >= p.K) ? zero : ra[c];
    }
    if constexpr (TRANS_B) {
#pragma unroll
      for (int c = 0; c < B_CHUNKS; ++c) {
        const int chunk = tid + c * THREADS;
        const int row = chunk / (BK / 8), kc = chunk % (BK / 8);
        *reinterpret_cast<u32x4*>(b + row * LD + kc * 8) = (tail && k0 + kc * 8 >= p.K) ? zero : rb[c];
      }
    } else {
#pragma unroll
      for (int c = 0; c < B_CHUNKS; ++c) {
        const int chunk = tid + c * THREADS;
        const int kr = chunk / (BN / 8), nc = chunk % (BN / 8);
        *reinterpret_cast<u32x4*>(b + kr * LDB + nc * 8) = (tail && k0 + kr >= p.K) ? zero : rb[c];
      }
    }
  }
};

// Writes the WM x WN accumulator blocks of one wavefront to C (rounded to the 16-bit type), through LDS: a lane's
// accumulators are 4 adjacent columns of 32 different rows, so a direct store would write 32 pieces of 16 bytes per
// instruction; here each 32-row block of the wavefront's tile is laid out in the wavefront's own slice of LDS (rows padded
// by 16 bytes) and read back 16 lanes per row, so a store instruction writes 4 rows of WN * 64 contiguous bytes.  A GEMM
// with a short K is a writer of its output: 16 x 4096 x 4096 outputs with K = 64 went from 1.7 TB/s to the rate of a fill.
// An auxiliary operand takes the same way in before: rows read 16 lanes at a time, picked up by the lanes that hold their
// sums, combined in fp32 and rounded once.  Rows of C that are not 16-byte aligned (any N, any pointer) are stored with
// vectors at element alignment, the columns past the last whole vector one by one.
// `lds` = this wavefront's slice, gemm_store_lds_bytes<WN>() bytes, nobody else touches it (no barrier needed: the LDS
// operations of one wavefront execute in order).  `stream`: store with the streaming hint.  `partial`: another half of the
// sums in this lane's order, 256 floats per (block, quad).
template <int WN>
constexpr int gemm_store_lds_bytes() { return 32 * (WN * 64 + 16); }

// Two sums as one word of the 16-bit type.
template <bool BF16>
__device__ __forceinline__ unsigned pack_16(float x, float y) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
  if constexpr (BF16) return __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{x, y}), bf16x2));
  else return __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{x, y}), f16x2));
}
template <bool BF16>
__device__ __forceinline__ void unpack_16(unsigned w, float& x, float& y) {
  if constexpr (BF16) {
    x = __uint_as_float(w << 16);
    y = __uint_as_float(w & 0xffff0000u);
  } else {
    x = (float)__builtin_bit_cast(_Float16, (unsigned short)(w & 0xffffu));
    y = (float)__builtin_bit_cast(_Float16, (unsigned short)(w >> 16));
  }
}

// The plain case of gemm_store_tile below: rows of whole 16-byte vectors, no row bias, no ReLU; AUX = its aux_mode (0: none).  Without a branch:
// stores are buffer stores, which drop what lies outside C (a lane whose row or column does not exist asks for the buffer's end).
// That is what an epilogue costs: its instructions run once per tile, out of a cold instruction cache, and the general code below
// is 60 KB of them for a 128 x 64 wavefront tile (one 256 x 256 tile and nothing else: 12.4 us, 4.8 without its epilogue, 8.0 with this one).
template <bool BF16, int WM, int WN, int AUX, bool STREAM, typename Acc>
__device__ __forceinline__ void gemm_store_whole(const GemmParams& p, const Acc& acc, unsigned short* C, const unsigned short* aux, int m0, int n0, int wm,
                                                 int wn, int lane, unsigned char* lds) {
  constexpr int ROWB = WN * 64 + 16, CPR = WN * 4, RPI = kWave / CPR;   // as below
  const int ldc = p.ldc ? p.ldc : p.N;
  const int chunk = lane % CPR, first = m0 + wm * WM * 32 + lane / CPR, gn = n0 + wn * WN * 32 + chunk * 8;
  const unsigned bytes = ((unsigned)(p.M - 1) * ldc + p.N) * 2u;   // (below 2^32: the host's limits)
  const auto c_buf = __builtin_amdgcn_make_buffer_rsrc(C, 0, bytes, 4 << 15);
  const auto aux_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned short*>(AUX ? aux : C), 0, bytes, 4 << 15);
  auto at = [&](int i, int t) {
    const int row = first + i * 32 + t * RPI;
    return row < p.M && gn < p.N ? ((unsigned)row * ldc + gn) * 2u : 0xfffffff0u;
  };
  u32x4 held[WM][32 / RPI];
  if constexpr (AUX != 0) {   // all of the tile's in flight together
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int t = 0; t < 32 / RPI; ++t) held[i][t] = __builtin_amdgcn_raw_buffer_load_b128(aux_buf, at(i, t), 0, 0);
  }
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    if constexpr (AUX != 0) {
#pragma unroll
      for (int t = 0; t < 32 / RPI; ++t) *reinterpret_cast<u32x4*>(lds + (t * RPI + lane / CPR) * ROWB + chunk * 16) = held[i][t];
    }
#pragma unroll
    for (int t = 0; t < 4 * WN; ++t) {
      u32x2* to = reinterpret_cast<u32x2*>(lds + Acc::row(t, lane) * ROWB + Acc::col(t, lane) * 2);
      f32x4 y = acc.quad(i, t);
      if constexpr (AUX != 0) {
        const u32x2 w = *to;
        float other[4];
        unpack_16<BF16>(w.x, other[0], other[1]);
        unpack_16<BF16>(w.y, other[2], other[3]);
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = AUX == kGemmAdd ? y[e] + other[e] : y[e] * (other[e] / (1.f + __expf(-other[e])));
      }
      *to = u32x2{pack_16<BF16>(y[0], y[1]), pack_16<BF16>(y[2], y[3])};
    }
#pragma unroll
    for (int t = 0; t < 32 / RPI; ++t)
      __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4*>(lds + (t * RPI + lane / CPR) * ROWB + chunk * 16), c_buf, at(i, t), 0, STREAM ? 2 : 0);
  }
}

template <bool BF16, int WM, int WN, typename Acc>
__device__ __forceinline__ void gemm_store_tile(const GemmParams& p, const Acc& acc, unsigned short* __restrict__ C,
                                                const unsigned short* aux, int m0, int n0, int wm, int wn, int lane, unsigned char* lds,
                                                bool stream, const float* partial = nullptr) {
  typedef unsigned short u16;
  typedef u32x4 u128_a2 __attribute__((aligned(2)));
  constexpr int ROWB = WN * 64 + 16;   // bytes of a padded row
  constexpr int CPR = WN * 4;          // 16-byte chunks per row
  constexpr int RPI = kWave / CPR;     // rows a store instruction covers
  static_assert(kWave % CPR == 0 && 32 % RPI == 0, "whole rows per instruction");
  const int ldc = p.ldc ? p.ldc : p.N;
  // rows of whole vectors and nothing but an auxiliary operand to do (uniform)
  if (p.N % 8 == 0 && ldc % 8 == 0 && ((reinterpret_cast<uintptr_t>(C) | reinterpret_cast<uintptr_t>(aux)) & 15) == 0 && !p.row_bias && !p.relu && !partial &&
      (long long)(p.M + 256) * ldc < (1ll << 31)) {
    const int mode = aux ? p.aux_mode : 0;
    auto store = [&](auto m, auto s) { gemm_store_whole<BF16, WM, WN, decltype(m)::value, decltype(s)::value>(p, acc, C, aux, m0, n0, wm, wn, lane, lds); };
    auto by_mode = [&](auto s) {
      if (mode == 0) store(std::integral_constant<int, 0>{}, s);
      else if (mode == kGemmAdd) store(std::integral_constant<int, kGemmAdd>{}, s);
      else store(std::integral_constant<int, kGemmTimesSilu>{}, s);
    };
    if (stream) by_mode(std::true_type{});
    else by_mode(std::false_type{});
    return;
  }
  const int chunk = lane % CPR;
  const int gn = n0 + wn * WN * 32 + chunk * 8;
  const int here = min(p.N - gn, 8);   // columns of this lane's chunk that exist (none: <= 0)
  const bool whole = p.N % 8 == 0 && ldc % 8 == 0 && (reinterpret_cast<uintptr_t>(C) & 15) == 0;   // (uniform)
  // the auxiliary operand of the whole tile, all loads in flight together (the fragments' registers are free by now)
  u32x4 held[WM][32 / RPI];
  if (aux) {
    const bool whole_aux = whole && (reinterpret_cast<uintptr_t>(aux) & 15) == 0;   // (uniform)
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int t = 0; t < 32 / RPI; ++t) {
        const u16* src = aux + (size_t)min(m0 + (wm * WM + i) * 32 + t * RPI + lane / CPR, p.M - 1) * ldc + gn;
        held[i][t] = u32x4{0u, 0u, 0u, 0u};
        if (here == 8) {
          held[i][t] = whole_aux ? *reinterpret_cast<const u32x4*>(src) : *reinterpret_cast<const u128_a2*>(src);
        } else {
          unsigned w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (e < here) w[e / 2] |= (unsigned)src[e] << (16 * (e & 1));
          held[i][t] = u32x4{w[0], w[1], w[2], w[3]};
        }
      }
  }
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const int row0 = m0 + (wm * WM + i) * 32;
    if (row0 >= p.M) break;  // (uniform)
    float bias[2] = {0.f, 0.f};   // of the row(s) this lane holds sums of
    if (p.row_bias) {
      bias[0] = p.row_bias[min(row0 + Acc::row(0, lane), p.M - 1)];
      bias[1] = p.row_bias[min(row0 + Acc::row(4 * WN - 1, lane), p.M - 1)];
    }
    if (aux) {
#pragma unroll
      for (int t = 0; t < 32 / RPI; ++t) *reinterpret_cast<u32x4*>(lds + (t * RPI + lane / CPR) * ROWB + chunk * 16) = held[i][t];
    }
#pragma unroll
    for (int t = 0; t < 4 * WN; ++t) {
      u16 h[4];
      u32x2* at = reinterpret_cast<u32x2*>(lds + Acc::row(t, lane) * ROWB + Acc::col(t, lane) * 2);
      const f32x4 mine = acc.quad(i, t);
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
      if (partial) o = *reinterpret_cast<const f32x4*>(partial + (i * 4 * WN + t) * 256);   // the other half of K
      float other[4] = {0.f, 0.f, 0.f, 0.f};
      if (aux) {
        const u32x2 w = *at;
        other[0] = f16_to_32((u16)(w.x & 0xffffu), BF16);
        other[1] = f16_to_32((u16)(w.x >> 16), BF16);
        other[2] = f16_to_32((u16)(w.y & 0xffffu), BF16);
        other[3] = f16_to_32((u16)(w.y >> 16), BF16);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float y = mine[e] + o[e] + bias[t / (2 * WN)];
        if (aux && p.aux_mode == kGemmAdd) y += other[e];
        if (p.relu) y = fmaxf(y, 0.f);
        if (aux && p.aux_mode == kGemmTimesSilu) y *= other[e] / (1.f + __expf(-other[e]));
        h[e] = f32_to_16(y, BF16);
      }
      u32x2 w;
      w.x = (unsigned)h[0] | ((unsigned)h[1] << 16);
      w.y = (unsigned)h[2] | ((unsigned)h[3] << 16);
      *at = w;
    }
#pragma unroll
    for (int t = 0; t < 32 / RPI; ++t) {
      const int r = t * RPI + lane / CPR;
      const u32x4 v = *reinterpret_cast<const u32x4*>(lds + r * ROWB + chunk * 16);
      if (row0 + r < p.M && here > 0) {
        u16* dst = C + (size_t)(row0 + r) * ldc + gn;
        if (whole && stream) {
          asm volatile("" : "+v"(dst));  // (keeps the compiler from merging this store with the plain one and dropping the hint)
          __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(dst));
        } else if (whole) {
          *reinterpret_cast<u32x4*>(dst) = v;
        } else if (here == 8) {
          *reinterpret_cast<u128_a2*>(dst) = v;
        } else {
          const unsigned w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (e < here) dst[e] = (u16)(w[e / 2] >> (16 * (e & 1)));
        }
      }
    }
  }
}

// One C tile.  `smem` must hold gemm_lds_bytes<WM,WN>() bytes, 16-byte aligned.
// All 2 * WCN * 64 threads of the workgroup must call this (it contains barriers).
template <bool BF16, bool TRANS_B, int WM, int WN, int SETS = kGemmSets, int WCN = 2, int BK = kGemmBK>
__device__ __forceinline__ void gemm_tile(const GemmParams& p, int tile_m, int tile_n, int z, unsigned char* smem) {
  constexpr int BM = 2 * WM * 32;
  constexpr int BN = WCN * WN * 32;
  constexpr int LD = BK + kGemmPad;
  static_assert(SETS == 2 || SETS == 3, "register sets in flight");
  constexpr int PERIOD = SETS == 2 ? 2 : 6;  // steps after which LDS buffer and register set repeat
  typedef unsigned short u16;

  typedef GemmStage<TRANS_B, BM, BN, 2 * WCN * 64, BK> Stage;
  constexpr int LDB = Stage::LDB;
  constexpr int B_ELEMS = Stage::B_ELEMS;
  u16* sA = reinterpret_cast<u16*>(smem);  // [2][BM][LD]
  u16* sB = sA + 2 * BM * LD;              // [2][BN][LD]  or  [2][BK][LDB]

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave / WCN, wn = wave % WCN;
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const u16* __restrict__ A = static_cast<const u16*>(p.A) + (size_t)z * p.stride_a;
  const u16* __restrict__ B = static_cast<const u16*>(p.B) + (size_t)z * p.stride_b;
  u16* __restrict__ C = static_cast<u16*>(p.C) + (size_t)z * p.stride_c;

  Acc32<WM, WN> acc;
  acc.clear();

  Stage regs[SETS];  // regs[t % SETS] carries tile t (statically indexed below)

  const int KT = (p.K + BK - 1) / BK;
  // prologue: tiles 0 .. SETS-1 in flight, tile 0 into LDS[0], then tile SETS replaces it
#pragma unroll
  for (int s = 0; s < SETS; ++s)
    regs[s].load(p, A, B, m0, n0, s, tid);  // (a tile beyond the last one loads clamped addresses and is never used)
  regs[0].store(p, sA, sB, 0, tid);
  regs[0].load(p, A, B, m0, n0, SETS, tid);
  __syncthreads();

  const int frag_row = lane & 31;      // row of the 32-row operand block this lane feeds
  const int frag_k = (lane >> 5) * 8;  // which 8 of the 16 k entries of a sub-step

  // One step; PH = t % (2*SETS) is a compile-time phase so that both the register set
  // ((t+1) % SETS) and the LDS buffer (t % 2) are static.
  auto step = [&](int kt, auto phase) {
    constexpr int PH = decltype(phase)::value;
    constexpr int buf = PH & 1;
    constexpr int set = (PH + 1) % SETS;
    const u16* a = sA + buf * BM * LD + (wm * WM * 32 + frag_row) * LD + frag_k;
    // (N,K) layout: 128-bit read of 8 k of row n.  (K,N) layout: two transpose reads; the lane
    // group q = lane/16 covers n-half (q%2) and k-half (q/2) of the sub-step, lane r of the
    // group points at k row r/4 and n columns 4*(r%4).., and receives column n0 + r of 4 k rows.
    const u16* b = TRANS_B ? sB + buf * B_ELEMS + (wn * WN * 32 + frag_row) * LD + frag_k
                           : sB + buf * B_ELEMS + ((lane >> 5) * 8 + ((lane & 15) >> 2)) * LDB + wn * WN * 32 +
                                 ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
    // the operand fragments of two 16-wide sub-steps are requested before their MFMAs: the reads
    // of the second land while the MFMAs of the first run
#pragma unroll
    for (int kp = 0; kp < BK / 32; ++kp) {
      u32x4 fa[2][WM], fb[2][WN];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int ks = kp * 2 + h;
#pragma unroll
        for (int i = 0; i < WM; ++i) fa[h][i] = *reinterpret_cast<const u32x4*>(a + i * 32 * LD + ks * 16);
#pragma unroll
        for (int j = 0; j < WN; ++j) {
          if constexpr (TRANS_B) {
            fb[h][j] = *reinterpret_cast<const u32x4*>(b + j * 32 * LD + ks * 16);
          } else {
            typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
            const u16* q0 = b + (ks * 16) * LDB + j * 32;
            const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(q0));
            const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(q0 + 4 * LDB));
            const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
            fb[h][j] = u32x4{l2.x, l2.y, h2.x, h2.y};
          }
        }
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
          for (int j = 0; j < WN; ++j) acc.v[i][j] = mfma_32x32x16<BF16>(fb[h][j], fa[h][i], acc.v[i][j]);
    }
    // unconditional on purpose (see GemmStage::load): past the last tile this writes zeros to the
    // idle buffer and fetches clamped addresses
    regs[set].store(p, sA + (buf ^ 1) * BM * LD, sB + (buf ^ 1) * B_ELEMS, kt + 1, tid);
    regs[set].load(p, A, B, m0, n0, kt + 1 + SETS, tid);
    __syncthreads();
  };

  int kt = 0;
  if constexpr (PERIOD == 6) {
    for (; kt + 6 <= KT; kt += 6) {
      step(kt + 0, std::integral_constant<int, 0>{});
      step(kt + 1, std::integral_constant<int, 1>{});
      step(kt + 2, std::integral_constant<int, 2>{});
      step(kt + 3, std::integral_constant<int, 3>{});
      step(kt + 4, std::integral_constant<int, 4>{});
      step(kt + 5, std::integral_constant<int, 5>{});
    }
    if (kt < KT) step(kt++, std::integral_constant<int, 0>{});
    if (kt < KT) step(kt++, std::integral_constant<int, 1>{});
    if (kt < KT) step(kt++, std::integral_constant<int, 2>{});
    if (kt < KT) step(kt++, std::integral_constant<int, 3>{});
    if (kt < KT) step(kt++, std::integral_constant<int, 4>{});
  } else {
    for (; kt + 2 <= KT; kt += 2) {
      step(kt + 0, std::integral_constant<int, 0>{});
      step(kt + 1, std::integral_constant<int, 1>{});
    }
    if (kt < KT) step(kt++, std::integral_constant<int, 0>{});
  }

  static_assert(2 * WCN * gemm_store_lds_bytes<WN>() <= gemm_lds_bytes<TRANS_B, WM, WN, WCN, BK>(), "the epilogue fits the buffers");
  __syncthreads();  // everybody has read its last fragments
  gemm_store_tile<BF16, WM, WN>(p, acc, C, nullptr, m0, n0, wm, wn, lane, smem + wave * gemm_store_lds_bytes<WN>(), p.stream_out != 0);
}

}  // namespace iex
