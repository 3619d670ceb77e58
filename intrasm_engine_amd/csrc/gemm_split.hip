// Host side of the fp32 product by three bf16 parts, and the kernels that make the parts and pick sampled entries.
#include <algorithm>
#include "gemm_split_device.cuh"

namespace iex {
namespace {

// ---- parts --------------------------------------------------------------------------------------------------------
// Two neighbours' parts, packed (the first in the lower half): each part rounded to nearest of what the ones before left,
// which is exact in fp32.
struct PartsPair {
  unsigned high, middle, low;
};
__device__ __forceinline__ PartsPair parts_of(float x, float y) {
  PartsPair r;
  r.high = pack_pair<true>(x, y);
  const float x1 = x - __uint_as_float(r.high << 16), y1 = y - __uint_as_float(r.high & 0xffff0000u);
  r.middle = pack_pair<true>(x1, y1);
  r.low = pack_pair<true>(x1 - __uint_as_float(r.middle << 16), y1 - __uint_as_float(r.middle & 0xffff0000u));
  return r;
}

// eight neighbours to 16 bytes of each plane
__device__ __forceinline__ void store_parts(const float (&x)[8], uint16_t* dst, long long plane) {
  u32x4 h, m, l;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const PartsPair p = parts_of(x[2 * e], x[2 * e + 1]);
    h[e] = p.high, m[e] = p.middle, l[e] = p.low;
  }
  *reinterpret_cast<u32x4*>(dst) = h;
  *reinterpret_cast<u32x4*>(dst + plane) = m;
  *reinterpret_cast<u32x4*>(dst + 2 * plane) = l;
}

template <int WAVES>
__device__ __forceinline__ void leave_range(SplitRange x, unsigned* at) {
  __shared__ unsigned of[WAVES];
  x.over_wave();
  if (lane_id() == 0) of[threadIdx.x >> 6] = x.word();
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 0; w < WAVES; ++w) x.add_word(of[w]);
    *at = x.word();
  }
}

__device__ __forceinline__ SplitRange split_dense_block(const SplitDense& s, int block, int blocks) {
  struct alignas(4) Any { float v[8]; };
  const int chunks = s.dst_cols / 8;
  const long long total = (long long)s.batch * s.dst_rows * chunks;
  SplitExtent range;
  for (long long i = (long long)block * 256 + threadIdx.x; i < total; i += (long long)blocks * 256) {
    const long long zr = i / chunks;
    const int c = (int)(i - zr * chunks) * 8;
    const int z = (int)(zr / s.dst_rows), r = (int)(zr - (long long)z * s.dst_rows);
    float x[8];
    const float* src = s.src + ((size_t)z * s.rows + r) * s.cols + c;
    if (r < s.rows && c + 8 <= s.cols) {
      const Any a = *reinterpret_cast<const Any*>(src);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = a.v[e];
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = r < s.rows && c + e < s.cols ? src[e] : 0.f;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) range.add(x[e]);
    store_parts(x, static_cast<uint16_t*>(s.dst) + (size_t)z * s.dst_batch + (size_t)r * s.ld + c, s.plane);
  }
  return range.range();
}

// As csr_to_dense_kernel (spmm_dense_device.cuh): a workgroup per row, the row (or 4096 columns of it) assembled in LDS in fp32, its parts taken on
// the way out, every byte written once.  (4096 x 4096: 27 us, of which 20 are the bytes; two rows side by side the same, four 40.)
constexpr int kPlanesSeg = 4096, kPlanesWaves = 4;
__device__ __forceinline__ SplitRange split_sparse_block(const SplitSparse& s, int block, int blocks) {
  __shared__ __align__(16) float srow[kPlanesSeg];
  const int lane = lane_id(), wave = uniform(threadIdx.x >> 6);
  const int* __restrict__ cols = s.cols;
  const float* __restrict__ values = s.values;
  uint16_t* __restrict__ dst = static_cast<uint16_t*>(s.dst);
  SplitExtent range;
  bool again = false;
  for (int row = block; row < s.m; row += blocks) {
    // this wavefront's quarter of the row's nonzeros, in whole chunks of 64
    const int first = uniform(s.row_offsets[row]), last = uniform(s.row_offsets[row + 1]);
    const int share = ((max(last - first, 0) + kWave * kPlanesWaves - 1) / (kWave * kPlanesWaves)) * kWave;
    int pos = min(first + wave * share, last);
    const int end = min(pos + share, last);
    for (int c0 = 0; c0 < s.ld; c0 += kPlanesSeg) {
      const int len = min(kPlanesSeg, s.ld - c0);   // a multiple of 32
      if (again) __syncthreads();   // the previous segment has been copied out
      again = true;
      for (int i = threadIdx.x * 4; i < len; i += kPlanesWaves * kWave * 4) *reinterpret_cast<f32x4*>(srow + i) = f32x4{0.f, 0.f, 0.f, 0.f};
      __syncthreads();
      for (bool more = pos < end; more;) {
        int c[4];
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int j = min(pos + u * kWave + lane, end - 1);
          c[u] = cols[j] - c0;
          v[u] = values[j];
        }
        int taken = 0;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          // (the test on c keeps a row whose columns do not ascend inside the row's slice of LDS)
          const bool mine = pos + u * kWave + lane < end && c[u] < len && c[u] >= 0;
          if (mine) {
            srow[c[u]] = v[u];
            range.add(v[u]);
          }
          taken += __popcll(__ballot(mine));
        }
        pos += taken;
        more = taken == 4 * kWave;   // a short take: the quarter ended or its next nonzero lies beyond this segment
      }
      __syncthreads();
      for (int i = threadIdx.x * 8; i < len; i += kPlanesWaves * kWave * 8) {
        const f32x4 lo = *reinterpret_cast<const f32x4*>(srow + i), hi = *reinterpret_cast<const f32x4*>(srow + i + 4);
        const float x[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        store_parts(x, dst + (size_t)row * s.ld + c0 + i, s.plane);
      }
    }
  }
  return range.range();
}

// Both operands' parts in one launch: the first workgroups make those of the second operand.  Bound by the bytes, 4 read and 6 written an entry, 6
// written a cell of a sparse operand.  (A word per workgroup, not atomics: 8192 of them on 64 words took 25 us.)
template <typename First>
__global__ __launch_bounds__(256) void split_operands_kernel(First a, SplitDense b, unsigned* ranges, int blocks_b) {
  if ((int)blockIdx.x < blocks_b) {
    leave_range<4>(split_dense_block(b, blockIdx.x, blocks_b), ranges + blockIdx.x);
  } else {
    const int block = blockIdx.x - blocks_b, blocks = gridDim.x - blocks_b;
    SplitRange range;
    if constexpr (std::is_same<First, SplitSparse>::value) range = split_sparse_block(a, block, blocks);
    else range = split_dense_block(a, block, blocks);
    leave_range<4>(range, ranges + kSplitSlots + block);
  }
}

// A wavefront per row, or (WIDE) a workgroup.  A score that is not finite (an infinity's parts give NaN) is computed as the dot product itself, and so are all where
// the product has found that parts do not hold the operands' entries: eight scores side by side, by eight lanes each, four vectors of both operands in
// flight, bound by the rows' way from L2 as the gather kernel is.  Us a call, 2160 x 1449 at 81 %, k = 221 / 986 x 10230 at 85 %, k = 1049 / 11008 x 4096 at 90 %,
// k = 256: gather kernel 39 / 608 / 204, by parts 32 / 166 / 228; all computed here 58 / 714 / 306 (one score at a time by the whole wavefront: 228 / 5765 / 873); an
// infinity in lhs, so one row of them, 49 / 386 / 230 (287 / 6436 / 673).
constexpr int kDotLanes = 8, kDots = kWave / kDotLanes;
__device__ __forceinline__ float dot_product(const SplitSample& s, int row, int col, int part) {
  typedef float any4 __attribute__((ext_vector_type(4), aligned(4)));
  float sums[4] = {0.f, 0.f, 0.f, 0.f};   // (short chains: the gather kernel's accuracy)
  for (int z = 0; z < s.batch; ++z) {
    const float* l = s.lhs + ((size_t)z * s.m + row) * s.k;
    const float* r = s.rhs + ((size_t)z * s.n + col) * s.k;
    int i = part * 4;
    for (; i + 3 * kDotLanes * 4 + 4 <= s.k; i += 4 * kDotLanes * 4) {
      any4 x[4], y[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) x[u] = *reinterpret_cast<const any4*>(l + i + u * kDotLanes * 4), y[u] = *reinterpret_cast<const any4*>(r + i + u * kDotLanes * 4);
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) sums[e] = fmaf(x[u][e], y[u][e], sums[e]);
    }
    for (; i < s.k; i += kDotLanes * 4) {
      if (i + 4 <= s.k) {
        const any4 x = *reinterpret_cast<const any4*>(l + i), y = *reinterpret_cast<const any4*>(r + i);
#pragma unroll
        for (int e = 0; e < 4; ++e) sums[e] = fmaf(x[e], y[e], sums[e]);
      } else {
        for (int e = i; e < s.k; ++e) sums[0] = fmaf(l[e], r[e], sums[0]);
      }
    }
  }
  float sum = (sums[0] + sums[1]) + (sums[2] + sums[3]);
#pragma unroll
  for (int d = kDotLanes / 2; d; d >>= 1) sum += __shfl_xor(sum, d);
  return sum;
}

template <bool WIDE>
__global__ __launch_bounds__(256) void split_sample_kernel(SplitSample s) {
  const int wave = uniform(threadIdx.x >> 6), lane = lane_id();
  const int row = WIDE ? (int)blockIdx.x : (int)blockIdx.x * 4 + wave;
  if (row >= s.m) return;
  const int start = s.row_offsets[row], end = s.row_offsets[row + 1];
  const bool all = s.ranges[kSplitVerdict] == 0;   // (uniform)
  const float* scores = s.scores + (size_t)row * s.ld;
  for (int j0 = start + (WIDE ? wave * kWave : 0); j0 < end; j0 += WIDE ? 4 * kWave : kWave) {
    const int j = min(j0 + lane, end - 1), col = s.cols[j];
    float x = 0.f;
    if (!all) {
      x = scores[col];
      for (int part = 1; part < s.parts; ++part) x += scores[(size_t)part * s.stride_part + col];
    }
    const bool mine = j0 + lane < end && (all || magnitude(x) >= 0x7f800000u);
    unsigned long long odd = __ballot(mine);
    const int place = __popcll(odd & ((1ull << lane) - 1));   // of mine among them
    for (int first = 0; odd; first += kDots) {
      int src = __ffsll(odd) - 1;   // of the eight lanes that I am of: theirs is the next one, the one after ..., or the first again
#pragma unroll
      for (int d = 0; d < kDots; ++d) {
        if (odd && lane / kDotLanes == d) src = __ffsll(odd) - 1;
        odd &= odd - 1;
      }
      const float sum = __shfl(dot_product(s, row, __shfl(col, src), lane % kDotLanes), (place - first) * kDotLanes & (kWave - 1));
      if (mine && place >= first && place < first + kDots) x = sum;
    }
    if (j0 + lane < end) s.out[j] = x;
  }
}

// ---- product ------------------------------------------------------------------------------------------------------
constexpr int kSplitTile = 128, kSplitStages = 3, kSplitFlush = 8;

template <bool TRANS_B>
__global__ __launch_bounds__(256, 1) void gemm_split_kernel(SplitParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int b = blockIdx.x;
  const int part = (b >> 3) % p.parts, slot = ((b >> 3) / p.parts) * kXcds + (b & 7);   // (a tile's parts on one XCD)
  int tile_m, tile_n;
  if (!xcd_tile(slot, p.tiles_m, p.tiles_n, tile_m, tile_n)) return;   // uniform per block
  gemm_split_tile<TRANS_B, 2, 2, kSplitStages, kSplitFlush>(p, tile_m, tile_n, blockIdx.y, part, smem);
}

// Rounds of workgroups (32 on an XCD at a time, which gets whole tiles: 81 tiles in three parts are 33 for one of them, a second round) times the steps
// of each, plus what a workgroup takes besides (8 steps) and the sums of the parts.
double split_rounds(int M, int N, int batch, int parts) {
  return std::ceil((double)ceil_div((long long)ceil_div(M, kSplitTile) * ceil_div(N, kSplitTile), kXcds) * batch * parts / 32.0);
}
double split_steps(int M, int N, int K, int batch, int parts) {
  return split_rounds(M, N, batch, parts) * (ceil_div(K / 32, parts) + 8) + (parts > 1 ? 1 + (parts + 1.0) * M * N * batch * 4 / 4e12 / 1.1e-6 : 0);
}

template <bool TRANS_B>
int launch_product(const SplitParams& p, int batch, hipStream_t stream) {
  auto kern = gemm_split_kernel<TRANS_B>;
  constexpr int lds = gemm_split_lds_bytes<2, 2, kSplitStages>();
  static thread_local bool raised = false;   // per instantiation
  if (!raised) {
    if (int rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds), "hipFuncSetAttribute(LDS size)"))
      return rc;
    raised = true;
  }
  const int per_xcd = ceil_div((long long)p.tiles_m * p.tiles_n, kXcds);
  note_kernel("gemm_split_kernel<%s> (fp32 by three bf16 parts, %d x %d tiles, K in %d parts)", TRANS_B ? "B(N,K)" : "B(K,N)", kSplitTile, kSplitTile, p.parts);
  hipLaunchKernelGGL(kern, dim3(per_xcd * kXcds * p.parts, batch), dim3(256), lds, stream, p);
  return check_hip(hipGetLastError(), "gemm (fp32 by parts) launch");
}

template <typename First>
int launch_operands(const First& a, int blocks_a, const SplitDense& b, unsigned* ranges, hipStream_t stream) {
  const int blocks_b = split_dense_blocks(b);
  note_kernel("split_operands_kernel");
  hipLaunchKernelGGL(split_operands_kernel<First>, dim3(blocks_a + blocks_b), dim3(256), 0, stream, a, b, ranges, blocks_b);
  return check_hip(hipGetLastError(), "parts of the operands, launch");
}

}  // namespace

int gemm_split_parts(int M, int N, int K, int batch) {
  const int steps = K / 32;
  int best = 1;
  for (int parts = 2; parts <= 8; ++parts) {
    const int per = ceil_div(steps, parts);
    if (per < 4 || (parts - 1) * per >= steps) continue;   // (every part has a step)
    if ((double)parts * M * N * batch * 4 > 256e6) continue;
    if (split_steps(M, N, K, batch, parts) < split_steps(M, N, K, batch, best)) best = parts;
  }
  return best;
}
double gemm_split_seconds(int M, int N, int K, int batch) {
  const int parts = gemm_split_parts(M, N, K, batch);
  return 1.1e-6 * split_rounds(M, N, batch, parts) * (ceil_div(K / 32, parts) + 8);
}

int gemm_split(const SplitParams& given, bool trans_b, int batch, hipStream_t stream) {
  SplitParams p = given;
  p.tiles_m = ceil_div(p.M, kSplitTile);
  p.tiles_n = ceil_div(p.N, kSplitTile);
  const int steps = p.K / 32, per = p.parts > 0 ? ceil_div(steps, p.parts) : 0;
  IEX_REQUIRE(p.parts > 0 && (p.parts - 1) * per < steps && p.K > 0 && p.K % 32 == 0 && p.lda % 8 == 0 && p.ldb % 8 == 0 && (p.parts == 1 || (p.stride_part > 0 && !p.row_bias && !p.relu)), IEX_ERR_STATE,
              "gemm (fp32 by parts): K=%d in %d parts, strides %d and %d", p.K, p.parts, p.lda, p.ldb);
  return trans_b ? launch_product<true>(p, batch, stream) : launch_product<false>(p, batch, stream);
}

int split_dense_blocks(const SplitDense& s) {
  const long long chunks = (long long)s.batch * s.dst_rows * (s.dst_cols / 8);
  return (int)std::min<long long>(kSplitSlots, (chunks + 255) / 256);
}
int split_sparse_blocks(const SplitSparse& s) { return std::min(kSplitSparseSlots, s.m); }
int launch_split_operands(const SplitSparse& a, const SplitDense& b, unsigned* ranges, hipStream_t stream) {
  return launch_operands(a, split_sparse_blocks(a), b, ranges, stream);
}
int launch_split_operands(const SplitDense& a, const SplitDense& b, unsigned* ranges, hipStream_t stream) {
  return launch_operands(a, split_dense_blocks(a), b, ranges, stream);
}
int launch_split_operand(const SplitDense& b, unsigned* ranges, hipStream_t stream) { return launch_operands(b, 0, b, ranges, stream); }
int launch_split_sample(const SplitSample& s, hipStream_t stream) {
  note_kernel("split_sample_kernel");
  if (s.wide) hipLaunchKernelGGL(split_sample_kernel<true>, dim3(s.m), dim3(256), 0, stream, s);
  else hipLaunchKernelGGL(split_sample_kernel<false>, dim3(ceil_div(s.m, 4)), dim3(256), 0, stream, s);
  return check_hip(hipGetLastError(), "sampling launch");
}

}  // namespace iex
