// CSR SpMM for a sparse operand with few columns (k <= 128) and a wide output: the products of
// sparse attention-style sweeps, a[M x K] * b[K x N] with K = 32 .. 128 and N in the thousands, where
// the output (batch * m * n elements) is the traffic that has to happen and everything else should
// stay out of its way.
//
// The row kernel spends a wavefront per (row, 64 * VEC columns): three dependent memory latencies
// (row offsets -> column indices / values -> dense row) to write one kilobyte, and every nonzero
// gathers its dense row segment from L2 although all rows of A share the same k dense rows.
// Here a workgroup of 8 or 16 wavefronts owns one tile of columns (1 or 2 vectors per lane; in the last tile the vectors that
// are left, and up to 64 columns beyond them one per lane), one batch entry and a long run of consecutive rows:
//   * the tile of the dense operand is loaded into LDS once, lane i's
//     vectors of every dense row at [row][vector][i]: the layout the gather reads;
//   * a wavefront walks its rows in natural order, so their nonzeros are one contiguous range:
//     row offsets are read 64 at a time, column indices and values 64 at a time (coalesced, one
//     per lane) and handed out with v_readlane; a nonzero is NV 128-bit LDS reads and NV * VEC FMAs;
//   * what is left per row is the store of its NV * 64 * VEC outputs, and stores do not wait.
// What bounds it besides the stores is instruction issue: per row and tile about 40 instructions whatever the row holds and 5
// per nonzero beside its FMAs.  So two vectors per lane (half as many rows to walk) are ahead wherever n exceeds one, a last
// tile does not compute vectors that hardly exist, nonzeros come through scalar loads where their types allow it, and
// nothing in the loop waits for stores.  384 x 785 x 785, k = 64, 6.4 nonzeros per row, fp32: 393 -> 299 us (946 MB; a plain
// fill of them takes 139; rows of 784, stored at aligned addresses, 223); the same in fp16: 263 -> 156.
// Accumulation is fp32, in ascending nonzero order (the order of the row kernel with one wavefront
// per row, so results are bit-equal to it); the swizzle (row_indices) is ignored: it only
// schedules.  Needs n % VEC == 0 and 16-byte aligned dense operand and output (full vectors), or
// RAGGED: any n >= VEC at element alignment -- rows then start at any element, vectors are moved with
// element-aligned 128-bit accesses, and the one lane per row whose vector would pass the row's end
// works on the last VEC elements of the row instead (shifted back), computes all of them and stores
// only the ones it owns (the others belong to the lane to its left, which stores the same values).
#pragma once
#include "spmm_device.cuh"

namespace iex {

constexpr int kSmallKMax = 128;   // dense rows (KB of LDS) a tile may have
// 8 wavefronts per workgroup up to 80 KB of LDS (two workgroups per CU), 16 beyond (one workgroup per CU only, which then
// brings the wavefronts)
constexpr int smallk_waves(int lds) { return lds <= 80 * 1024 ? 8 : 16; }

// How n columns are dealt to tiles of up to `most` vectors per lane: `tiles` of them, the last with `nv` vectors and, if
// `single`, up to 64 columns more, one per lane.
struct SmallkTiles { int tiles, nv; bool single; };
inline __host__ __device__ SmallkTiles smallk_tiles(int n, int most, int vec) {
  const int wide = kWave * vec, width = most * wide;
  SmallkTiles t;
  t.tiles = n <= width + kWave ? 1 : (n - kWave + width - 1) / width;
  const int last = n - (t.tiles - 1) * width;
  t.single = last % wide != 0 && last % wide <= kWave && last > wide;
  t.nv = t.single ? last / wide : (last + wide - 1) / wide;
  return t;
}
constexpr __host__ __device__ int smallk_row_bytes(int nv, bool single, int elem_size) { return nv * kWave * 16 + (single ? kWave * elem_size : 0); }

// PLAIN: no bias, ReLU or accumulation.  (A load that a row's sums may depend on makes the compiler wait, row by row, for
// everything in flight, the last row's stores included.)
template <typename T, typename IT, int VEC, bool RAGGED, int WAVES, int NV, bool SINGLE, bool PLAIN>
__device__ __forceinline__ void spmm_smallk_tile(const SpmmParams& p, int rows_per_wave, int bx, int base, int bz, unsigned char* smem) {
  typedef vec_t<T, VEC> V;
  constexpr int ROW_BYTES = smallk_row_bytes(NV, SINGLE, sizeof(T));   // of a dense row's slice in the tile
  const int lane = lane_id();
  const int wave = uniform(threadIdx.x >> 6);
  const int z = bz;
  int col0[NV], shift[NV];
  bool live[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int c = base + v * (kWave * VEC) + lane * VEC;
    live[v] = c < p.n;
    shift[v] = (RAGGED && live[v] && c + VEC > p.n) ? c + VEC - p.n : 0;
    col0[v] = c - shift[v];
  }
  const int col1 = base + NV * (kWave * VEC) + lane;   // this lane's single column
  const T* __restrict__ dense = static_cast<const T*>(p.dense) + (size_t)z * p.k * p.n;
  unsigned char* mine = smem + lane * 16;   // this lane's vectors of dense row 0
  const T* mine1 = reinterpret_cast<const T*>(smem + NV * (kWave * 16)) + lane;   // ... and its single column
  for (int kr = wave; kr < p.k; kr += WAVES) {
#pragma unroll
    for (int v = 0; v < NV; ++v)
      *reinterpret_cast<V*>(mine + kr * ROW_BYTES + v * (kWave * 16)) = load_vec<T, VEC, !RAGGED>(dense + (size_t)kr * p.n + min(col0[v], p.n - VEC));
    if constexpr (SINGLE)
      *reinterpret_cast<T*>(smem + kr * ROW_BYTES + NV * (kWave * 16) + lane * sizeof(T)) = dense[(size_t)kr * p.n + min(col1, p.n - 1)];
  }
  __syncthreads();

  const T* __restrict__ values = static_cast<const T*>(p.values) + (p.per_batch_values ? (size_t)z * p.nnz : (size_t)0);
  const IT* __restrict__ cols = static_cast<const IT*>(p.cols);
  // one or two nonzeros (byte offsets of their dense rows, values), their LDS reads in flight together
  auto add_one = [&](float (&acc)[NV][VEC], float& acc1, int at, float x) {
#pragma unroll
    for (int v = 0; v < NV; ++v) fma_vec<T, VEC>(acc[v], x, *reinterpret_cast<const V*>(mine + at + v * (kWave * 16)));
    if constexpr (SINGLE) acc1 = fmaf(x, elem<T>::to_float(*reinterpret_cast<const T*>(reinterpret_cast<const unsigned char*>(mine1) + at)), acc1);
  };
  auto add_two = [&](float (&acc)[NV][VEC], float& acc1, int at_a, int at_b, float xa, float xb) {
    V a[NV], b[NV];
    T a1, b1;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      a[v] = *reinterpret_cast<const V*>(mine + at_a + v * (kWave * 16));
      b[v] = *reinterpret_cast<const V*>(mine + at_b + v * (kWave * 16));
    }
    if constexpr (SINGLE) {
      a1 = *reinterpret_cast<const T*>(reinterpret_cast<const unsigned char*>(mine1) + at_a);
      b1 = *reinterpret_cast<const T*>(reinterpret_cast<const unsigned char*>(mine1) + at_b);
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      fma_vec<T, VEC>(acc[v], xa, a[v]);
      fma_vec<T, VEC>(acc[v], xb, b[v]);
    }
    if constexpr (SINGLE) acc1 = fmaf(xb, elem<T>::to_float(b1), fmaf(xa, elem<T>::to_float(a1), acc1));
  };
  const int r_begin = min(p.m, (bx * WAVES + wave) * rows_per_wave);
  const int r_end = min(p.m, r_begin + rows_per_wave);
  // fp32 values and int32 columns come through scalar loads: dword-aligned, uniform, and ready as operands
  constexpr bool kScalar = std::is_same<T, float>::value && std::is_same<IT, int>::value;
  typedef int i32x8 __attribute__((ext_vector_type(8)));
  typedef float f32x8 __attribute__((ext_vector_type(8)));
  typedef int i32x8_a4 __attribute__((ext_vector_type(8), aligned(4)));
  typedef float f32x8_a4 __attribute__((ext_vector_type(8), aligned(4)));
  typedef const __attribute__((address_space(4))) i32x8_a4 const_i32x8;   // (the constant address space: read-only while the kernel runs)
  typedef const __attribute__((address_space(4))) f32x8_a4 const_f32x8;
  const __attribute__((address_space(4))) int* scalar_cols = (const __attribute__((address_space(4))) int*)(uintptr_t)p.cols;
  const __attribute__((address_space(4))) float* scalar_vals = (const __attribute__((address_space(4))) float*)(uintptr_t)values;
  i32x8 next_c = {};
  f32x8 next_v = {};
  int cbase = -kWave;  // first nonzero held in (cc, vv); none yet
  int cc = 0;          // byte offset of its dense row in the tile
  float vv = 0.f;
  for (int g0 = r_begin; g0 < r_end; g0 += kWave - 1) {
    // offsets of up to 63 rows: lane l holds row_offsets[g0 + l]
    const int rows = min(kWave - 1, r_end - g0);
    const int off = p.row_offsets[min(g0 + lane, p.m)];
    int s = bcast_i(off, 0);
    if (kScalar && s + 8 <= p.nnz) {
      next_c = *reinterpret_cast<const_i32x8*>(scalar_cols + s);
      next_v = *reinterpret_cast<const_f32x8*>(scalar_vals + s);
    }
    for (int i = 0; i < rows; ++i) {
      const int row = g0 + i;
      const int e = bcast_i(off, i + 1);
      float acc[NV][VEC];
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int u = 0; u < VEC; ++u) acc[v][u] = 0.f;
      float acc1 = 0.f;
      if constexpr (kScalar) {
        // eight nonzeros at a time through scalar loads (counted apart from the stores: waiting for them waits for no store);
        // the first eight of the next row are fetched while this row's are worked on
        i32x8 c8 = next_c;
        f32x8 v8 = next_v;
        if (i + 1 < rows && e + 8 <= p.nnz) {
          next_c = *reinterpret_cast<const_i32x8*>(scalar_cols + e);
          next_v = *reinterpret_cast<const_f32x8*>(scalar_vals + e);
        }
        for (int j = s; j < e; j += 8) {
          if (j + 8 > p.nnz) {   // the last few of the pattern
            for (int t = j; t < e; ++t) add_one(acc, acc1, scalar_cols[t] * ROW_BYTES, scalar_vals[t]);
            break;
          }
          if (j > s) {
            c8 = *reinterpret_cast<const_i32x8*>(scalar_cols + j);
            v8 = *reinterpret_cast<const_f32x8*>(scalar_vals + j);
          }
          const int here = e - j;
#pragma unroll
          for (int t = 0; t < 8; t += 2) {
            if (here >= t + 2) {
              add_two(acc, acc1, c8[t] * ROW_BYTES, c8[t + 1] * ROW_BYTES, v8[t], v8[t + 1]);
            } else if (here == t + 1) {
              add_one(acc, acc1, c8[t] * ROW_BYTES, v8[t]);
            }
          }
        }
      } else {
        for (int j = s; j < e;) {
          if (j - cbase >= kWave) {  // (uniform) the next 64 nonzeros, one per lane
            cbase = j;
            const int idx = min(j + lane, p.nnz - 1);
            cc = (int)cols[idx] * ROW_BYTES;
            vv = elem<T>::to_float(values[idx]);
          }
          // the row's nonzeros that (cc, vv) holds, two at a time, summed in order
          const int tl = min(e, cbase + kWave) - cbase;
          int t = j - cbase;
          for (; t + 2 <= tl; t += 2) add_two(acc, acc1, bcast_i(cc, t), bcast_i(cc, t + 1), bcast_f(vv, t), bcast_f(vv, t + 1));
          if (t < tl) add_one(acc, acc1, bcast_i(cc, t), bcast_f(vv, t));
          j = cbase + tl;
        }
      }
      s = e;
      const float bias = !PLAIN && p.bias ? p.bias[row] : 0.f;
      T* __restrict__ out_row = static_cast<T*>(p.out) + ((size_t)z * p.m + row) * p.n;
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        if (!live[v]) continue;
        T* __restrict__ out = out_row + col0[v];
        if (!PLAIN && p.accumulate) {
          const V prev = load_vec<T, VEC, !RAGGED>(out);
#pragma unroll
          for (int u = 0; u < VEC; ++u) acc[v][u] += elem<T>::to_float(prev.v[u]);
        }
        V o;
#pragma unroll
        for (int u = 0; u < VEC; ++u) {
          float r = PLAIN ? acc[v][u] : acc[v][u] + bias;
          if (!PLAIN && p.relu) r = fmaxf(r, 0.f);
          o.v[u] = elem<T>::from_float(r);
        }
        if (RAGGED && shift[v] > 0) {
#pragma unroll
          for (int u = 0; u < VEC; ++u)
            if (u >= shift[v]) out[u] = o.v[u];
        } else if (p.stream_out) {
          store_vec_stream<T, VEC, !RAGGED>(out, o);  // leaves L2 to the tile loads
        } else {
          store_vec<T, VEC, !RAGGED>(out, o);
        }
      }
      if constexpr (SINGLE) {
        if (col1 < p.n) {
          float r = acc1;
          if (!PLAIN && p.accumulate) r += elem<T>::to_float(out_row[col1]);
          if (!PLAIN) r += bias;
          if (!PLAIN && p.relu) r = fmaxf(r, 0.f);
          out_row[col1] = elem<T>::from_float(r);
        }
      }
    }
  }
}

// MOST vectors per lane in every tile but the last.
template <typename T, typename IT, int VEC, bool RAGGED, int WAVES, int MOST, bool PLAIN>
__device__ __forceinline__ void spmm_smallk_block(const SpmmParams& p, int rows_per_wave, int bx, int by, int bz, unsigned char* smem) {
  const SmallkTiles t = smallk_tiles(p.n, MOST, VEC);
  const int base = by * (MOST * kWave * VEC);
  if (by + 1 < t.tiles || (t.nv == MOST && !t.single)) return spmm_smallk_tile<T, IT, VEC, RAGGED, WAVES, MOST, false, PLAIN>(p, rows_per_wave, bx, base, bz, smem);
  if (t.nv == MOST) return spmm_smallk_tile<T, IT, VEC, RAGGED, WAVES, MOST, true, PLAIN>(p, rows_per_wave, bx, base, bz, smem);
  if constexpr (MOST == 2) {
    if (t.single) return spmm_smallk_tile<T, IT, VEC, RAGGED, WAVES, 1, true, PLAIN>(p, rows_per_wave, bx, base, bz, smem);
    return spmm_smallk_tile<T, IT, VEC, RAGGED, WAVES, 1, false, PLAIN>(p, rows_per_wave, bx, base, bz, smem);
  }
}

}  // namespace iex
