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
// tile does not compute vectors that hardly exist, nonzeros wait in registers (many per row: come through scalar loads), and nothing
// in the loop waits for stores.  384 x 784 x 784, k = 64, 6.4 nonzeros per row, fp32: 200 us (944 MB; a plain
// fill of them takes 139); rows that are no whole lines: spmm_smallk_lines_tile; 384 x 785 x 785 in fp16: 156.
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

// The rows r_begin .. of a wavefront: begin(), then one(place, value) or two(places, values) over a row's nonzeros in order, then end(row);
// place = the nonzero's column times ROW_BYTES.  Nonzeros are loaded one per lane, 512 of them at a time (16-bit values: 64, which
// measured the same), and handed out with v_readlane: the memory system is busy with stores, a load takes microseconds there, and waiting for it means waiting for all
// stores before it, too.  (Scalar loads, eight nonzeros at a time, the next row's in flight: waiting for an LDS read or for this row's eight is
// waiting for them as well, so every row paid their way to memory: 62 % of the wavefronts' time on 384 x 785 x 785, 262 us where
// this takes 219; rows of whole vectors 2 - 7 % less, too.)
template <int ROW_BYTES, typename T, typename IT, typename Begin, typename One, typename Two, typename End>
__device__ __forceinline__ void smallk_walk_rows(const SpmmParams& p, const T* __restrict__ values, int r_begin, int r_end, int lane, Begin begin, One one, Two two,
                                                 End end) {
  constexpr int kSmallkChunks = sizeof(T) == 4 ? 8 : 1;
  const IT* __restrict__ cols = static_cast<const IT*>(p.cols);
  int place[kSmallkChunks];    // of nonzeros held + 64 i + lane, i = 0 ..
  float value[kSmallkChunks];
  int held = 0, chunks = 0;    // chunks: how many of them are still to come, the current one included
  for (int g0 = r_begin; g0 < r_end; g0 += kWave - 1) {
    // offsets of up to 63 rows: lane l holds row_offsets[g0 + l]
    const int rows = min(kWave - 1, r_end - g0);
    const int off = p.row_offsets[min(g0 + lane, p.m)];
    int s = bcast_i(off, 0);
    for (int i = 0; i < rows; ++i) {
      const int e = bcast_i(off, i + 1);
      begin();
      for (int j = s; j < e;) {
        if (chunks == 0 || j - held >= kWave) {   // (uniform)
          if (chunks > 1) {
            --chunks;
            held += kWave;
#pragma unroll
            for (int q = 0; q + 1 < kSmallkChunks; ++q) place[q] = place[q + 1], value[q] = value[q + 1];
          } else {
            chunks = kSmallkChunks;
            held = j;
#pragma unroll
            for (int q = 0; q < kSmallkChunks; ++q) {
              const int idx = min(j + q * kWave + lane, p.nnz - 1);
              place[q] = (int)cols[idx];
              value[q] = elem<T>::to_float(values[idx]);
            }
#pragma unroll
            for (int q = 0; q < kSmallkChunks; ++q) place[q] *= ROW_BYTES;
          }
        }
        // the row's nonzeros that the current chunk holds, two at a time
        const int tl = min(e, held + kWave) - held;
        int t = j - held;
        for (; t + 2 <= tl; t += 2) two(bcast_i(place[0], t), bcast_i(place[0], t + 1), bcast_f(value[0], t), bcast_f(value[0], t + 1));
        if (t < tl) one(bcast_i(place[0], t), bcast_f(value[0], t));
        j = held + tl;
      }
      s = e;
      end(g0 + i);
    }
  }
}

// The same for fp32 values and int32 columns through scalar loads, eight nonzeros at a time, the first eight of the next row fetched while this
// row's are worked on: uniform and ready as operands, two instructions a nonzero less.  For rows of more than kSmallkScalarRows nonzeros, which
// are bound by instructions (us, held in registers / by scalar loads: 384 x 785 x 785, k = 64, 19 per row 411 / 400, 300 x 500 x 500, k = 128, 38
// per row 296 / 281; but k = 128, 13 per row 372 / 390, and 24 x 3136 x 3136 332 / 353).
constexpr int kSmallkScalarRows = 16;
template <int ROW_BYTES, typename Begin, typename One, typename Two, typename End>
__device__ __forceinline__ void smallk_walk_rows_scalar(const SpmmParams& p, const float* values, int r_begin, int r_end, int lane, Begin begin, One one, Two two,
                                                        End end) {
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
  for (int g0 = r_begin; g0 < r_end; g0 += kWave - 1) {
    const int rows = min(kWave - 1, r_end - g0);
    const int off = p.row_offsets[min(g0 + lane, p.m)];
    int s = bcast_i(off, 0);
    if (s + 8 <= p.nnz) {
      next_c = *reinterpret_cast<const_i32x8*>(scalar_cols + s);
      next_v = *reinterpret_cast<const_f32x8*>(scalar_vals + s);
    }
    for (int i = 0; i < rows; ++i) {
      const int e = bcast_i(off, i + 1);
      begin();
      i32x8 c8 = next_c;
      f32x8 v8 = next_v;
      if (i + 1 < rows && e + 8 <= p.nnz) {
        next_c = *reinterpret_cast<const_i32x8*>(scalar_cols + e);
        next_v = *reinterpret_cast<const_f32x8*>(scalar_vals + e);
      }
      for (int j = s; j < e; j += 8) {
        if (j + 8 > p.nnz) {   // the last few of the pattern
          for (int t = j; t < e; ++t) one(scalar_cols[t] * ROW_BYTES, scalar_vals[t]);
          break;
        }
        if (j > s) {
          c8 = *reinterpret_cast<const_i32x8*>(scalar_cols + j);
          v8 = *reinterpret_cast<const_f32x8*>(scalar_vals + j);
        }
        const int here = e - j;
#pragma unroll
        for (int t = 0; t < 8; t += 2) {
          if (here >= t + 2) two(c8[t] * ROW_BYTES, c8[t + 1] * ROW_BYTES, v8[t], v8[t + 1]);
          else if (here == t + 1) one(c8[t] * ROW_BYTES, v8[t]);
        }
      }
      s = e;
      end(g0 + i);
    }
  }
}

// PLAIN: no bias, ReLU or accumulation.  (A load that a row's sums may depend on makes the compiler wait, row by row, for
// everything in flight, the last row's stores included.)
template <typename T, typename IT, int VEC, bool RAGGED, int WAVES, int NV, bool SINGLE, bool PLAIN, bool SCALAR>
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
  float acc[NV][VEC], acc1 = 0.f;
  auto clear = [&]() {
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int u = 0; u < VEC; ++u) acc[v][u] = 0.f;
    acc1 = 0.f;
  };
  auto finish = [&](int row) {
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
  };
  auto one = [&](int at, float x) { add_one(acc, acc1, at, x); };
  auto two = [&](int at_a, int at_b, float xa, float xb) { add_two(acc, acc1, at_a, at_b, xa, xb); };
  if constexpr (SCALAR) smallk_walk_rows_scalar<ROW_BYTES>(p, values, r_begin, r_end, lane, clear, one, two, finish);
  else smallk_walk_rows<ROW_BYTES, T, IT>(p, values, r_begin, r_end, lane, clear, one, two, finish);
}

// MOST vectors per lane in every tile but the last.
// SCALAR: nonzeros through scalar loads (fp32 values, int32 columns).
template <typename T, typename IT, int VEC, bool RAGGED, int WAVES, int MOST, bool PLAIN, bool SCALAR>
__device__ __forceinline__ void spmm_smallk_block(const SpmmParams& p, int rows_per_wave, int bx, int by, int bz, unsigned char* smem) {
  const SmallkTiles t = smallk_tiles(p.n, MOST, VEC);
  const int base = by * (MOST * kWave * VEC);
  if (by + 1 < t.tiles || (t.nv == MOST && !t.single)) return spmm_smallk_tile<T, IT, VEC, RAGGED, WAVES, MOST, false, PLAIN, SCALAR>(p, rows_per_wave, bx, base, bz, smem);
  if (t.nv == MOST) return spmm_smallk_tile<T, IT, VEC, RAGGED, WAVES, MOST, true, PLAIN, SCALAR>(p, rows_per_wave, bx, base, bz, smem);
  if constexpr (MOST == 2) {
    if (t.single) return spmm_smallk_tile<T, IT, VEC, RAGGED, WAVES, 1, true, PLAIN, SCALAR>(p, rows_per_wave, bx, base, bz, smem);
    return spmm_smallk_tile<T, IT, VEC, RAGGED, WAVES, 1, false, PLAIN, SCALAR>(p, rows_per_wave, bx, base, bz, smem);
  }
}

// ---- rows that do not start at whole lines ---------------------------------------------------------------------
// fp32 rows whose length is no multiple of 64 bytes: wherever columns are cut, a line (128 bytes) at a cut, and every line that
// holds one row's end and the next one's start, is written in part by two workgroups, at different times, through different
// L2s, and such lines cost a multiple of whole ones.  So every line is written by one wavefront: a middle tile has, of every row,
// `width` columns from the row's first whole line on (column h, 0 .. 31, another one in every row), and the last tile has
// both edges, the columns before h and those behind the middle tiles: always n - tiles * width of them, and a row's end and
// the next row's start, the two parts of one line, follow each other in one wavefront's stores.  Tiles begin at any column,
// so a lane has columns 64 apart, one dword of LDS each.  The L2 has to put lines together: no streaming hint.
// 384 x (785 x 64 at 90 %) x 785: 295 -> 219 us.  Stores alone (the same kernel without its sums): two tiles cut at column 512 with /
// without the streaming hint 299 / 273, cut at whole lines 248 / 247, whole rows per workgroup 250 / 190 (64 rows of 785 floats are more than
// an LDS holds), lines owned by one wavefront 241 / 184; rows of 784, half lines, 189 / 219 and whole rows 197 / 181.
struct SmallkLines { int tiles, width, rest; };   // middle tiles, their columns (a multiple of 64), columns of the last tile (0: does not apply)
constexpr int kSmallkLineMost = 512;              // columns of a tile: 8 per lane
inline SmallkLines smallk_lines(int n, int k) {
  const int room = 160 * 1024 / 4 / k - 32, most = room < kSmallkLineMost ? room / 64 * 64 : kSmallkLineMost;
  if (most < 128) return SmallkLines{0, 0, 0};
  for (int t = (n + most - 1) / most - 1; t < 64; ++t) {
    if (t == 0) return SmallkLines{0, 64, n};
    for (int w = (n / (t + 1) + 63) / 64 * 64; w >= 128; w -= 64) {   // (about as wide as the rest)
      const int rest = n - t * w;
      if (w <= most && rest >= 31 && rest <= most) return SmallkLines{t, w, rest};
    }
  }
  return SmallkLines{0, 0, 0};
}
inline int smallk_lines_lds(const SmallkLines& t, int k) { return k * ((((t.tiles && t.width > t.rest ? t.width : t.rest) + 63) / 64 * 64) + 32) * 4; }

// `cols` columns (J per lane) of the rows: from column first + h on, or (EDGES) those before h and those from first + h on.
template <int WAVES, int J, bool EDGES>
__device__ __forceinline__ void spmm_smallk_lines_tile(const SpmmParams& p, int rows_per_wave, int bx, int first, int cols, int z, unsigned char* smem) {
  constexpr int ROW_BYTES = (J * kWave + 32) * 4;   // of a dense row's slice: columns first .. (EDGES: 0 .. 31, then first ..)
  const int lane = lane_id(), wave = uniform(threadIdx.x >> 6);
  const float* __restrict__ dense = static_cast<const float*>(p.dense) + (size_t)z * p.k * p.n;
  for (int kr = wave; kr < p.k; kr += WAVES) {
#pragma unroll
    for (int j = 0; j <= J; ++j) {
      const int i = j * kWave + lane, c = EDGES ? (i < 32 ? i : first + i - 32) : first + i;
      if (j < J || lane < 32) *reinterpret_cast<float*>(smem + kr * ROW_BYTES + i * 4) = dense[(size_t)kr * p.n + min(c, p.n - 1)];
    }
  }
  __syncthreads();
  const float* __restrict__ values = static_cast<const float*>(p.values) + (p.per_batch_values ? (size_t)z * p.nnz : (size_t)0);
  const int r_begin = min(p.m, (bx * WAVES + wave) * rows_per_wave), r_end = min(p.m, r_begin + rows_per_wave);
  float* __restrict__ out = static_cast<float*>(p.out) + (size_t)z * p.m * p.n;
  // the row's first element among the 32 of its line
  unsigned at = (unsigned)((reinterpret_cast<uintptr_t>(out) >> 2) + (size_t)r_begin * p.n);
  float acc[J];
  const unsigned char *mine0 = nullptr, *mine = nullptr;   // column 0's and (64 j behind) the others' place in a dense row's slice
  int h = 0;
  smallk_walk_rows<ROW_BYTES, float, int>(
      p, values, r_begin, r_end, lane,
      [&]() {
        h = (int)(0u - at) & 31;
        at += p.n;
        mine = smem + (EDGES ? 32 + lane : h + lane) * 4;
        mine0 = EDGES && lane < h ? smem + lane * 4 : mine;
#pragma unroll
        for (int j = 0; j < J; ++j) acc[j] = 0.f;
      },
      [&](int row, float x) {
        acc[0] = fmaf(x, *reinterpret_cast<const float*>(mine0 + row), acc[0]);
#pragma unroll
        for (int j = 1; j < J; ++j) acc[j] = fmaf(x, *reinterpret_cast<const float*>(mine + row + j * (kWave * 4)), acc[j]);
      },
      [&](int ra, int rb, float xa, float xb) {
        float a[J], b[J];
        a[0] = *reinterpret_cast<const float*>(mine0 + ra);
        b[0] = *reinterpret_cast<const float*>(mine0 + rb);
#pragma unroll
        for (int j = 1; j < J; ++j) {
          a[j] = *reinterpret_cast<const float*>(mine + ra + j * (kWave * 4));
          b[j] = *reinterpret_cast<const float*>(mine + rb + j * (kWave * 4));
        }
#pragma unroll
        for (int j = 0; j < J; ++j) acc[j] = fmaf(xb, b[j], fmaf(xa, a[j], acc[j]));
      },
      [&](int row) {
        float* __restrict__ to = out + (size_t)row * p.n;
        const int c = first + lane + (EDGES ? 0 : h);
        const int c0 = EDGES && lane < h ? lane : c;
        if (J > 1 || lane < cols) to[c0] = acc[0];
#pragma unroll
        for (int j = 1; j < J; ++j)
          if (!EDGES || j + 1 < J || j * kWave + lane < cols) to[c + j * kWave] = acc[j];
      });
}

template <int WAVES>
__device__ __forceinline__ void spmm_smallk_lines_block(const SpmmParams& p, const SmallkLines& t, int rows_per_wave, int bx, int by, int bz, unsigned char* smem) {
  auto middle = [&](auto j) { spmm_smallk_lines_tile<WAVES, decltype(j)::value, false>(p, rows_per_wave, bx, by * t.width, t.width, bz, smem); };
  auto edges = [&](auto j) { spmm_smallk_lines_tile<WAVES, decltype(j)::value, true>(p, rows_per_wave, bx, t.tiles * t.width, t.rest, bz, smem); };
  auto by_width = [](int j, auto run) {   // (uniform)
    if (j <= 1) run(std::integral_constant<int, 1>{});
    else if (j == 2) run(std::integral_constant<int, 2>{});
    else if (j == 3) run(std::integral_constant<int, 3>{});
    else if (j == 4) run(std::integral_constant<int, 4>{});
    else if (j == 5) run(std::integral_constant<int, 5>{});
    else if (j == 6) run(std::integral_constant<int, 6>{});
    else if (j == 7) run(std::integral_constant<int, 7>{});
    else run(std::integral_constant<int, 8>{});
  };
  if (by < t.tiles) by_width(t.width / kWave, middle);
  else by_width((t.rest + kWave - 1) / kWave, edges);
}

}  // namespace iex
