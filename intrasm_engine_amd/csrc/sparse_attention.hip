// Host side of sparse attention over a CSR mask in one kernel (sparse_attention_device.cuh).
#include "sparse_attention_device.cuh"

namespace iex {
namespace {

// Entries of a 128 x 64 tile from which it counts as dense (fewer where only some groups of 32 rows have entries there).  A tile costs the matrix-core
// path about 1100 (16-bit) and 8200 (fp32, HD = 64) clocks of a wavefront for 32 rows, an entry on its own about 20 and 40 beside its two rows from L2.  (16
// heads x 1500 tokens, 175 scattered entries per tile, fp16: 45 us from 128 on, 30 from 224 on.  262 per tile, bf16, us from 224 / 288 / 448 on: 4 x 1000
// of 128 20.4 / 13.8 / 12.7, 32 x 1000 of 32 20.8 / 16.3 / 15.5, of 64 25.8 / 24.2 / 23.2; 327 per tile, 32 x 800 of 128 36.9 / 36.9 / 39.6;
// 655, 4 x 400 of 64 8.2 / 9.4 / 11.9.  8 x 1000, 260 per tile, fp32: 28 from 224 on, 22 from 400 on.)
inline int dense_min(int dtype) { return dtype == IEX_F32 ? 800 : 288; }
// ... and from which some launches take it for dense all the same (SparseAttentionShape::takes_either)
inline int either_min(int dtype) { return dtype == IEX_F32 ? 800 : 224; }

template <int TYPE, int HD, int QW, int KW>
int launch(const SparseAttentionParams& p, hipStream_t stream) {
  constexpr int lds = SparseAttentionShape<TYPE, HD>::lds(QW, KW);
  auto kern = sparse_attention_kernel<TYPE, HD, QW, KW>;
  if (lds > 64 * 1024) {
    static thread_local bool raised = false;  // per instantiation
    if (!raised) {
      if (int rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds),
                             "hipFuncSetAttribute(LDS size)"))
        return rc;
      raised = true;
    }
  }
  note_kernel("sparse_attention_kernel<%s, %d, %d, %d>", TYPE == 2 ? "float" : TYPE == 1 ? "bf16" : "f16", HD, QW, KW);
  hipLaunchKernelGGL(kern, dim3((unsigned)(ceil_div(p.tokens, QW * 32) * (long long)p.heads)), dim3((QW * KW + SparseAttentionShape<TYPE, HD>::extra(KW)) * kWave), lds, stream, p);
  return check_hip(hipGetLastError(), "sparse attention launch");
}

// Four wavefronts with 32 queries each share every tile they load; where that leaves the chip empty, several share 32 queries
// (as many as there is LDS for).  Us by four / by shared queries, fp16 and fp32: 64 workgroups of four (8 heads x 1000) 9.9 /
// 7.3 and 32 / 16; 128 (4 x 4096) 17.1 / 14.9 and 33 / 27; 192 (16 x 1500) 27.7 / 29.4 and 49 / 50; 288 (12 x 3000) 14.7 / 16.9
// and 34 / 29; 512 (16 x 4096) 44 / 97 and 117 / 190.  (Workgroups of two are never ahead of both.)
template <int TYPE, int HD>
int launch_wide(const SparseAttentionParams& p, hipStream_t stream) {
  if ((long long)ceil_div(p.tokens, 128) * p.heads >= (TYPE == 2 ? 320 : 160)) return launch<TYPE, HD, 4, 1>(p, stream);
  return launch<TYPE, HD, 1, HD == 128 ? 2 : 4>(p, stream);
}

template <int TYPE>
int launch_type(const SparseAttentionParams& p, int head_dim, hipStream_t stream) {
  if (head_dim == 32) return launch_wide<TYPE, 32>(p, stream);
  if (head_dim == 64) return launch_wide<TYPE, 64>(p, stream);
  return launch_wide<TYPE, 128>(p, stream);
}

}  // namespace
}  // namespace iex

extern "C" size_t iex_mask_tables_bytes(int m, int n, int nonzeros) {
  if (m <= 0 || n <= 0 || m > iex::kMaMaxTokens || n > iex::kMaMaxTokens || nonzeros <= 0) return 0;
  return iex::mask_tables_layout(m, n, nonzeros).bytes;
}

extern "C" int iex_mask_tables(int dtype, int m, int n, int nonzeros, const int* row_offsets, const int* column_indices, void* tables, size_t bytes,
                               void* stream) {
  using namespace iex;
  trail_reset();
  const size_t need = iex_mask_tables_bytes(m, n, nonzeros);
  IEX_REQUIRE(need > 0, IEX_ERR_UNSUPPORTED, "mask tables: 1 .. %d rows and columns, at least one entry (m=%d n=%d nnz=%d)", kMaMaxTokens, m, n, nonzeros);
  IEX_REQUIRE(row_offsets && column_indices, IEX_ERR_BAD_ARGUMENT, "mask tables: null pointer argument");
  IEX_REQUIRE(tables && aligned(tables, 256) && bytes >= need, IEX_ERR_BAD_ARGUMENT, "mask tables: needs 256-byte aligned memory of %zu bytes", need);
  const MaskTables t = mask_tables_layout(m, n, nonzeros);
  note_kernel("mask_tables_kernel");
  hipLaunchKernelGGL(mask_tables_kernel, dim3(t.blocks), dim3(kMtWaves * kWave), mask_tables_lds_bytes(t.tiles), static_cast<hipStream_t>(stream), m, n,
                     nonzeros, dense_min(dtype), either_min(dtype), row_offsets, column_indices, static_cast<unsigned char*>(tables));
  return check_hip(hipGetLastError(), "mask tables launch");
}

extern "C" int iex_sparse_attention_fits(int dtype, int head_dim, int tokens) {
  return (dtype == IEX_F32 || dtype == IEX_F16 || dtype == IEX_BF16) && (head_dim == 32 || head_dim == 64 || head_dim == 128) && tokens > 0 &&
         tokens <= iex::kMaMaxTokens;
}

extern "C" int iex_sparse_attention(int dtype, int heads, int tokens, int head_dim, int nonzeros, const int* row_offsets, const void* q, const void* k,
                                    const void* v, float scale, void* out, const void* tables, size_t bytes, void* stream) {
  using namespace iex;
  trail_reset();
  IEX_REQUIRE(heads >= 0 && tokens >= 0, IEX_ERR_BAD_ARGUMENT, "sparse attention: negative dimension");
  if (heads == 0 || tokens == 0) return 0;
  IEX_REQUIRE(iex_sparse_attention_fits(dtype, head_dim, tokens), IEX_ERR_UNSUPPORTED,
              "sparse attention: fp32, fp16 or bf16, heads of 32, 64 or 128, up to %d tokens (head_dim=%d tokens=%d)", kMaMaxTokens, head_dim, tokens);
  IEX_REQUIRE(row_offsets && q && k && v && out, IEX_ERR_BAD_ARGUMENT, "sparse attention: null pointer argument");
  IEX_REQUIRE(scale > 0.f, IEX_ERR_UNSUPPORTED, "sparse attention: the scale must be positive");
  IEX_REQUIRE(aligned(q, 16) && aligned(k, 16) && aligned(v, 16) && aligned(out, 16), IEX_ERR_UNSUPPORTED, "sparse attention: operands must be 16-byte aligned");
  const size_t need = iex_mask_tables_bytes(tokens, tokens, nonzeros);
  IEX_REQUIRE(need > 0 && tables && aligned(tables, 256) && bytes >= need, IEX_ERR_BAD_ARGUMENT, "sparse attention: needs the mask's tables (iex_mask_tables, same dtype)");
  IEX_REQUIRE((long long)ceil_div(tokens, 32) * heads < (1ll << 31), IEX_ERR_TOO_LARGE, "sparse attention: too many blocks of queries");
  SparseAttentionParams p{heads, tokens, nonzeros, q, k, v, out, scale * 1.44269504088896340736f, static_cast<const unsigned char*>(tables)};
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == IEX_F32) return launch_type<2>(p, head_dim, s);
  return dtype == IEX_BF16 ? launch_type<1>(p, head_dim, s) : launch_type<0>(p, head_dim, s);
}
