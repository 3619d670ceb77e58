// Host side of the two-of-four path (spmm_two_four_device.cuh): laying a sparse 16-bit weight out once, and products with
// what was laid out.  A form is of one kind: the dense form of the weight, or pairs and spill in panels of 128, 192 or 256 rows.
#include "spmm_two_four_device.cuh"

namespace iex {
double spmm_seconds(int m, int k, int n, int nonzeros);   // spmm.hip
namespace {

inline bool two_four_kind(int kind) { return kind == 128 || kind == 192 || kind == 256; }

template <bool BF16, int WM>
__global__ __launch_bounds__(512, 1) void two_four_kernel(GemmParams p, TwoFourOperand f) {
  extern __shared__ __align__(16) unsigned char smem[];
  int tile_m, tile_n;
  if (!xcd_tile(blockIdx.x, p.tiles_m, p.tiles_n, tile_m, tile_n)) return;  // uniform per block
  two_four_tile<BF16, WM>(p, f, tile_m, tile_n, smem);
}

template <typename Kernel>
int allow_lds(Kernel kernel, int bytes, bool& raised) {
  if (raised) return 0;
  if (int rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes), "hipFuncSetAttribute(LDS size)"))
    return rc;
  raised = true;
  return 0;
}

template <bool BF16, int WM>
int launch_product(GemmParams p, const TwoFourOperand& f, hipStream_t stream) {
  constexpr int BM = 64 * WM, lds = two_four_lds_bytes(BM);
  auto kern = two_four_kernel<BF16, WM>;
  static thread_local bool raised = false;   // per instantiation
  if (int rc = allow_lds(kern, lds, raised)) return rc;
  p.tiles_m = ceil_div(p.M, BM);
  p.tiles_n = ceil_div(p.N, kTwoFourBN);
  const int per_xcd = ceil_div((long long)p.tiles_m * p.tiles_n, kXcds);
  note_kernel("two_four_kernel<%s> (%d x %d tiles)", BF16 ? "bf16" : "f16", BM, kTwoFourBN);
  hipLaunchKernelGGL(kern, dim3(per_xcd * kXcds), dim3(512), lds, stream, p, f);
  return check_hip(hipGetLastError(), "two-of-four product launch");
}

template <typename IT>
int launch_marks(int m, int k, const int* row_offsets, const void* cols, unsigned* marks, hipStream_t stream) {
  const int words = ceil_div(k, 32);
  note_kernel("two_four_marks_kernel<%s>", type_name<IT>());
  hipLaunchKernelGGL((two_four_marks_kernel<IT>), dim3(ceil_div(m, 32)), dim3(kTwoFourThreads), words * (int)sizeof(unsigned), stream, m, k, row_offsets,
                     static_cast<const IT*>(cols), words, marks);
  return check_hip(hipGetLastError(), "two-of-four marks launch");
}

template <typename IT>
int launch_form(const TwoFourForm& f, int m, int k, const int* row_offsets, const void* cols, const void* values, unsigned char* form, unsigned* marks,
                hipStream_t stream) {
  if (int rc = launch_marks<IT>(m, k, row_offsets, cols, marks, stream)) return rc;
  const TwoFourSource s{m, k, row_offsets, cols, static_cast<const uint16_t*>(values)};
  const TwoFourTarget t{form, reinterpret_cast<int*>(form + f.counts_at), reinterpret_cast<unsigned*>(form + f.lists_at), reinterpret_cast<uint2*>(form + f.ranks_at),
                        f.bm, f.phases, f.spill_phases, f.list_room, f.words, f.block, f.panel};
  note_kernel("two_four_rank_kernel");
  hipLaunchKernelGGL(two_four_rank_kernel, dim3(f.panels * 2), dim3(256), 0, stream, t, marks, ceil_div(m, 32));
  const int rows = two_four_rows(k), lds = two_four_rows_lds_bytes(rows, f.phases);
  auto kern = two_four_form_kernel<IT>;
  static thread_local bool raised = false;   // per instantiation
  if (int rc = allow_lds(kern, 80 * 1024, raised)) return rc;
  note_kernel("two_four_form_kernel<%s>", type_name<IT>());
  hipLaunchKernelGGL(kern, dim3(f.panels * f.bm / rows), dim3(kTwoFourRowThreads), lds, stream, s, t, rows);
  return check_hip(hipGetLastError(), "two-of-four form launch");
}

inline bool form_shape_fits(int kind, int m, int k) {
  if (m <= 0 || k <= 0) return false;
  if (kind == 0) return (long long)m * round8(k) < (1ll << 31);
  return two_four_kind(kind) && k <= kTwoFourMaxK && (long long)ceil_div(m, kind) * kind * round8(k) < (1ll << 31);
}

// Seconds of a product with a two-of-four form: rounds of workgroups (a last round with a share f of the CUs at work as in gemm.hip:
// 0.65 + 0.35 f) of `steps` steps, and launch, prologue and epilogue.  Steps measured at 4096 x 4096 x 8192 (256 rows: 128 steps in
// 139 us, 192: 169), 4096 x 11008 x 2048 at 90 % (128: 194 steps in 128).  With these and gemm_seconds the choice was the fastest kind or within 8 %
// of it at 70 of 74 points of m x k = 512^2 .. 11008 x 4096, 2:4 / 80 % / 90 %, n = 64 .. 8192 (us, dense / 128 / 192 / 256 rows: 2:4 4096^2,
// n = 1024 35 / 38 / 40 / 45, 2048 61 / 46 / 49 / 53, 4096 99 / 88 / 93 / 70, 8192 195 / 180 / 155 / 136; 2048^2, n = 8192 53 / 52 / 54 / 40;
// 90 % 11008 x 4096, n = 2048 148 / 145 / 121 / 144; 80 % 11008 x 4096, n = 2048 152 / 238 / 205 / 236).
double two_four_seconds(int kind, int m, int n, double steps) {
  const double tiles = (double)ceil_div(m, kind) * ceil_div(n, kTwoFourBN), full = std::floor(tiles / 256), rest = tiles - full * 256;
  const double rounds = full + (rest > 0 ? 0.65 + 0.35 * rest / 256 : 0.0);
  return 6e-6 + rounds * (4e-6 + steps * (kind == 256 ? 0.98e-6 : kind == 192 ? 0.80e-6 : 0.63e-6));
}

// Seconds of laying a form out (us measured: 4096^2 dense 8.5 at 10 % / 12.5 at 2:4, two-of-four 19 / 31; 11008 x 4096 18.4 / 28.3, 31 / 56; 4096 x
// 11008 19.6 / 32.7, 50 / 69; 1024^2, 2:4 4.5, 12; the longer rows of the last one leave a workgroup of the two-of-four form two of them).
double layout_seconds(int kind, int m, int k, int nonzeros) {
  const double cells = (double)m * k;
  return kind == 0 ? 3.5e-6 + cells * 3.2e-13 + nonzeros * 4.5e-13 : 10e-6 + cells * (two_four_rows(k) <= 2 ? 6e-13 : 3.5e-13) + nonzeros * 1.4e-12;
}

}  // namespace
}  // namespace iex

using namespace iex;

extern "C" size_t iex_form_scratch_bytes(int m, int k) {
  return m > 0 && k > 0 && k <= kTwoFourMaxK ? round256((size_t)ceil_div(m, 32) * ceil_div(k, 32) * sizeof(unsigned)) : 0;
}

extern "C" int iex_form_measure(int itype, int m, int k, int nonzeros, const int* row_offsets, const void* column_indices, void* scratch, size_t scratch_bytes,
                                int* spill_phases, void* stream) {
  trail_reset();
  IEX_REQUIRE(m > 0 && k > 0 && k <= kTwoFourMaxK && nonzeros >= 0, IEX_ERR_BAD_ARGUMENT, "form: m and k must be positive, k at most %d (m=%d k=%d nnz=%d)", kTwoFourMaxK, m, k, nonzeros);
  IEX_REQUIRE(itype == IEX_I32 || (itype == IEX_I16 && k <= 32768), IEX_ERR_BAD_ARGUMENT, "form: column indices must be int32, or int16 for k <= 32768");
  IEX_REQUIRE(row_offsets && spill_phases && (column_indices || nonzeros == 0) && scratch, IEX_ERR_BAD_ARGUMENT, "form: null pointer argument");
  IEX_REQUIRE(aligned(scratch, 16) && scratch_bytes >= iex_form_scratch_bytes(m, k), IEX_ERR_BAD_ARGUMENT, "form: measuring needs %zu bytes of scratch memory", iex_form_scratch_bytes(m, k));
  if (nonzeros < 3) return 0;   // (a spilled entry is a row's third at least)
  hipStream_t s = static_cast<hipStream_t>(stream);
  unsigned* marks = static_cast<unsigned*>(scratch);
  if (int rc = itype == IEX_I16 ? launch_marks<short>(m, k, row_offsets, column_indices, marks, s) : launch_marks<int>(m, k, row_offsets, column_indices, marks, s)) return rc;
  note_kernel("two_four_measure_kernel");
  hipLaunchKernelGGL(two_four_measure_kernel, dim3(ceil_div(m, 64) + ceil_div(m, 96) + ceil_div(m, 128)), dim3(256), 0, s, m, ceil_div(k, 32), marks, spill_phases);
  return check_hip(hipGetLastError(), "two-of-four measure launch");
}

extern "C" size_t iex_form_bytes(int kind, int m, int k, int spill_phases) {
  if (!form_shape_fits(kind, m, k) || spill_phases < 0) return 0;
  return kind == 0 ? round256((size_t)m * round8(k) * 2) : two_four_form(m, k, kind, std::min(spill_phases, two_four_spill_room(k))).bytes;
}

extern "C" int iex_form_build(int itype, int kind, int m, int k, int nonzeros, const int* row_offsets, const void* column_indices, const void* values, int spill_phases,
                              void* form, size_t form_bytes, void* scratch, size_t scratch_bytes, void* stream) {
  trail_reset();
  IEX_REQUIRE(form_shape_fits(kind, m, k) && spill_phases >= 0, IEX_ERR_BAD_ARGUMENT, "form: no form of kind %d for a %d x %d matrix", kind, m, k);
  IEX_REQUIRE(itype == IEX_I32 || (itype == IEX_I16 && k <= 32768), IEX_ERR_BAD_ARGUMENT, "form: column indices must be int32, or int16 for k <= 32768");
  IEX_REQUIRE(nonzeros >= 3 && nonzeros < (1 << 29), IEX_ERR_UNSUPPORTED, "form: needs three nonzeros, and fewer than 2^29 (nnz=%d)", nonzeros);
  IEX_REQUIRE(row_offsets && column_indices && values && form, IEX_ERR_BAD_ARGUMENT, "form: null pointer argument");
  IEX_REQUIRE(aligned(form, 256) && form_bytes >= iex_form_bytes(kind, m, k, spill_phases), IEX_ERR_BAD_ARGUMENT, "form: needs 256-byte aligned memory of %zu bytes",
              iex_form_bytes(kind, m, k, spill_phases));
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (kind == 0) {
    note_kernel("csr_to_dense_kernel");
    if (itype == IEX_I16) launch_csr_to_dense<short>(m, round8(k), row_offsets, column_indices, values, form, nullptr, 0, s);
    else launch_csr_to_dense<int>(m, round8(k), row_offsets, column_indices, values, form, nullptr, 0, s);
    return check_hip(hipGetLastError(), "dense form launch");
  }
  IEX_REQUIRE(scratch && aligned(scratch, 16) && scratch_bytes >= iex_form_scratch_bytes(m, k), IEX_ERR_BAD_ARGUMENT, "form: needs %zu bytes of scratch memory", iex_form_scratch_bytes(m, k));
  const TwoFourForm f = two_four_form(m, k, kind, std::min(spill_phases, two_four_spill_room(k)));
  unsigned char* at = static_cast<unsigned char*>(form);
  unsigned* marks = static_cast<unsigned*>(scratch);
  return itype == IEX_I16 ? launch_form<short>(f, m, k, row_offsets, column_indices, values, at, marks, s) : launch_form<int>(f, m, k, row_offsets, column_indices, values, at, marks, s);
}

extern "C" size_t iex_form_product_workspace_bytes(int kind, int m, int k, int n) {
  return kind == 0 && m > 0 && k > 0 && n > 0 ? gemm_auto_split_bytes(m, n, round8(k), 1) : 0;
}

extern "C" int iex_form_product(int dtype, int kind, int m, int k, int n, int spill_phases, const void* form, const void* dense, const void* aux, int aux_mode, void* out,
                                void* workspace, size_t workspace_bytes, void* stream) {
  trail_reset();
  IEX_REQUIRE(dtype == IEX_F16 || dtype == IEX_BF16, IEX_ERR_UNSUPPORTED, "form product: dtype must be fp16 or bf16");
  IEX_REQUIRE(form_shape_fits(kind, m, k) && n > 0 && spill_phases >= 0, IEX_ERR_BAD_ARGUMENT, "form product: no form of kind %d for a %d x %d matrix, or n=%d", kind, m, k, n);
  IEX_REQUIRE(n % 8 == 0 && aligned(dense, 16) && aligned(form, 256), IEX_ERR_UNSUPPORTED, "form product: n must be a multiple of 8, the dense operand 16-byte aligned, the form 256-byte aligned (n=%d)", n);
  IEX_REQUIRE(form && dense && out, IEX_ERR_BAD_ARGUMENT, "form product: null pointer argument");
  IEX_REQUIRE(!aux || aux_mode == kGemmAdd || aux_mode == kGemmTimesSilu, IEX_ERR_BAD_ARGUMENT, "form product: unknown mode %d", aux_mode);
  IEX_REQUIRE((long long)k * n < (1ll << 31) && (long long)m * n < (1ll << 31), IEX_ERR_TOO_LARGE, "form product: a dense operand exceeds 2^31 elements");
  hipStream_t s = static_cast<hipStream_t>(stream);
  GemmParams p{m, n, round8(k), form, dense, out, 0, 0, 0, 0, 0};
  p.aux = aux;
  p.aux_mode = aux ? aux_mode : 0;
  p.kb = k;
  if (kind == 0) return gemm_dispatch(dtype, 0, p, 1, s, workspace, workspace_bytes);
  p.ldb = p.ldc = n;
  p.stream_out = (double)m * n * 2 >= 128e6;
  const TwoFourForm f = two_four_form(m, k, kind, std::min(spill_phases, two_four_spill_room(k)));
  const unsigned char* at = static_cast<const unsigned char*>(form);
  const TwoFourOperand o{at, reinterpret_cast<const int*>(at + f.counts_at), reinterpret_cast<const unsigned*>(at + f.lists_at), f.phases, f.spill_phases, f.list_room, f.panel};
  const bool bf = dtype == IEX_BF16;
  if (kind == 256) return bf ? launch_product<true, 4>(p, o, s) : launch_product<false, 4>(p, o, s);
  if (kind == 192) return bf ? launch_product<true, 3>(p, o, s) : launch_product<false, 3>(p, o, s);
  return bf ? launch_product<true, 2>(p, o, s) : launch_product<false, 2>(p, o, s);
}

extern "C" int iex_form_choose(int kinds, int m, int k, int n, int nonzeros, const int* spill_phases) {
  int best = -1;
  double seconds = 1e9;
  if (m <= 0 || k <= 0 || n <= 0 || nonzeros <= 0) return best;
  // IEX_FORM_EACH_CALL: the laying out counts too.  A weight multiplied once as it is laid out: two-of-four forms pay from many columns on (us of
  // the product, layout and all, dense / two-of-four, 2:4 11008 x 4096: n = 512 80 / 94, 1024 106 / 111, 2048 187 / 167), dense ones not for few (2752 x
  // 1024, 2:4, n = 64 14.1, CSR 10.1; 4096 x 11008, 10 %, n = 64 45, CSR 24.5).  A weight of up to 2^17 cells keeps the kind, and the bits, of a call
  // with a kept form: laying it out is one launch of less than 4 us.
  const bool each_call = (kinds & IEX_FORM_EACH_CALL) && (long long)m * k > (1 << 17);
  auto layout = [&](int kind) { return each_call ? layout_seconds(kind, m, k, nonzeros) : 0.0; };
  if ((kinds & 1) && form_shape_fits(0, m, k)) best = 0, seconds = gemm_seconds(m, n, round8(k)) + layout(0);
  for (int i = 0; i < 3; ++i) {
    const int kind = 128 + 64 * i, half_panels = ceil_div(m, kind / 2);
    if (!(kinds >> (i + 1) & 1) || !form_shape_fits(kind, m, k) || !spill_phases) continue;
    const double steps = ceil_div(k, 128) * 2 + 1.1 * spill_phases[i] / half_panels;   // (a panel takes the longer of its halves)
    const double mine = two_four_seconds(kind, m, n, steps) + layout(kind);
    if (mine < 0.95 * seconds || best < 0) best = kind, seconds = mine;
  }
  double by_rows = spmm_seconds(m, k, n, nonzeros);
  // (narrow products: 250 nonzeros a ns whatever n is, 2:4 11008 x 4096, n = 8 .. 32 88 us; a near tie goes to the form, for the bits of a call)
  if (each_call) by_rows = 1.15 * std::max(by_rows, 5e-6 + nonzeros * 4e-12);
  return best >= 0 && by_rows < seconds ? -1 : best;
}
