// The operators' calls as native code: what stands between torch.ops.iex_ops.* (and the autograd functions built on
// them) and the C entry points of libiex_hip.so.
//
// Small products are bound by the host: 1024 x 1024 at 90 %, n = 256 runs 7 us on the GPU, and a call whose checks,
// allocation and launch are Python took 18.  So the call everybody makes -- operands that fit, a pattern that has been
// looked at before, nothing forced -- is served here; everything else (operands to refuse, with the texts of the
// checks; a pattern's first look; kernel choices forced by ops.kernel_params; plans) goes to the Python functions of
// pytorch/ops.py, which stay the one place that raises and that looks at patterns.
//
// A pattern's note (what ops._look found) is kept here as well as on the column_indices tensor object: by the tensor's
// address, with weak references to both index tensors and their version counters, so that a note never outlives its
// tensors or passes for another pattern's, and keeps no memory of theirs alive.
#include <ATen/ATen.h>
#include <ATen/hip/HIPEvent.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/library.h>

#include <array>
#include <mutex>
#include <optional>
#include <shared_mutex>
#include <unordered_map>

#include "../../../include/iex_hip.h"

namespace py = pybind11;
using at::Tensor;

namespace {

// ---- the Python side -----------------------------------------------------------------------------------------
// (leaked on purpose: they are used until the interpreter ends)
py::object* python_ops = nullptr;   // the functions of pytorch/ops.py by operator name

thread_local bool forced = false;   // an ops.kernel_params block is active on this thread

template <typename Result, typename... Args>
Result ask_python(const char* name, const Args&... args) {
  py::gil_scoped_acquire gil;
  TORCH_CHECK(python_ops, "iex_ops: the package has not been initialised");
  return py::cast<Result>((*python_ops)[name](args...));
}

// The same for what is called for its effect: its result goes while the interpreter's lock is held.
template <typename... Args>
void tell_python(const char* name, const Args&... args) {
  py::gil_scoped_acquire gil;
  TORCH_CHECK(python_ops, "iex_ops: the package has not been initialised");
  (*python_ops)[name](args...);
}

int dtype_code(at::ScalarType t) { return t == at::kFloat ? IEX_F32 : t == at::kHalf ? IEX_F16 : t == at::kBFloat16 ? IEX_BF16 : -1; }

void check(int rc, const char* what) {
  TORCH_CHECK(rc == 0, what, ": ", iex_last_error(), " (code ", rc, ")");
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

// (of the current device)
bool capturing() { return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None; }

// ---- notes about patterns --------------------------------------------------------------------------------------
typedef c10::weak_intrusive_ptr<c10::TensorImpl> Weak;
struct Note {
  Weak columns, offsets;
  int64_t columns_version, offsets_version, k;
  int status;
  bool has_histogram;
  std::array<int, 16> histogram;
  double dense_share;   // < 0: not known
  Weak tables;          // of the kernels for patterns with structure; may be gone
  int64_t tables_stream;   // ... the stream whose memory they are, -1: not known
  Weak mask_tables[2];  // of sparse attention in one kernel, for 16-bit types and fp32; may be gone
  int64_t mask_stream[2];
  unsigned recorded;    // attention_form()s whose first call was captured, by three launches
};
// A type and head size that sparse attention in one kernel serves, as a bit.
unsigned attention_form(int dtype, int64_t head_dim) { return 1u << (dtype * 3 + (head_dim == 32 ? 0 : head_dim == 64 ? 1 : 2)); }
Weak weak_of(const std::optional<Tensor>& t) {
  return Weak(t.has_value() ? t->getIntrusivePtr() : c10::intrusive_ptr<c10::TensorImpl, c10::UndefinedTensorImpl>());
}
struct Known {   // what a call needs of it
  int status;
  bool has_histogram;
  std::array<int, 16> histogram;
  double dense_share;
  Tensor tables;
  int64_t tables_stream;
};

std::shared_mutex notes_mutex;
std::unordered_map<const c10::TensorImpl*, Note>& notes() {
  static auto* map = new std::unordered_map<const c10::TensorImpl*, Note>;   // (outlives every tensor)
  return *map;
}
size_t notes_sweep_at = 256;

int64_t version_of(const Tensor& t) { return t.is_inference() ? 0 : t._version(); }

// (with notes_mutex held; null: nothing is known)
Note* find_note(const Tensor& row_offsets, const Tensor& column_indices, int64_t k) {
  auto& map = notes();
  const auto it = map.find(column_indices.unsafeGetTensorImpl());
  if (it == map.end()) return nullptr;
  Note& n = it->second;
  // (a weak reference that has not expired holds the address: nobody else can have it)
  if (n.k != k || n.columns.expired() || n.offsets.expired() || n.offsets._unsafe_get_target() != row_offsets.unsafeGetTensorImpl() ||
      n.columns_version != version_of(column_indices) || n.offsets_version != version_of(row_offsets))
    return nullptr;
  return &n;
}

void set_note(const Tensor& row_offsets, const Tensor& column_indices, int64_t k, int status, const std::optional<std::vector<int>>& histogram,
              const std::optional<double>& dense_share, const std::optional<Tensor>& tables, int64_t tables_stream) {
  Note n{Weak(column_indices.getIntrusivePtr()), Weak(row_offsets.getIntrusivePtr()), version_of(column_indices), version_of(row_offsets), k, status,
         histogram.has_value(), {}, dense_share.value_or(-1.0),
         weak_of(tables), tables_stream, {weak_of({}), weak_of({})}, {-1, -1}, 0};
  if (histogram) std::copy_n(histogram->begin(), 16, n.histogram.begin());
  std::unique_lock lock(notes_mutex);
  if (const Note* before = find_note(row_offsets, column_indices, k)) {   // more is known about the same arrays
    std::copy_n(before->mask_tables, 2, n.mask_tables);
    std::copy_n(before->mask_stream, 2, n.mask_stream);
    n.recorded = before->recorded;
  }
  auto& map = notes();
  if (map.size() >= notes_sweep_at) {   // notes of tensors that are gone
    for (auto it = map.begin(); it != map.end();) it = it->second.columns.expired() ? map.erase(it) : std::next(it);
    notes_sweep_at = std::max<size_t>(256, 2 * map.size());
  }
  map.insert_or_assign(column_indices.unsafeGetTensorImpl(), std::move(n));
}

void forget_note(const Tensor& column_indices) {
  std::unique_lock lock(notes_mutex);
  notes().erase(column_indices.unsafeGetTensorImpl());
}

// for calls of q's type on the mask; lifts what an earlier capture has settled for calls like q
void set_mask_tables(const Tensor& q, const Tensor& row_offsets, const Tensor& column_indices, const Tensor& tables, int64_t stream) {
  std::unique_lock lock(notes_mutex);
  Note* n = find_note(row_offsets, column_indices, q.size(1));
  const int dtype = dtype_code(q.scalar_type()), which = dtype == IEX_F32;
  if (!n || dtype < 0) return;
  n->mask_tables[which] = weak_of(tables);
  n->mask_stream[which] = stream;
  n->recorded &= ~attention_form(dtype, q.size(2));
}

std::optional<Known> note_of(const Tensor& row_offsets, const Tensor& column_indices, int64_t k) {
  std::shared_lock lock(notes_mutex);
  const Note* found = find_note(row_offsets, column_indices, k);
  if (!found) return {};
  const Note& n = *found;
  Known known{n.status, n.has_histogram, n.histogram, n.dense_share, Tensor(), n.tables_stream};
  if (auto alive = n.tables.lock()) known.tables = Tensor(std::move(alive));
  return known;
}

// Memory that outlives a call is memory of the stream it was made on.  Work on another one is told to its allocator.
void use_memory(const Tensor& memory, int64_t made_on) {
  const auto stream = c10::hip::getCurrentHIPStream(memory.get_device());
  if (stream.id() != made_on) memory.record_stream(c10::Stream(c10::Stream::UNSAFE, memory.device(), stream.id()));   // (a tensor's device is "cuda", the stream's "hip")
}

// The same for tables kept with a pattern; a call that is captured has them kept as long as the pattern's tensor, also where later calls
// replace them.
void use_tables(const Tensor& tables, int64_t tables_stream, const Tensor& column_indices, bool captured) {
  if (captured) tell_python("keep_recorded", column_indices, tables);
  else use_memory(tables, tables_stream);
}

// ---- operands that fit -------------------------------------------------------------------------------------------
// Whether a call may pass the dispatcher by: no tensor that wraps another (vmap, jvp, functionalize, a subclass with a dispatch of its own),
// and nobody who follows the operators called (a dispatch mode, a tracer).
bool unwatched(const Tensor& t) {
  using K = c10::DispatchKey;
  constexpr c10::DispatchKeySet wrappers({K::Python, K::FuncTorchBatched, K::FuncTorchGradWrapper, K::Functionalize});
  return t.has_storage() && !t.key_set().has_any(wrappers) && !c10::impl::TorchDispatchModeTLS::any_modes_set() && !c10::impl::tls_is_dispatch_key_included(K::Tracer);
}

bool plain(const Tensor& t, int64_t dim) { return t.is_cuda() && t.layout() == at::kStrided && t.dim() == dim && t.is_contiguous(); }

bool plain_csr(const Tensor& row_indices, const Tensor& row_offsets, const Tensor& column_indices, const Tensor& with, int64_t m) {
  return plain(row_indices, 1) && plain(row_offsets, 1) && plain(column_indices, 1) && row_indices.scalar_type() == at::kInt &&
         row_offsets.scalar_type() == at::kInt && row_indices.size(0) == m && row_offsets.size(0) == m + 1 && column_indices.size(0) > 0 &&
         row_indices.device() == with.device() && row_offsets.device() == with.device() && column_indices.device() == with.device();
}

constexpr int kBadPattern = IEX_CSR_BAD_OFFSETS | IEX_CSR_COLUMN_OUT_OF_RANGE;
// Patterns of attention-sized products with at least this share of their nonzeros in dense 128 x 128 blocks go to the
// kernels for patterns with structure (ops._STRUCTURE_SHARE).
constexpr double kStructureShare = 0.5;
constexpr double kStructureCells = 1 << 25;

Tensor workspace(size_t bytes, const Tensor& like) {
  return bytes ? at::empty({(int64_t)bytes}, like.options().dtype(at::kByte)) : Tensor();
}

// ... that a call can do without: nothing where there is no memory for it
Tensor optional_workspace(size_t bytes, const Tensor& like) {
  try {
    return workspace(bytes, like);
  } catch (const c10::OutOfMemoryError&) {
    return Tensor();
  }
}

// ---- SpMM ----------------------------------------------------------------------------------------------------------
enum class Spmm { kSharedF32, kSharedHalf, kPerEntry, kAtomic };

const char* spmm_name(Spmm kind) {
  switch (kind) {
    case Spmm::kSharedF32: return "spmm_sputnik_reuse_weight";
    case Spmm::kSharedHalf: return "spmm_sputnik_reuse_weight_half";
    case Spmm::kPerEntry: return "spmm_sputnik_batched_values";
    default: return "spmm_sputnik_atomic";
  }
}

// flat: b is (k, n) and the result (m, n), without the batch dimension.  aux: (16-bit, shared values) an operand of the
// result's shape, mode 1 added, mode 2 its SiLU multiplied; undefined is returned where the call is not served here
template <Spmm kind, bool flat>
Tensor spmm_call(const Tensor& b, const Tensor& row_indices, const Tensor& values, const Tensor& row_offsets, const Tensor& column_indices, int64_t m,
                 const Tensor& aux = Tensor(), int aux_mode = 0) {
  constexpr bool per_entry = kind == Spmm::kPerEntry || kind == Spmm::kAtomic, accumulate = kind == Spmm::kAtomic;
  auto python = [&] {
    if (aux.defined()) return Tensor();
    const Tensor out = ask_python<Tensor>(spmm_name(kind), flat ? b.unsqueeze(0) : b, row_indices, values, row_offsets, column_indices, m);
    return flat ? at::_unsafe_view(out, {out.size(1), out.size(2)}) : out;
  };
  if (forced || !plain(b, flat ? 2 : 3) || !plain(values, per_entry ? 2 : 1) || values.device() != b.device() || values.scalar_type() != b.scalar_type() ||
      !plain_csr(row_indices, row_offsets, column_indices, b, m))
    return python();
  const int dtype = dtype_code(b.scalar_type());
  const bool i16 = column_indices.scalar_type() == at::kShort;
  const bool type_fits = kind == Spmm::kPerEntry ? dtype >= 0 : kind == Spmm::kSharedHalf ? (dtype == IEX_F16 || dtype == IEX_BF16) : dtype == IEX_F32;
  const bool index_fits = i16 ? dtype == IEX_F16 : column_indices.scalar_type() == at::kInt;
  const int64_t batch = flat ? 1 : b.size(0), k = b.size(-2), n = b.size(-1), nonzeros = column_indices.size(0);
  const bool shape_fits = values.size(-1) == nonzeros && (!per_entry || values.size(0) == batch) && (!accumulate || batch == 1 || nonzeros % 4 == 0);
  if (!type_fits || !index_fits || !shape_fits || batch * m * n == 0) return python();
  const auto known = note_of(row_offsets, column_indices, k);
  if (!known || (known->status & kBadPattern)) return python();
  const bool any_order = known->status & IEX_CSR_NOT_ASCENDING;
  const int itype = i16 ? IEX_I16 : IEX_I32;
  int flags = IEX_SPMM_PAD_OPERANDS | (per_entry ? IEX_SPMM_PER_BATCH_VALUES : 0) | (accumulate ? IEX_SPMM_ACCUMULATE : 0) | (any_order ? IEX_SPMM_ANY_COLUMN_ORDER : 0);
  auto kind_of = [&](int f) { return iex_spmm_workspace_kind(dtype, itype, f, m, k, n, nonzeros, batch); };
  if (kind == Spmm::kPerEntry && !any_order && dtype != IEX_F32 && known->dense_share >= 0 && (double)batch * m * k >= kStructureCells) {
    // by the pattern's structure where a look at it has told, not by its density (the library's rule)
    if (known->dense_share >= kStructureShare) flags |= kind_of(flags | IEX_SPMM_FORCE_VARIANT(10)) == 10 ? IEX_SPMM_FORCE_VARIANT(10) : 0;
    else if (kind_of(flags) == 10) flags |= IEX_SPMM_FORCE_VARIANT(1);
  }
  const c10::DeviceGuard guard(b.device());
  const int64_t shape[3] = {batch, m, n};
  const at::IntArrayRef out_shape(shape + flat, 3 - flat);
  Tensor out = accumulate ? at::zeros(out_shape, b.options()) : at::empty(out_shape, b.options());
  const size_t ws_bytes = iex_spmm_workspace_bytes(dtype, itype, flags, m, k, n, nonzeros, batch);
  Tensor ws;
  if (ws_bytes && kind_of(flags) == 10) {
    if (!known->tables.defined() || (size_t)known->tables.numel() < ws_bytes) return python();   // (it makes them)
    ws = known->tables;
    use_tables(ws, known->tables_stream, column_indices, capturing());
    flags |= IEX_SPMM_TABLES_READY | IEX_SPMM_LISTS_READY;
  } else {
    ws = optional_workspace(ws_bytes, b);
  }
  if (aux.defined()) {
    if ((ws_bytes && !ws.defined()) || !plain(aux, 3 - flat) || aux.sizes() != out_shape || aux.scalar_type() != b.scalar_type() || aux.device() != b.device()) return Tensor();
    check(iex_spmm_aux(dtype, itype, flags, m, k, n, nonzeros, row_indices.const_data_ptr<int>(), values.const_data_ptr(),
                       row_offsets.const_data_ptr<int>(), column_indices.const_data_ptr(), b.const_data_ptr(), aux.const_data_ptr(), aux_mode,
                       out.data_ptr(), stream_of(b), batch, ws.defined() ? ws.data_ptr() : nullptr, ws_bytes,
                       known->has_histogram ? known->histogram.data() : nullptr),
          "spmm");
    return out;
  }
  check(iex_spmm_sched(dtype, itype, flags, m, k, n, nonzeros, row_indices.const_data_ptr<int>(), values.const_data_ptr(),
                       row_offsets.const_data_ptr<int>(), column_indices.const_data_ptr(), b.const_data_ptr(), nullptr, out.data_ptr(), stream_of(b),
                       batch, ws.defined() ? ws.data_ptr() : nullptr, ws_bytes, known->has_histogram ? known->histogram.data() : nullptr),
        "spmm");
  return out;
}

template <Spmm kind>
Tensor spmm(const Tensor& b, const Tensor& row_indices, const Tensor& values, const Tensor& row_offsets, const Tensor& column_indices, int64_t m) {
  return spmm_call<kind, false>(b, row_indices, values, row_offsets, column_indices, m);
}

// ---- SDDMM ---------------------------------------------------------------------------------------------------------
// flat: a is (m, k), b (n, k) and the result (nnz), without the batch dimension
template <bool summed, bool flat = false>
Tensor sddmm(const Tensor& a, const Tensor& b, const Tensor& row_indices, const Tensor& row_offsets, const Tensor& column_indices) {
  auto python = [&] {
    const Tensor out = ask_python<Tensor>(summed ? "sddmm_sputnik_atomic_upd_weight" : "sddmm_sputnik_half", flat ? a.unsqueeze(0) : a,
                                          flat ? b.unsqueeze(0) : b, row_indices, row_offsets, column_indices);
    return flat && !summed ? at::_unsafe_view(out, {out.size(1)}) : out;
  };
  if (forced || !plain(a, flat ? 2 : 3) || !plain(b, flat ? 2 : 3) || b.device() != a.device() || b.scalar_type() != a.scalar_type() ||
      (!flat && a.size(0) != b.size(0)) || a.size(-1) != b.size(-1) || !plain_csr(row_indices, row_offsets, column_indices, a, a.size(-2)) ||
      column_indices.scalar_type() != at::kInt)
    return python();
  const int dtype = dtype_code(a.scalar_type());
  const int64_t batch = flat ? 1 : a.size(0), m = a.size(-2), k = a.size(-1), n = b.size(-2), nonzeros = column_indices.size(0);
  if (dtype < 0 || (summed && dtype != IEX_F32) || batch * m == 0) return python();
  const auto known = note_of(row_offsets, column_indices, n);
  if (!known || (known->status & kBadPattern)) return python();
  const bool any_order = known->status & IEX_CSR_NOT_ASCENDING;
  int flags = IEX_SDDMM_PAD_OPERANDS | (summed ? IEX_SDDMM_SUM_OVER_BATCH : 0) | (any_order ? IEX_SDDMM_ANY_COLUMN_ORDER : 0);
  auto kind_of = [&](int f) { return iex_sddmm_workspace_kind(dtype, f, m, k, n, nonzeros, batch); };
  if (!summed && !any_order && dtype != IEX_F32 && known->dense_share >= 0 && (double)batch * m * n >= kStructureCells) {
    if (known->dense_share >= kStructureShare) flags |= kind_of(flags | IEX_SDDMM_FORCE_VARIANT(3)) == 3 ? IEX_SDDMM_FORCE_VARIANT(3) : 0;
    else if (kind_of(flags) == 3) flags |= IEX_SDDMM_FORCE_VARIANT(1);
  }
  const c10::DeviceGuard guard(a.device());
  Tensor out = summed || flat ? at::empty({nonzeros}, a.options()) : at::empty({batch, nonzeros}, a.options());
  const size_t ws_bytes = iex_sddmm_workspace_bytes(dtype, flags, m, k, n, nonzeros, batch);
  Tensor ws;
  if (ws_bytes && kind_of(flags) == 3) {
    if (!known->tables.defined() || (size_t)known->tables.numel() < ws_bytes) return python();   // (it makes them)
    ws = known->tables;
    use_tables(ws, known->tables_stream, column_indices, capturing());
    flags |= IEX_SDDMM_TABLES_READY | IEX_SDDMM_LISTS_READY;
  } else {
    ws = optional_workspace(ws_bytes, a);
  }
  check(iex_sddmm_ws(dtype, flags, m, k, n, nonzeros, row_indices.const_data_ptr<int>(), row_offsets.const_data_ptr<int>(),
                     column_indices.const_data_ptr<int>(), a.const_data_ptr(), b.const_data_ptr(), out.data_ptr(), stream_of(a), batch,
                     ws.defined() ? ws.data_ptr() : nullptr, ws_bytes),
        "sddmm");
  return out;
}

// ---- softmax, GEMM -------------------------------------------------------------------------------------------------
Tensor csr_softmax(Tensor values, const Tensor& row_indices, const Tensor& row_offsets, double scale) {
  const int dtype = dtype_code(values.scalar_type());
  const int64_t m = row_indices.dim() == 1 ? row_indices.size(0) : -1;
  if (!plain(values, 2) || !plain(row_indices, 1) || !plain(row_offsets, 1) || dtype < 0 || row_indices.scalar_type() != at::kInt ||
      row_offsets.scalar_type() != at::kInt || row_offsets.size(0) != m + 1 || row_indices.device() != values.device() ||
      row_offsets.device() != values.device()) {
    tell_python("csr_softmax_", values, row_indices, row_offsets, scale);
    return values;
  }
  const c10::DeviceGuard guard(values.device());
  check(iex_csr_softmax(dtype, m, values.size(1), row_indices.const_data_ptr<int>(), row_offsets.const_data_ptr<int>(), values.data_ptr(), (float)scale,
                        stream_of(values), values.size(0)),
        "csr_softmax");
  return values;
}

Tensor gemm(const Tensor& a, const Tensor& b, bool trans_b) {
  const int dtype = dtype_code(a.scalar_type());
  const bool fits = !forced && (a.dim() == 2 || a.dim() == 3) && (b.dim() == 2 || b.dim() == 3) && plain(a, a.dim()) && plain(b, b.dim()) &&
                    a.device() == b.device() && (dtype == IEX_F16 || dtype == IEX_BF16) && b.scalar_type() == a.scalar_type() &&
                    b.size(trans_b ? -1 : -2) == a.size(-1) && (a.dim() == 2 || b.dim() == 2 || a.size(0) == b.size(0));
  if (!fits) return ask_python<Tensor>("gemm_mfma", a, b, trans_b);
  const int64_t M = a.size(-2), K = a.size(-1), N = b.size(trans_b ? -2 : -1);
  const bool batched = a.dim() == 3 || b.dim() == 3;
  const int64_t batch = a.dim() == 3 ? a.size(0) : b.dim() == 3 ? b.size(0) : 1;
  const c10::DeviceGuard guard(a.device());
  Tensor out = batched ? at::empty({batch, M, N}, a.options()) : at::empty({M, N}, a.options());
  const size_t ws_bytes = iex_gemm_workspace_bytes(dtype, trans_b, M, N, K, batch);
  const Tensor ws = optional_workspace(ws_bytes, a);
  check(iex_gemm_ws(dtype, trans_b, M, N, K, a.const_data_ptr(), b.const_data_ptr(), out.data_ptr(), batch, a.dim() == 3 ? M * K : 0,
                    b.dim() == 3 ? N * K : 0, M * N, stream_of(a), ws.defined() ? ws.data_ptr() : nullptr, ws_bytes),
        "gemm");
  return out;
}

// a^T @ b for a (K, M), b (K, N): the gradient of a linear layer's weight, without a transposed copy of a
Tensor gemm_transposed_a(const Tensor& a, const Tensor& b) {
  const int dtype = dtype_code(a.scalar_type());
  if (forced || !plain(a, 2) || !plain(b, 2) || (dtype != IEX_F16 && dtype != IEX_BF16) || b.scalar_type() != a.scalar_type() ||
      b.device() != a.device() || b.size(0) != a.size(0) || a.size(0) == 0 || a.size(1) % 8 != 0 || b.size(1) % 8 != 0)
    return gemm(a.t().contiguous(), b, false);
  const int64_t K = a.size(0), M = a.size(1), N = b.size(1);
  const c10::DeviceGuard guard(a.device());
  Tensor out = at::empty({M, N}, a.options());
  const size_t ws_bytes = iex_gemm_workspace_bytes(dtype, 2, M, N, K, 1);
  const Tensor ws = optional_workspace(ws_bytes, a);
  check(iex_gemm_ws(dtype, 2, M, N, K, a.const_data_ptr(), b.const_data_ptr(), out.data_ptr(), 1, 0, 0, 0, stream_of(a),
                    ws.defined() ? ws.data_ptr() : nullptr, ws_bytes),
        "gemm");
  return out;
}

// ---- the steps of a decoder layer around its products --------------------------------------------------------------
// W_csr @ x combined with a second operand (see spmm above); None where that is not served natively
std::optional<Tensor> spmm_with(const Tensor& x, const Tensor& row_indices, const Tensor& values, const Tensor& row_offsets, const Tensor& column_indices,
                                int64_t m, const Tensor& aux, int mode) {
  if (at::GradMode::is_enabled() && (x.requires_grad() || values.requires_grad() || aux.requires_grad())) return {};
  const Tensor out = spmm_call<Spmm::kSharedHalf, true>(x, row_indices, values, row_offsets, column_indices, m, aux, mode);
  return out.defined() ? std::optional<Tensor>(out) : std::nullopt;
}

// A sparse weight for a program that keeps it (ops.WeightForm makes it): the product with x, combined with `other` as in spmm_with.  Nothing is
// returned where the call is not served here -- operands that do not fit, a gradient wanted, kernels forced, an operator on the CSR arrays that is
// faster.  The first product that takes a kind of form lays it out, on its stream and without waiting; later ones find it, on other streams behind
// an event.  A captured call lays the weight out inside the graph, so that replays follow the CSR arrays; it takes another way through the product than a
// call, with the sums in another order, where laying out at every replay would cost more than it gains.
struct WeightForm {
  static constexpr int kAnyRoom = 1 << 20;
  struct Layout {
    Tensor memory;
    at::cuda::CUDAEvent ready;
    int64_t made_on = -1;   // the stream whose memory it is
    uint64_t of = 0;        // the generation of the values that are laid out
  };
  int dtype;
  int64_t m, k, nonzeros;
  std::array<Layout, 4> layouts;   // kinds 0, 128, 192, 256
  std::mutex layouts_mutex;
  std::array<int, 3> phases, rooms;
  int kinds;                       // a bit for each that the weight can be laid out as
  Tensor row_offsets, column_indices;
  std::array<int64_t, 2> pattern_versions;   // when the form was made for them
  // the values, their version, how many there were before; for copies only, so that it may be waited for with the interpreter's lock in hand
  mutable std::mutex values_mutex;
  Tensor values;
  int64_t values_version;
  uint64_t generation = 1;

  WeightForm(const Tensor& values, const Tensor& row_offsets, const Tensor& column_indices, const std::array<int64_t, 3>& versions, int64_t m, int64_t k, int kinds,
             const std::vector<int>& measured)
      : dtype(dtype_code(values.scalar_type())), m(m), k(k), nonzeros(column_indices.numel()), kinds(kinds), row_offsets(row_offsets), column_indices(column_indices),
        pattern_versions{versions[1], versions[2]}, values(values), values_version(versions[0]) {
    TORCH_CHECK(measured.size() == 6, "WeightForm: six numbers");
    std::copy_n(measured.begin(), 3, phases.begin());
    std::copy_n(measured.begin() + 3, 3, rooms.begin());
  }

  static bool unchanged(const Tensor& mine, const Tensor& given, int64_t version) { return given.is_same(mine) && !given.is_inference() && given._version() == version; }
  bool is_of_pattern(const Tensor& offsets, const Tensor& columns) const {
    return unchanged(row_offsets, offsets, pattern_versions[0]) && unchanged(column_indices, columns, pattern_versions[1]);
  }
  // whether these are its tensors, unchanged since (never of tensors that count no changes)
  bool is_of(const Tensor& v, const Tensor& offsets, const Tensor& columns) const {
    std::lock_guard lock(values_mutex);
    return unchanged(values, v, values_version) && is_of_pattern(offsets, columns);
  }

  int laid_out() {   // a bit for each kind that is
    std::scoped_lock lock(layouts_mutex, values_mutex);
    int bits = 0;
    for (int i = 0; i < 4; ++i) bits |= (layouts[i].memory.defined() && layouts[i].of == generation) << i;
    return bits;
  }

  Tensor lay_out(int kind, int room, const Tensor& values, const Tensor& like) const {
    Tensor form = workspace(iex_form_bytes(kind, m, k, room), like);
    const Tensor scratch = workspace(kind ? iex_form_scratch_bytes(m, k) : 0, like);
    check(iex_form_build(column_indices.scalar_type() == at::kShort ? IEX_I16 : IEX_I32, kind, m, k, nonzeros, row_offsets.const_data_ptr<int>(),
                         column_indices.const_data_ptr(), values.const_data_ptr(), room, form.data_ptr(), form.numel(),
                         scratch.defined() ? scratch.data_ptr() : nullptr, scratch.defined() ? scratch.numel() : 0, stream_of(like)),
          "form");
    return form;
  }

  // the kind of form that serves the call, -1: none; `captured` is looked up where it matters
  int kind_for(const Tensor& x, const std::optional<Tensor>& other, bool& captured) const {
    const int64_t n = x.dim() == 2 ? x.size(1) : 0;
    if (forced || !unwatched(x) || (other && !unwatched(*other)) || !plain(x, 2) || x.size(0) != k || n == 0 || n % 8 || k * n >= (1ll << 31) || m * n >= (1ll << 31) || dtype_code(x.scalar_type()) != dtype ||
        x.device() != row_offsets.device() || reinterpret_cast<uintptr_t>(x.const_data_ptr()) % 16 ||
        (at::GradMode::is_enabled() && (x.requires_grad() || (other && other->requires_grad()))))
      return -1;
    if (other && (!plain(*other, 2) || other->size(0) != m || other->size(1) != n || other->scalar_type() != x.scalar_type() || other->device() != x.device())) return -1;
    const int kept = iex_form_choose(kinds, m, k, n, nonzeros, phases.data()), each_call = iex_form_choose(kinds | IEX_FORM_EACH_CALL, m, k, n, nonzeros, phases.data());
    captured = false;
    if (kept < 0 && each_call < 0) return -1;
    const c10::DeviceGuard guard(x.device());
    captured = capturing();
    return captured ? each_call : kept;
  }

  // Takes values that were changed, or others, of the same pattern; the next product lays them out.  (Captured: the caller sees to it.)
  bool renew(const Tensor& v, const Tensor& offsets, const Tensor& columns) {
    if (v.is_inference() || !unwatched(v) || !plain(v, 1) || v.numel() != nonzeros || dtype_code(v.scalar_type()) != dtype || v.device() != row_offsets.device() ||
        !is_of_pattern(offsets, columns))
      return false;
    {
      const c10::DeviceGuard guard(v.device());
      if (capturing()) return false;
    }
    Tensor taken = v;
    std::lock_guard lock(values_mutex);
    std::swap(values, taken);   // (what goes is released without the lock)
    values_version = v._version();
    ++generation;
    return true;
  }

  // None: an operator on the CSR arrays serves the call.  False: the form is not of this pattern as it is now.
  py::object serve(const Tensor& v, const Tensor& offsets, const Tensor& columns, const Tensor& x, const std::optional<Tensor>& other, int mode) {
    if (!is_of(v, offsets, columns) && !renew(v, offsets, columns)) return py::bool_(false);
    bool captured;
    const int kind = kind_for(x, other, captured);
    return kind < 0 ? py::object(py::none()) : py::cast(product_by(kind, captured, x, other, mode));
  }

  std::optional<Tensor> product(const Tensor& x, const std::optional<Tensor>& other, int mode) {
    bool captured;
    const int kind = kind_for(x, other, captured);
    return kind < 0 ? std::nullopt : std::optional<Tensor>(product_by(kind, captured, x, other, mode));
  }

  Tensor product_by(int kind, bool captured, const Tensor& x, const std::optional<Tensor>& aux, int mode) {
    const py::gil_scoped_release nobody_waits_for_layouts_mutex_with_it;
    const c10::DeviceGuard guard(x.device());
    const int64_t n = x.size(1);
    int room = kind ? rooms[kind / 64 - 2] : 0;
    Tensor form, v;
    uint64_t now;
    {
      std::lock_guard lock(values_mutex);
      v = values, now = generation;
    }
    if (captured) {
      room = kind ? kAnyRoom : 0;   // (the pattern of a later replay may spill more)
      form = lay_out(kind, room, v, x);
    } else {
      std::lock_guard lock(layouts_mutex);
      Layout& layout = layouts[kind ? kind / 64 - 1 : 0];
      const auto stream = at::cuda::getCurrentHIPStreamMasqueradingAsCUDA(x.get_device());
      if (!layout.memory.defined() || layout.of != now) {
        for (Layout& other : layouts)
          if (other.of != now) other.memory = Tensor();
        const Tensor made = lay_out(kind, room, v, x);
        layout.of = now;
        layout.ready.record(stream);
        layout.made_on = c10::hip::getCurrentHIPStream(x.get_device()).id();
        layout.memory = made;
      } else if (c10::hip::getCurrentHIPStream(x.get_device()).id() != layout.made_on) {
        layout.ready.block(stream);
        use_memory(layout.memory, layout.made_on);
      }
      form = layout.memory;
    }
    const size_t ws_bytes = iex_form_product_workspace_bytes(kind, m, k, n);
    const Tensor ws = optional_workspace(ws_bytes, x);
    Tensor out = at::empty({m, n}, x.options());
    check(iex_form_product(dtype, kind, m, k, n, room, form.const_data_ptr(), x.const_data_ptr(), aux ? aux->const_data_ptr() : nullptr, mode,
                           out.data_ptr(), ws.defined() ? ws.data_ptr() : nullptr, ws_bytes, stream_of(x)),
          "form product");
    return out;
  }
};

// softmax(scale * q^T k) v per head and sequence on feature-major operands; None where the kernel does not serve them
std::optional<Tensor> attention(const Tensor& q, const Tensor& k, const Tensor& v, int64_t heads, int64_t seqs, double scale) {
  const int dtype = dtype_code(q.scalar_type());
  if (forced || !plain(q, 2) || !plain(k, 2) || !plain(v, 2) || k.sizes() != q.sizes() || v.sizes() != q.sizes() || k.scalar_type() != q.scalar_type() ||
      v.scalar_type() != q.scalar_type() || k.device() != q.device() || v.device() != q.device() || heads <= 0 || seqs <= 0 || q.size(0) % heads != 0 ||
      q.size(1) % seqs != 0 || !(scale > 0) || !iex_attention_fits(dtype, q.size(0) / heads, q.size(1) / seqs))
    return {};
  if (at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad())) return {};
  for (const Tensor* t : {&q, &k, &v})
    if (reinterpret_cast<uintptr_t>(t->const_data_ptr()) % 16) return {};
  const c10::DeviceGuard guard(q.device());
  Tensor out = at::empty_like(q);
  check(iex_attention(dtype, heads, q.size(0) / heads, seqs, q.size(1) / seqs, q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(), (float)scale,
                      out.data_ptr(), stream_of(q)),
        "attention");
  return out;
}

// sparse attention in one kernel.  None where it does not serve the call, True where it will once the mask has its tables
// (ops.prepare_mask).
py::object sparse_attention(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& row_indices, const Tensor& row_offsets,
                            const Tensor& column_indices, double scale) {
  const int dtype = dtype_code(q.scalar_type());
  if (forced || dtype < 0 || !plain(q, 3) || !plain(k, 3) || !plain(v, 3) || k.sizes() != q.sizes() || v.sizes() != q.sizes() ||
      k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type() || k.device() != q.device() || v.device() != q.device() || q.size(0) == 0 ||
      !(scale > 0) || !iex_sparse_attention_fits(dtype, q.size(2), q.size(1)) || !plain_csr(row_indices, row_offsets, column_indices, q, q.size(1)) ||
      column_indices.scalar_type() != at::kInt)
    return py::none();
  if (at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad())) return py::none();
  for (const Tensor* t : {&q, &k, &v})
    if (reinterpret_cast<uintptr_t>(t->const_data_ptr()) % 16) return py::none();
  const c10::DeviceGuard guard(q.device());
  const bool captured = capturing();
  const int which = dtype == IEX_F32;
  Tensor tables;
  int64_t tables_stream = -1;
  {
    std::unique_lock lock(notes_mutex);
    Note* n = find_note(row_offsets, column_indices, q.size(1));
    if (!n) return captured ? py::object(py::none()) : py::object(py::bool_(true));   // (nobody has looked at it)
    const unsigned form = attention_form(dtype, q.size(2));
    // (columns in any order; a pattern that nobody may look at: it changes from call to call; one whose first call like this
    // was captured before it had tables: replays and eager calls give the same bits)
    if (n->status != 0 || !n->has_histogram || (n->recorded & form)) return py::none();
    if (auto alive = n->mask_tables[which].lock()) tables = Tensor(std::move(alive));
    tables_stream = n->mask_stream[which];
    if (!tables.defined()) {
      if (!captured) return py::bool_(true);
      n->recorded |= form;
      return py::none();
    }
  }
  use_tables(tables, tables_stream, column_indices, captured);
  Tensor out = at::empty_like(q);
  check(iex_sparse_attention(dtype, q.size(0), q.size(1), q.size(2), column_indices.size(0), row_offsets.const_data_ptr<int>(), q.const_data_ptr(),
                             k.const_data_ptr(), v.const_data_ptr(), (float)scale, out.data_ptr(), tables.const_data_ptr(), tables.numel(), stream_of(q)),
        "sparse attention");
  return py::cast(out);
}

// ---- autograd: the plain calls of MySpMM and MyLinear (no recording, no forced kernels) -----------------------------
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

Tensor spmm_shared(const Tensor& b, const Tensor& row_indices, const Tensor& values, const Tensor& row_offsets, const Tensor& column_indices, int64_t m) {
  return values.scalar_type() == at::kFloat ? spmm_call<Spmm::kSharedF32, true>(b, row_indices, values, row_offsets, column_indices, m)
                                            : spmm_call<Spmm::kSharedHalf, true>(b, row_indices, values, row_offsets, column_indices, m);
}

// values[perm]: the values of the transposed matrix
Tensor permuted(const Tensor& values, const Tensor& perm) {
  const int64_t n = perm.numel();
  if (!plain(values, 1) || !plain(perm, 1) || perm.scalar_type() != at::kLong || values.numel() != n || dtype_code(values.scalar_type()) < 0 ||
      perm.device() != values.device() || reinterpret_cast<uintptr_t>(perm.const_data_ptr()) % 16 != 0)
    return values.detach().index_select(0, perm);
  const c10::DeviceGuard guard(values.device());
  Tensor out = at::empty({n}, values.options());
  check(iex_gather_values(values.element_size(), n, values.const_data_ptr(), reinterpret_cast<const long long*>(perm.const_data_ptr<int64_t>()),
                          out.data_ptr(), stream_of(values)),
        "gather_values");
  return out;
}

// A^T * grad from the CSR form of A where the transposed pattern's product would go by its dense form anyway (undefined
// elsewhere)
Tensor transposed_product(const Tensor& grad, const Tensor& values, const Tensor& row_offsets, const Tensor& column_indices, int64_t k) {
  const int dtype = dtype_code(values.scalar_type());
  if (dtype == IEX_F32 || dtype < 0 || forced || !plain(grad, 2) || !plain(values, 1) || grad.scalar_type() != values.scalar_type() ||
      grad.device() != values.device() || values.size(0) != column_indices.size(0))
    return Tensor();
  const int64_t m = grad.size(0), n = grad.size(1), nonzeros = values.size(0);
  const size_t bytes = m * k * n ? iex_spmm_transposed_workspace_bytes(dtype, m, k, n, nonzeros) : 0;
  const auto known = note_of(row_offsets, column_indices, k);
  if (!bytes || !known || known->status != 0) return Tensor();   // (canonical CSR only)
  const c10::DeviceGuard guard(grad.device());
  const Tensor ws = optional_workspace(bytes, grad);
  if (!ws.defined()) return Tensor();
  Tensor out = at::empty({k, n}, grad.options());
  check(iex_spmm_transposed(dtype, column_indices.scalar_type() == at::kShort ? IEX_I16 : IEX_I32, m, k, n, nonzeros, values.const_data_ptr(),
                            row_offsets.const_data_ptr<int>(), column_indices.const_data_ptr(), grad.const_data_ptr(), out.data_ptr(), stream_of(grad),
                            ws.data_ptr(), bytes),
        "spmm (transposed)");
  return out;
}

struct TrainableSpmm : torch::autograd::Function<TrainableSpmm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& b, const Tensor& row_indices, const Tensor& values, const Tensor& row_offsets,
                        const Tensor& column_indices, int64_t m, const Tensor& row_indices_t, const Tensor& row_offsets_t,
                        const Tensor& column_indices_t, const Tensor& perm) {
    const Tensor dense = b.contiguous();
    ctx->save_for_backward({dense, row_indices, values, row_offsets, column_indices, row_indices_t, row_offsets_t, column_indices_t, perm});
    return spmm_shared(dense, row_indices, values, row_offsets, column_indices, m);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &dense = saved[0], &row_indices = saved[1], &values = saved[2], &row_offsets = saved[3], &column_indices = saved[4];
    const Tensor grad = grads[0].contiguous();
    variable_list out(10);
    if (ctx->needs_input_grad(2)) {
      // lhs = grad (m, n), rhs = b (k, n): rows of rhs are indexed by the CSR column
      const Tensor columns = column_indices.scalar_type() == at::kInt ? column_indices : ask_python<Tensor>("int32_columns", column_indices);
      out[2] = grad.scalar_type() == at::kFloat ? sddmm<true, true>(grad, dense, row_indices, row_offsets, columns)
                                                : sddmm<false, true>(grad, dense, row_indices, row_offsets, columns);
    }
    if (ctx->needs_input_grad(0)) out[0] = transposed_product(grad, values, row_offsets, column_indices, dense.size(0));
    if (ctx->needs_input_grad(0) && !out[0].defined()) out[0] = spmm_shared(grad, saved[5], permuted(values, saved[8]), saved[6], saved[7], dense.size(0));
    return out;
  }
};

Tensor trainable_spmm(const Tensor& b, const Tensor& row_indices, const Tensor& values, const Tensor& row_offsets, const Tensor& column_indices, int64_t m,
                      const Tensor& row_indices_t, const Tensor& row_offsets_t, const Tensor& column_indices_t, const Tensor& perm) {
  py::gil_scoped_release no_gil;
  return TrainableSpmm::apply(b, row_indices, values, row_offsets, column_indices, m, row_indices_t, row_offsets_t, column_indices_t, perm);
}

struct TrainableLinear : torch::autograd::Function<TrainableLinear> {
  static Tensor forward(AutogradContext* ctx, const Tensor& input, const Tensor& weight) {
    const Tensor x = input.contiguous(), w = weight.contiguous();
    ctx->save_for_backward({x, w});
    return gemm(x, w, true);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor grad = grads[0].contiguous();
    variable_list out(2);
    if (ctx->needs_input_grad(0)) out[0] = gemm(grad, saved[1], false);
    if (ctx->needs_input_grad(1)) out[1] = gemm_transposed_a(grad, saved[0]);
    return out;
  }
};

Tensor trainable_linear(const Tensor& input, const Tensor& weight) {
  py::gil_scoped_release no_gil;
  return TrainableLinear::apply(input, weight);
}

}  // namespace

TORCH_LIBRARY(iex_ops, lib) {
  const char* spmm_schema = "(Tensor b, Tensor row_indices, Tensor values, Tensor row_offsets, Tensor column_indices, int m) -> Tensor";
  const char* sddmm_schema = "(Tensor a, Tensor b, Tensor row_indices, Tensor row_offsets, Tensor column_indices) -> Tensor";
  // one implementation for every backend: operands that are not device tensors are refused with the reference's message
  auto define = [&](const std::string& name, const char* schema, auto fn) {
    lib.def((name + schema).c_str());
    lib.impl(name.c_str(), torch::dispatch(c10::DispatchKey::CompositeExplicitAutograd, fn));
  };
  define("spmm_sputnik_reuse_weight", spmm_schema, TORCH_FN(spmm<Spmm::kSharedF32>));
  define("spmm_sputnik_atomic", spmm_schema, TORCH_FN(spmm<Spmm::kAtomic>));
  define("spmm_sputnik_reuse_weight_half", spmm_schema, TORCH_FN(spmm<Spmm::kSharedHalf>));
  define("spmm_sputnik_batched_values", spmm_schema, TORCH_FN(spmm<Spmm::kPerEntry>));
  define("sddmm_sputnik_atomic_upd_weight", sddmm_schema, TORCH_FN(sddmm<true>));
  define("sddmm_sputnik_half", sddmm_schema, TORCH_FN(sddmm<false>));
  define("csr_softmax_", "(Tensor(a!) values, Tensor row_indices, Tensor row_offsets, float scale) -> Tensor(a!)", TORCH_FN(csr_softmax));
  define("gemm_mfma", "(Tensor a, Tensor b, bool trans_b=False) -> Tensor", TORCH_FN(gemm));
}

PYBIND11_MODULE(_iex_host, module) {
  module.def("bind", [](py::object functions) { python_ops = new py::object(std::move(functions)); });
  module.def("set_forced", [](bool on) { forced = on; });
  module.def("set_note", &set_note);
  module.def("forget_note", &forget_note);
  module.def("spmm_with", &spmm_with);
  module.def("attention", &attention);
  py::class_<WeightForm>(module, "WeightForm")
      .def(py::init<const Tensor&, const Tensor&, const Tensor&, const std::array<int64_t, 3>&, int64_t, int64_t, int, const std::vector<int>&>())
      .def("is_of", &WeightForm::is_of)
      .def_readonly("kinds", &WeightForm::kinds)
      .def_property_readonly("laid_out", &WeightForm::laid_out, py::call_guard<py::gil_scoped_release>())
      .def("product", &WeightForm::product, py::arg("x"), py::arg("other") = std::nullopt, py::arg("mode") = 0)
      .def("serve", &WeightForm::serve);
  module.def("sparse_attention", &sparse_attention);
  module.def("set_mask_tables", &set_mask_tables);
  module.def("trainable_spmm", &trainable_spmm);
  module.def("trainable_linear", &trainable_linear);
}
