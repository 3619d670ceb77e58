// The row kernel for narrow outputs whose rows are no whole 128-bit vectors: 128-bit gathers at element alignment, several nonzeros at a time as for
// whole vectors (spmm_kernel in spmm.hip), the lane at a row's end shifted back inside it.  A wavefront on one nonzero with the widest vector that
// divides n, as these outputs had it, gathers single elements for an odd n.
// Bound by the gathers' way from L2, at half the rate of aligned ones where rows start at odd elements.  MI355X, us before -> now: 5136 x 5904 at 71 %, n = 14
// fp32 117 -> 50;  8435 x 4485 at 86 %, n = 42 bf16 68 -> 38;  979 x 7616 at 76 %, uneven rows, n = 17 fp32 56 -> 20;  both sides of the
// rule that takes it stand beside ragged_narrow_waves (spmm.hip).
#include "spmm_device.cuh"

namespace iex {
namespace {

template <typename T, typename IT, int VEC, int LPG, int WPR, bool SHORT>
__global__ __launch_bounds__(4 * kWave) void spmm_ragged_narrow_kernel(SpmmParams p) {
  __shared__ float red[spmm_lds_floats<VEC, WPR, 1>()];
  spmm_block<T, IT, VEC, LPG, WPR, (SHORT ? kSpmmUnroll / 2 : kSpmmUnroll), 1, true, (SHORT || sizeof(T) == 2)>(p, blockIdx.x, blockIdx.y, blockIdx.z, red);
}

template <typename T, typename IT, int LPG, int WPR>
int launch_narrow(const SpmmParams& p, int batch, hipStream_t stream) {
  constexpr int kMax = 16 / (int)sizeof(T);
  const dim3 grid(ceil_div(p.m, 4 / WPR), 1, batch);
  // (windows of four gathers for many short rows, as in spmm.hip: launch_one)
  const bool brief = p.nnz <= 128ll * p.m && (long long)p.m * batch * WPR > 16384;
  note_kernel("spmm_ragged_narrow_kernel<%s, %s, %d, %d, %d, %s>", type_name<T>(), type_name<IT>(), kMax, LPG, WPR, brief ? "true" : "false");
  if (brief) hipLaunchKernelGGL((spmm_ragged_narrow_kernel<T, IT, kMax, LPG, WPR, true>), grid, dim3(4 * kWave), 0, stream, p);
  else hipLaunchKernelGGL((spmm_ragged_narrow_kernel<T, IT, kMax, LPG, WPR, false>), grid, dim3(4 * kWave), 0, stream, p);
  return check_hip(hipGetLastError(), "spmm (narrow ragged rows) launch");
}

template <typename T, typename IT>
int launch_typed(const SpmmParams& p, int batch, int wpr, hipStream_t stream) {
  constexpr int kMax = 16 / (int)sizeof(T);
  auto with = [&](auto lanes) {
    constexpr int LPG = decltype(lanes)::value;
    return wpr == 1 ? launch_narrow<T, IT, LPG, 1>(p, batch, stream) : launch_narrow<T, IT, LPG, 4>(p, batch, stream);
  };
  if (p.n <= 8 * kMax) return with(std::integral_constant<int, 8>{});
  if (p.n <= 16 * kMax) return with(std::integral_constant<int, 16>{});
  return with(std::integral_constant<int, 32>{});
}

}  // namespace

int launch_spmm_ragged(int dtype, int itype, const SpmmParams& p, int batch, int wpr, hipStream_t stream) {
  IEX_REQUIRE(p.n >= (dtype == IEX_F32 ? 4 : 8) && p.n <= (dtype == IEX_F32 ? 128 : 256) && (wpr == 1 || wpr == 4), IEX_ERR_STATE, "spmm: narrow ragged rows of %d columns, %d wavefronts each", p.n, wpr);
  if (dtype == IEX_F32) return launch_typed<float, int>(p, batch, wpr, stream);
  if (dtype == IEX_BF16) return launch_typed<__hip_bfloat16, int>(p, batch, wpr, stream);
  return itype == IEX_I16 ? launch_typed<__half, short>(p, batch, wpr, stream) : launch_typed<__half, int>(p, batch, wpr, stream);
}

}  // namespace iex
