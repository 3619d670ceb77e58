// Host side of the dense attention on feature-major operands (attention_device.cuh).
#include "attention_device.cuh"

namespace iex {
namespace {

template <bool BF16, int HD>
int launch(const AttentionParams& p, hipStream_t stream) {
  constexpr int lds = attention_lds_bytes<HD>();
  const long long total = (long long)ceil_div(p.length, kAttnQ) * p.heads * p.seqs;
  IEX_REQUIRE(total < (1ll << 31), IEX_ERR_TOO_LARGE, "attention: too many blocks of queries");
  note_kernel("attention_kernel<%s, %d>", BF16 ? "bf16" : "f16", HD);
  hipLaunchKernelGGL((attention_kernel<BF16, HD>), dim3((unsigned)total), dim3(kAttnThreads), lds, stream, p);
  return check_hip(hipGetLastError(), "attention launch");
}

}  // namespace
}  // namespace iex

extern "C" int iex_attention_fits(int dtype, int head_dim, int length) {
  return (dtype == IEX_F16 || dtype == IEX_BF16) && (head_dim == 64 || head_dim == 128) && length > 0 && length % 8 == 0;
}

extern "C" int iex_attention(int dtype, int heads, int head_dim, int seqs, int length, const void* q, const void* k, const void* v, float scale, void* out,
                             void* stream) {
  using namespace iex;
  IEX_REQUIRE(heads >= 0 && head_dim >= 0 && seqs >= 0 && length >= 0, IEX_ERR_BAD_ARGUMENT, "attention: negative dimension");
  trail_reset();
  if (heads == 0 || seqs == 0 || length == 0) return 0;
  IEX_REQUIRE(q && k && v && out, IEX_ERR_BAD_ARGUMENT, "attention: null pointer argument");
  IEX_REQUIRE(iex_attention_fits(dtype, head_dim, length), IEX_ERR_UNSUPPORTED,
              "attention: fp16 / bf16, heads of 64 or 128 and a length that is a multiple of 8 (head_dim=%d length=%d)", head_dim, length);
  IEX_REQUIRE(scale > 0.f, IEX_ERR_UNSUPPORTED, "attention: the scale must be positive");
  IEX_REQUIRE(aligned(q, 16) && aligned(k, 16) && aligned(v, 16) && aligned(out, 2), IEX_ERR_UNSUPPORTED, "attention: operands must be 16-byte aligned");
  AttentionParams p{heads, seqs, length, q, k, v, out, scale * 1.44269504088896340736f};
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (head_dim == 64) return dtype == IEX_BF16 ? launch<true, 64>(p, s) : launch<false, 64>(p, s);
  return dtype == IEX_BF16 ? launch<true, 128>(p, s) : launch<false, 128>(p, s);
}
