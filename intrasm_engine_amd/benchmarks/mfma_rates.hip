// Rates of the 16-bit matrix-core forms with nothing beside them: eight wavefronts per CU, each multiplying fragments that stay
// in registers into independent accumulators, on random and on all-zero operands.  The difference between the two is the
// card's power limit: the clock follows what the matrix cores move.
//
//   hipcc --offload-arch=gfx950 -O3 -std=c++17 -Xclang -target-feature -Xclang -packed-fp32-ops \
//         intrasm_engine_amd/benchmarks/mfma_rates.hip -o mfma_rates && ./mfma_rates
#include "../csrc/gemm_device.cuh"

#include <cstdio>
#include <cstdlib>
#include <vector>

using namespace iex;

constexpr int kWavesPerBlock = 8, kBlocks = 256, kFragments = 8;

// FORM 0: 32 x 32 x 16, 1: 16 x 16 x 32.  The same flops per iteration: 4 x 2 blocks of 32 x 32 by 32 k.
template <bool BF16, int FORM>
__global__ __launch_bounds__(kWavesPerBlock * 64, 2) void mfma_kernel(const u32x4* __restrict__ from, f32x4* __restrict__ to, int iterations) {
  const int lane = threadIdx.x & 63, id = blockIdx.x * blockDim.x + threadIdx.x;
  u32x4 a[kFragments], b[kFragments];
#pragma unroll
  for (int i = 0; i < kFragments; ++i) a[i] = from[i * 64 + lane], b[i] = from[(kFragments + i) * 64 + lane];
  f32x4 out = {0.f, 0.f, 0.f, 0.f};
  if constexpr (FORM == 0) {
    f32x16 acc[4][2] = {};
    for (int n = 0; n < iterations; ++n)
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[i][j] = mfma_32x32x16<BF16>(a[k * 4 + i], b[k * 2 + j], acc[i][j]);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) out[r % 4] += acc[i][j][r];
  } else {
    f32x4 acc[8][4] = {};
    for (int n = 0; n < iterations; ++n)
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = mfma_16x16x32<BF16>(a[i], b[j], acc[i][j]);
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) out[r] += acc[i][j][r];
  }
  to[id] = out;
}

template <bool BF16, int FORM>
static double rate(const u32x4* from, f32x4* to) {
  constexpr int iterations = 20000, reps = 10;
  auto launch = [&] { hipLaunchKernelGGL((mfma_kernel<BF16, FORM>), dim3(kBlocks), dim3(kWavesPerBlock * 64), 0, 0, from, to, iterations); };
  hipEvent_t start, stop;
  if (hipEventCreate(&start) != hipSuccess || hipEventCreate(&stop) != hipSuccess) return -1.0;
  for (int i = 0; i < 5; ++i) launch();
  (void)hipEventRecord(start);
  for (int i = 0; i < reps; ++i) launch();
  (void)hipEventRecord(stop);
  if (hipEventSynchronize(stop) != hipSuccess || hipGetLastError() != hipSuccess) return -1.0;
  float ms = 0;
  (void)hipEventElapsedTime(&ms, start, stop);
  return 2.0 * 128 * 64 * 32 * iterations * kBlocks * kWavesPerBlock * reps / (ms * 1e-3) / 1e12;
}

int main() {
  const size_t words = 2 * kFragments * 64 * 4;
  std::vector<unsigned> host(words);
  u32x4* from = nullptr;
  f32x4* to = nullptr;
  if (hipMalloc(&from, words * 4) != hipSuccess || hipMalloc(&to, (size_t)kBlocks * kWavesPerBlock * 64 * 16) != hipSuccess) return 1;
  for (int zero = 0; zero < 2; ++zero) {
    for (unsigned& w : host) {   // two 16-bit values between 0.5 and 2 (fp16) or of that exponent range (bf16), random signs and mantissas
      auto one = [] { return (unsigned)((rand() & 1) << 15 | 0x3800 | (rand() & 0x7ff)); };
      w = zero ? 0u : one() | one() << 16;
    }
    if (hipMemcpy(from, host.data(), words * 4, hipMemcpyHostToDevice) != hipSuccess) return 1;
    printf("%s operands (TFLOP/s): bf16 32x32x16 %.0f, 16x16x32 %.0f; fp16 32x32x16 %.0f, 16x16x32 %.0f\n", zero ? "all-zero" : "random", rate<true, 0>(from, to),
           rate<true, 1>(from, to), rate<false, 0>(from, to), rate<false, 1>(from, to));
  }
  return 0;
}
