// The divisions of dev_common.hh against the compiler's, bit for bit:
//   DivSmall    a / n for every n it takes: every float mantissa, and doubles
//               half of them next to a multiple of n;
//   DivInRange  a / b over divisors and quotients well beyond those of vexp and
//               vlog, half of the dividends next to a multiple of b, and 0 / b.
#include <cstdio>
#include <cstdlib>

#include "device/dev_common.hh"

using namespace hepem;

namespace {

constexpr int kBlocks = 2048, kThreads = 256;
constexpr uint32_t kPerThread = 64;

// a double with the fraction bits of w and an exponent in [lo, hi)
__device__ double Random(uint64_t w, uint32_t e, int lo, int hi) {
  const uint64_t x = (uint64_t)(1023 + lo + (int)(e % (uint32_t)(hi - lo))) << 52;
  return __longlong_as_double((long long)(x | (w >> 12)));
}
// `ulps` representable numbers above x > 0
__device__ double Next(double x, int ulps) { return __longlong_as_double(__double_as_longlong(x) + ulps); }

__device__ void Words(uint32_t i, uint32_t k, uint32_t key, uint32_t w[4]) {
  w[0] = i;
  w[1] = k;
  w[2] = w[3] = 0u;
  philox4x32_10(w, key, 0xD1Fu);
}

__global__ void k_small_float(uint32_t* bad) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  for (uint32_t m = i; m < (1u << 23); m += kBlocks * kThreads) {
    for (int n = 1; n <= kPoissonSmall; ++n) {
      const int e = 127 - 40 + (int)((m + (uint32_t)n) % 60u);
      const float a = __uint_as_float(((uint32_t)e << 23) | m);
      if (__float_as_uint(DivSmall(a, n)) != __float_as_uint(a / (float)n)) atomicAdd(bad, 1u);
    }
  }
  if (i < kPoissonSmall && DivSmall(0.0f, (int)i + 1) != 0.0f) atomicAdd(bad, 1u);
}

__global__ void k_small_double(uint32_t* bad) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  for (uint32_t k = 0; k < kPerThread; ++k) {
    uint32_t w[4];
    Words(i, k, 1u, w);
    const double r = Random(((uint64_t)w[1] << 32) | w[0], w[2], -60, 20);
    for (int n = 1; n <= kPoissonSmall; ++n) {
      const double a = (k & 1u) ? r : Next(r * (double)n, (int)(w[3] % 9u) - 4);
      if (__double_as_longlong(DivSmall(a, n)) != __double_as_longlong(a / (double)n)) atomicAdd(bad, 1u);
    }
  }
}

__global__ void k_in_range(uint32_t* bad) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  for (uint32_t k = 0; k < 16u * kPerThread; ++k) {
    uint32_t w[4], v[4];
    Words(i, k, 2u, w);
    Words(i, k, 3u, v);
    const double b = Random(((uint64_t)w[1] << 32) | w[0], w[2], -8, 12);
    const double q = Random(((uint64_t)v[1] << 32) | v[0], v[2], -200, 40);
    double a = (k & 1u) ? q : Next(q * b, (int)(v[3] % 9u) - 4);
    a = (w[3] & 1u) ? -a : a;
    if (__double_as_longlong(DivInRange(a, b)) != __double_as_longlong(a / b)) atomicAdd(bad, 1u);
    if (__double_as_longlong(DivInRange(0.0, b)) != 0) atomicAdd(bad, 1u);
  }
}

void Check(hipError_t e) {
  if (e != hipSuccess) {
    std::printf("%s\n", hipGetErrorString(e));
    std::exit(1);
  }
}

}  // namespace

int main() {
  uint32_t* bad;
  Check(hipMalloc(&bad, 3 * sizeof(uint32_t)));
  const uint32_t none[3] = {0u, 0u, 0u};
  Check(hipMemcpy(bad, none, sizeof none, hipMemcpyHostToDevice));
  hipLaunchKernelGGL(k_small_float, dim3(kBlocks), dim3(kThreads), 0, 0, bad);
  hipLaunchKernelGGL(k_small_double, dim3(kBlocks), dim3(kThreads), 0, 0, bad + 1);
  hipLaunchKernelGGL(k_in_range, dim3(kBlocks), dim3(kThreads), 0, 0, bad + 2);
  Check(hipGetLastError());
  uint32_t n[3];
  Check(hipMemcpy(n, bad, sizeof n, hipMemcpyDeviceToHost));
  Check(hipFree(bad));
  std::printf("differences: DivSmall float %u, double %u, DivInRange %u\n", n[0], n[1], n[2]);
  if (n[0] || n[1] || n[2]) return 1;
  std::printf("ALL OK\n");
  return 0;
}
