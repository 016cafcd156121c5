// Test probe: the device arithmetic of gartus_amd/csrc/device.h beside the compiler's operators, element by element.
// Built in-tree by gartus_amd.build, loaded by tests/test_gpu_device_math.py.
#include <hip/hip_runtime.h>

#include "../gartus_amd/csrc/device.h"

using namespace gtd;

namespace {

// Mantissa and exponent field of element i of a sweep over all 2^23 mantissas of one exponent.
__device__ __forceinline__ float sweep(uint32_t i, uint32_t exponent, uint32_t sign) {
  return __uint_as_float(sign << 31 | exponent << 23 | i);
}

__global__ void k_unary(int op, uint32_t exponent, uint32_t sign, unsigned long long* bad) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;  // 2^23 threads
  const float x = sweep(i, exponent, sign);
  const float got = op == 0 ? rcp_rn(x) : op == 1 ? reciprocal(x) : sqrt_rn(x);
  const float want = op < 2 ? 1.0f / x : sqrtf(x);
  if (__float_as_uint(got) != __float_as_uint(want)) atomicAdd(bad, 1ull);
}

// n / d with all mantissas of the divisor (or d itself when fixed != 0) and a hashed numerator of exponent ne.
__global__ void k_div(uint32_t de, uint32_t ne, uint32_t seed, float fixed, unsigned long long* bad) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  const float d = fixed != 0.f ? fixed : sweep(i, de, 0);
  const uint32_t m = uint32_t(mix64(uint64_t(seed) << 32 | i)) & 0x7fffffu;
  const float n = sweep(fixed != 0.f ? i : m, ne, (seed ^ i) & 1u);
  if (__float_as_uint(div_rn(n, d, reciprocal(d))) != __float_as_uint(n / d)) atomicAdd(bad, 1ull);
}

__global__ void k_div31(Div31 k, const uint32_t* n, uint32_t* out, uint32_t count) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  uint32_t rem;
  out[2 * i] = div31(n[i], k, &rem);
  out[2 * i + 1] = rem;
}

__global__ void k_normalized(const float* in, float* out, uint32_t count) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const f3 a = mk(in[3 * i], in[3 * i + 1], in[3 * i + 2]);
  const f3 got = normalized(a);
  const float l = sqrtf(len2(a));
  const f3 want = l < EPS ? mk(0.f, 0.f, 0.f) : mk(a.x / l, a.y / l, a.z / l);
  out[6 * i] = got.x; out[6 * i + 1] = got.y; out[6 * i + 2] = got.z;
  out[6 * i + 3] = want.x; out[6 * i + 4] = want.y; out[6 * i + 5] = want.z;
}

constexpr uint32_t kMantissas = 1u << 23;

}  // namespace

// All pointers are device memory. op 0 rcp_rn, 1 reciprocal, 2 sqrt_rn; returns the HIP status.
extern "C" int probe_unary(int op, uint32_t exponent, uint32_t sign, unsigned long long* bad) {
  hipLaunchKernelGGL(k_unary, dim3(kMantissas / 256), dim3(256), 0, 0, op, exponent, sign, bad);
  return int(hipGetLastError());
}
extern "C" int probe_div(uint32_t de, uint32_t ne, uint32_t seed, float fixed, unsigned long long* bad) {
  hipLaunchKernelGGL(k_div, dim3(kMantissas / 256), dim3(256), 0, 0, de, ne, seed, fixed, bad);
  return int(hipGetLastError());
}
extern "C" int probe_div31(uint32_t d, const uint32_t* n, uint32_t* out, uint32_t count) {
  hipLaunchKernelGGL(k_div31, dim3((count + 255) / 256), dim3(256), 0, 0, make_div31(d), n, out, count);
  return int(hipGetLastError());
}
extern "C" int probe_normalized(const float* in, float* out, uint32_t count) {
  hipLaunchKernelGGL(k_normalized, dim3((count + 255) / 256), dim3(256), 0, 0, in, out, count);
  return int(hipGetLastError());
}
