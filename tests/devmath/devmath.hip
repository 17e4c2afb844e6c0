// Test-only device build of svo_math.hpp's reciprocal, quotient and root
// without the handling of extreme exponents.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../shocovox_amd/csrc/svo_math.hpp"

// op 0: rcp_mid(b), 1: quot_mid(a, b, rcp_mid(b)), 2: sqrt_mid(b)
__global__ __launch_bounds__(256) void devmath_kernel(int op, const float* __restrict__ a,
                                                      const float* __restrict__ b,
                                                      float* __restrict__ out, uint32_t n) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n) return;
#if defined(__HIP_DEVICE_COMPILE__)
  out[i] = op == 0 ? svo::rcp_mid(b[i])
                   : (op == 1 ? svo::quot_mid(a[i], b[i], svo::rcp_mid(b[i])) : svo::sqrt_mid(b[i]));
#endif
}

// Device arrays of n floats, n < 2^31 (a only for op 1); 0 or a HIP error.
extern "C" int devmath(int op, const float* a, const float* b, float* out, uint32_t n,
                       void* stream) {
  if (n == 0) return 0;
  if (op < 0 || op > 2 || !b || !out || (op == 1 && !a) || n >= 1u << 31)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(devmath_kernel, dim3((n + 255u) / 256u), dim3(256), 0,
                     static_cast<hipStream_t>(stream), op, a, b, out, n);
  return hipGetLastError();
}
