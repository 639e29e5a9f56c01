// fp32 -> bf16 copy that reports whether every value was a bf16 value.
//
// The tuner's fp32 copies of 16-bit queries and keys (model_tuner.py:53-77) hold
// bf16 values and then take the bf16 kernels.  One pass, 6 bytes moved a value
// (HBM-bound: 12 heads of 32760 rows and 128 features 58 us); converting,
// converting back and comparing with library calls moved 30 in 300 us.
#include "common.h"

namespace va {

__global__ __launch_bounds__(256) void bf16_copy_kernel(const float* __restrict__ x, int64_t n,
                                                        uint16_t* __restrict__ out,
                                                        int32_t* __restrict__ inexact) {
  const int64_t i = (int64_t(blockIdx.x) * 256 + threadIdx.x) * 8;
  bool bad = false;
  // A value is kept when its low 16 bits are zero (NaNs count as changed: they
  // equal nothing).
  auto bits = [&](float f) {
    bad |= (float_to_bits(f) & 0xffffu) != 0u || f != f;
    return uint32_t(rne_bf16_bits(f));
  };
  if (i + 8 <= n) {
    const float4 a = *reinterpret_cast<const float4*>(x + i);
    const float4 b = *reinterpret_cast<const float4*>(x + i + 4);
    uint4 w;
    w.x = bits(a.x) | (bits(a.y) << 16);
    w.y = bits(a.z) | (bits(a.w) << 16);
    w.z = bits(b.x) | (bits(b.y) << 16);
    w.w = bits(b.z) | (bits(b.w) << 16);
    *reinterpret_cast<uint4*>(out + i) = w;
  } else {
    for (int64_t j = i; j < n; ++j) out[j] = uint16_t(bits(x[j]));
  }
  if (bad) *inexact = 1;  // every writer writes the same value
}

hipError_t launch_bf16_copy(const float* x, int64_t n, void* out, int32_t* inexact,
                            hipStream_t stream) {
  hipLaunchKernelGGL(bf16_copy_kernel, dim3(unsigned((n + 2047) / 2048)), dim3(256), 0, stream, x,
                     n, static_cast<uint16_t*>(out), inexact);
  return hipGetLastError();
}

}  // namespace va
