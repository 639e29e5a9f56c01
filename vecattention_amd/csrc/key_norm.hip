// Per-(batch, kv head) maximum key norm, rounded up: the K-side factor of the
// error bound the MFMA selection kernels certify their decisions with
// (|s_mfma - s| <= gamma * ||q|| * max_c ||k_c||).
//
// One launch of partial maxima over kNormParts key ranges per head, no atomics
// and no memset; the selection kernels reduce the partials themselves
// (key_norm_bound).  HBM-bound (reads K once); the squared norms are summed in
// fp64 (exact products of the 16-bit inputs).
#include "key_norm.h"

namespace va {

template <typename T, int VPR>
__global__ __launch_bounds__(256) void key_norm_partial_vec_kernel(
    const T* __restrict__ k, int64_t skb, int64_t skh, int64_t sks, int64_t Hk, int64_t Sk,
    float* __restrict__ partial) {
  key_norm_part_vec<T, VPR, 4>(k, skb, skh, sks, Hk, Sk, blockIdx.y, blockIdx.x, partial);
}

// Any layout: one row per thread, element by element.
template <typename T>
__global__ __launch_bounds__(256) void key_norm_partial_kernel(
    const T* __restrict__ k, int64_t skb, int64_t skh, int64_t sks, int64_t Hk, int64_t Sk,
    int64_t D, float* __restrict__ partial) {
  const int64_t bh = blockIdx.y;
  const int64_t b = bh / Hk, h = bh % Hk;
  const T* kh = k + b * skb + h * skh;
  const int64_t per = (Sk + kNormParts - 1) / kNormParts;
  const int64_t k0 = int64_t(blockIdx.x) * per;
  const int64_t k1 = (k0 + per < Sk) ? k0 + per : Sk;
  double best = 0.0;
  for (int64_t key = k0 + threadIdx.x; key < k1; key += blockDim.x) {
    const T* kr = kh + key * sks;
    double ss = 0.0;
    for (int64_t d = 0; d < D; ++d) {
      const double x = double(to_f32(kr[d]));
      ss = __builtin_fma(x, x, ss);
    }
    ss = ss == ss ? ss : __builtin_inf();  // a NaN bounds nothing
    best = ss > best ? ss : best;
  }
  __shared__ double red[256];
  red[threadIdx.x] = best;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (int(threadIdx.x) < s) {
      const double o = red[threadIdx.x + s];
      if (o > red[threadIdx.x]) red[threadIdx.x] = o;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[bh * kNormParts + blockIdx.x] = float(red[0]);
}

template <typename T>
static hipError_t launch_key_norm_t(const void* k, int64_t skb, int64_t skh, int64_t sks,
                                    int64_t B, int64_t Hk, int64_t Sk, int64_t D, float* partial,
                                    hipStream_t stream) {
  const dim3 grid(kNormParts, unsigned(B * Hk));
  const T* kp = static_cast<const T*>(k);
  const int64_t row_bytes = D * int64_t(sizeof(T)), a = 16 / int64_t(sizeof(T));
  const bool vec = reinterpret_cast<uintptr_t>(k) % 16 == 0 && skb % a == 0 && skh % a == 0 &&
                   sks % a == 0 && row_bytes % 16 == 0;
  const int64_t vpr = row_bytes / 16;
  if (vec && vpr == 8)
    hipLaunchKernelGGL((key_norm_partial_vec_kernel<T, 8>), grid, dim3(256), 0, stream, kp, skb,
                       skh, sks, Hk, Sk, partial);
  else if (vec && vpr == 16)
    hipLaunchKernelGGL((key_norm_partial_vec_kernel<T, 16>), grid, dim3(256), 0, stream, kp, skb,
                       skh, sks, Hk, Sk, partial);
  else if (vec && vpr == 32)
    hipLaunchKernelGGL((key_norm_partial_vec_kernel<T, 32>), grid, dim3(256), 0, stream, kp, skb,
                       skh, sks, Hk, Sk, partial);
  else
    hipLaunchKernelGGL((key_norm_partial_kernel<T>), grid, dim3(256), 0, stream, kp, skb, skh,
                       sks, Hk, Sk, D, partial);
  return hipGetLastError();
}

int64_t key_norm_scratch_floats(int64_t B, int64_t Hk) { return B * Hk * kNormParts; }

// scratch: key_norm_scratch_floats(B, Hk) floats; kNormParts partial squared
// norms per head, from the first float on.
hipError_t launch_key_norm(int dtype, const void* k, int64_t skb, int64_t skh, int64_t sks,
                           int64_t B, int64_t Hk, int64_t Sk, int64_t D, float* scratch,
                           hipStream_t stream) {
  switch (dtype) {
    case kF32: return launch_key_norm_t<float>(k, skb, skh, sks, B, Hk, Sk, D, scratch, stream);
    case kBF16: return launch_key_norm_t<bf16_t>(k, skb, skh, sks, B, Hk, Sk, D, scratch, stream);
    case kF16: return launch_key_norm_t<f16_t>(k, skb, skh, sks, B, Hk, Sk, D, scratch, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace va
