// Block-mean pooling of the queries, fused with the selection's query scaling.
//
// Follows spattn/src/utils.py:340-351 (average_vector: fp32 mean over qps rows,
// the last block divided by its real row count, result cast back to the input
// dtype) and spattn/src/kernels/vecattention_kernels.py:94,244-245 (the
// selection multiplies the pooled rows by fp32(1/sqrt(D)) and rounds back to
// the input dtype before the score product).
//
// Canonical arithmetic: rows are summed sequentially in fp64, the sum is
// rounded to fp32, divided in fp32 by the real row count, and rounded to the
// element type.  The divide runs in fp64 and is rounded once to fp32, which is
// the correctly rounded fp32 quotient of two fp32 operands.
//
// HBM-bound: each Q element is read once.  A thread owns VEC consecutive
// features of one pooled row, so 16-byte loads of a full Q row are coalesced
// across D/VEC neighbouring threads, and keeps U rows' loads in flight.
#include "common.h"
#include "key_norm.h"

namespace va {

// Work-group `blk` (of kThreads threads) of head bh: kThreads / (D / VEC)
// pooled rows.
template <typename T, int VEC, int U>
__device__ inline void pool_rows(const T* __restrict__ q, uint32_t H, int64_t S, uint32_t D,
                                 int64_t sqb, int64_t sqh, int64_t sqs, int64_t qps, int64_t nqb,
                                 float sm, T* __restrict__ pooled, T* __restrict__ scaled,
                                 uint32_t blk, uint32_t bh) {
  const uint32_t lanes_per_row = D / VEC;
  const uint32_t rows_per_block = blockDim.x / lanes_per_row;
  const uint32_t local = threadIdx.x / lanes_per_row;
  const uint32_t dv = (threadIdx.x % lanes_per_row) * VEC;
  const int64_t J = int64_t(blk) * rows_per_block + local;
  if (local >= rows_per_block || J >= nqb) return;
  const uint32_t b = bh / H, h = bh % H;
  const int64_t r0 = J * qps;
  const int rows = int((S - r0 < qps) ? (S - r0) : qps);
  const T* src = q + b * sqb + h * sqh + r0 * sqs + dv;

  double acc[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) acc[e] = 0.0;

  auto load = [&](T (&v)[VEC], int r) {
    if constexpr (VEC * sizeof(T) == 16) {
      *reinterpret_cast<uint4*>(v) = *reinterpret_cast<const uint4*>(src + r * sqs);
    } else {
#pragma unroll
      for (int e = 0; e < VEC; ++e) v[e] = src[r * sqs + e];
    }
  };
  // Rows are loaded U at a time (U loads in flight per thread) and added in
  // row order, so the sums are those of the sequential loop.
  int r = 0;
  for (; r + U <= rows; r += U) {
    T v[U][VEC];
#pragma unroll
    for (int u = 0; u < U; ++u) load(v[u], r + u);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < VEC; ++e) acc[e] += double(to_f32(v[u][e]));
  }
  if (r < rows) {  // the last block's remainder: the loads past it read its last row
    T v[U][VEC];
#pragma unroll
    for (int u = 0; u < U; ++u) load(v[u], r + u < rows ? r + u : rows - 1);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (r + u < rows)
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[e] += double(to_f32(v[u][e]));
  }

  const int64_t o = (int64_t(bh) * nqb + J) * D + dv;
#pragma unroll
  for (int e = 0; e < VEC; ++e) {
    const float sum32 = float(acc[e]);
    const float mean32 = float(double(sum32) / double(rows));
    const float p = Round<T>::rt(mean32);
    if (pooled) pooled[o + e] = Round<T>::store(p);
    if (scaled) scaled[o + e] = Round<T>::store(p * sm);
  }
}

template <typename T, int VEC, int U>
__global__ __launch_bounds__(256) void pool_scale_kernel(
    const T* __restrict__ q, uint32_t H, int64_t S, uint32_t D, int64_t sqb, int64_t sqh,
    int64_t sqs, int64_t qps, int64_t nqb, float sm, T* __restrict__ pooled,
    T* __restrict__ scaled) {
  pool_rows<T, VEC, U>(q, H, S, D, sqb, sqh, sqs, qps, nqb, sm, pooled, scaled, blockIdx.x,
                       blockIdx.y);
}

constexpr int kPoolThreads = 128;

// The prefill's first launch: the pooled queries and, in the work-groups
// after them, the partial key norms.  Both only read their input, and beside
// each other they hide what each waits for: 22.8 -> 9.2 us at 2333 keys of 28
// heads, 34 -> 25 us at 16411, 62 -> 56 us at 32768, 48 -> 36 us at 32760 of
// 12 unshared heads (pooling, partial norms and their reduction as three
// launches before; the selection reduces the partials itself now).
// Zeroes the work queues of the prefill's attention launches, if given.
template <typename T, int VPR, int U>
__global__ __launch_bounds__(kPoolThreads) void pool_norm_kernel(
    const T* __restrict__ q, uint32_t H, int64_t S, int64_t sqb, int64_t sqh, int64_t sqs,
    int64_t qps, int64_t nqb, float sm, T* __restrict__ scaled, uint32_t pool_blocks, uint32_t BH,
    const T* __restrict__ k, int64_t skb, int64_t skh, int64_t sks, int64_t Hk, int64_t Sk,
    float* __restrict__ partial, uint32_t* __restrict__ queue) {
  constexpr uint32_t kD = VPR * 16 / sizeof(T);
  const uint32_t np = pool_blocks * BH;
  if (queue && blockIdx.x == np)
    for (uint32_t i = threadIdx.x; i < kQueueSets * WorkOrder::kQueueWords; i += kPoolThreads)
      queue[i] = 0u;
  if (blockIdx.x < np) {
    pool_rows<T, int(16 / sizeof(T)), U>(q, H, S, kD, sqb, sqh, sqs, qps, nqb, sm, nullptr, scaled,
                                         blockIdx.x % pool_blocks, blockIdx.x / pool_blocks);
  } else {
    const uint32_t i = blockIdx.x - np;
    key_norm_part_vec<T, VPR, kPoolThreads / 64>(k, skb, skh, sks, Hk, Sk, i / kNormParts,
                                                 i % kNormParts, partial);
  }
}

// Work-groups below which a pooling launch leaves the chip partly idle.
constexpr int64_t kFewPoolGroups = 512;

// Loads in flight per thread: 8 where the launch fills the chip (bound by
// HBM: 5.5 TB/s on 128K x 28 heads), more below that, where a work-group's
// serial round trips are what the launch takes: 32 alone, 16 beside the key
// norms, whose waves share the registers (with 32: 98 us instead of 36 at
// 32760 keys of 12 heads, 34 instead of 25 at 16411 of 28).
static bool few_pool_groups(int64_t groups) { return groups < kFewPoolGroups; }

// 16-byte rows of 16-bit or fp32 queries.
template <typename T>
static bool pool_vec_ok(const void* q, int64_t D, int64_t sqb, int64_t sqh, int64_t sqs) {
  constexpr int V16 = int(16 / sizeof(T));
  return D % V16 == 0 && reinterpret_cast<uintptr_t>(q) % 16 == 0 && sqb % V16 == 0 &&
         sqh % V16 == 0 && sqs % V16 == 0;
}

template <typename T>
static hipError_t launch_pool_t(const void* q, int64_t B, int64_t H, int64_t S,
                                int64_t D, int64_t sqb, int64_t sqh, int64_t sqs,
                                int64_t qps, void* pooled, void* scaled,
                                hipStream_t stream) {
  const int64_t nqb = (S + qps - 1) / qps;
  const float sm = float(1.0 / __builtin_sqrt(double(D)));
  constexpr int V16 = int(16 / sizeof(T));
  auto go = [&](auto kernel, int threads, int64_t rows_per_block) {
    const dim3 grid(unsigned((nqb + rows_per_block - 1) / rows_per_block), unsigned(B * H));
    hipLaunchKernelGGL(kernel, grid, dim3(threads), 0, stream, static_cast<const T*>(q),
                       uint32_t(H), S, uint32_t(D), sqb, sqh, sqs, qps, nqb, sm,
                       static_cast<T*>(pooled), static_cast<T*>(scaled));
  };
  if (pool_vec_ok<T>(q, D, sqb, sqh, sqs)) {  // D / V16 <= 64 lanes per row (D <= 256)
    // 128 threads per work-group measured 3-6% faster than 256 at 32K and 128K keys.
    const int64_t rows_per_block = kPoolThreads / (D / V16);
    if (few_pool_groups((nqb + rows_per_block - 1) / rows_per_block * B * H))
      go(pool_scale_kernel<T, V16, 32>, kPoolThreads, rows_per_block);
    else
      go(pool_scale_kernel<T, V16, 8>, kPoolThreads, rows_per_block);
  } else {
    go(pool_scale_kernel<T, 1, 8>, 256, 256 / D);  // one thread per feature, D <= 256
  }
  return hipGetLastError();
}

hipError_t launch_pool(int dtype, const void* q, int64_t B, int64_t H, int64_t S,
                       int64_t D, int64_t sqb, int64_t sqh, int64_t sqs, int64_t qps,
                       void* pooled, void* scaled, hipStream_t stream) {
  switch (dtype) {
    case kF32: return launch_pool_t<float>(q, B, H, S, D, sqb, sqh, sqs, qps, pooled, scaled, stream);
    case kBF16: return launch_pool_t<bf16_t>(q, B, H, S, D, sqb, sqh, sqs, qps, pooled, scaled, stream);
    case kF16: return launch_pool_t<f16_t>(q, B, H, S, D, sqb, sqh, sqs, qps, pooled, scaled, stream);
  }
  return hipErrorInvalidValue;
}

template <typename T>
static hipError_t launch_pool_norm_t(const void* q, int64_t B, int64_t H, int64_t S, int64_t D,
                                     int64_t sqb, int64_t sqh, int64_t sqs, int64_t qps,
                                     void* scaled, const void* k, int64_t skb, int64_t skh,
                                     int64_t sks, int64_t Hk, int64_t Sk, float* partial,
                                     uint32_t* queue, hipStream_t stream) {
  const int64_t nqb = (S + qps - 1) / qps;
  const float sm = float(1.0 / __builtin_sqrt(double(D)));
  const int64_t rows_per_block = kPoolThreads / (D / 8);
  const int64_t pool_blocks = (nqb + rows_per_block - 1) / rows_per_block;
  const int64_t np = pool_blocks * B * H;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(unsigned(np + kNormParts * B * Hk)), dim3(kPoolThreads), 0,
                       stream, static_cast<const T*>(q), uint32_t(H), S, sqb, sqh, sqs, qps, nqb,
                       sm, static_cast<T*>(scaled), uint32_t(pool_blocks), uint32_t(B * H),
                       static_cast<const T*>(k), skb, skh, sks, Hk, Sk, partial, queue);
    return hipGetLastError();
  };
  if (few_pool_groups(np))
    return D == 128 ? go(pool_norm_kernel<T, 16, 16>) : go(pool_norm_kernel<T, 8, 16>);
  return D == 128 ? go(pool_norm_kernel<T, 16, 8>) : go(pool_norm_kernel<T, 8, 8>);
}

// Whether the fused launch takes these operands (bf16/fp16, head_dim 64 or
// 128, 16-byte rows of q and k).
bool pool_norm_supported(int dtype, const void* q, int64_t B, int64_t H, int64_t S, int64_t D,
                         int64_t sqb, int64_t sqh, int64_t sqs, int64_t qps, const void* k,
                         int64_t skb, int64_t skh, int64_t sks, int64_t Hk) {
  if ((dtype != kBF16 && dtype != kF16) || (D != 64 && D != 128)) return false;
  const int64_t nqb = (S + qps - 1) / qps;  // at most nqb work-groups per head
  return pool_vec_ok<bf16_t>(q, D, sqb, sqh, sqs) && pool_vec_ok<bf16_t>(k, D, skb, skh, sks) &&
         nqb * B * H + kNormParts * B * Hk < (int64_t(1) << 31);
}

// Scaled pooled queries and partial key norms (key_norm_bound) in one launch.
hipError_t launch_pool_norm(int dtype, const void* q, int64_t B, int64_t H, int64_t S, int64_t D,
                            int64_t sqb, int64_t sqh, int64_t sqs, int64_t qps, void* scaled,
                            const void* k, int64_t skb, int64_t skh, int64_t sks, int64_t Hk,
                            int64_t Sk, float* partial, uint32_t* queue, hipStream_t stream) {
  if (dtype == kBF16)
    return launch_pool_norm_t<bf16_t>(q, B, H, S, D, sqb, sqh, sqs, qps, scaled, k, skb, skh, sks,
                                      Hk, Sk, partial, queue, stream);
  if (dtype == kF16)
    return launch_pool_norm_t<f16_t>(q, B, H, S, D, sqb, sqh, sqs, qps, scaled, k, skb, skh, sks,
                                     Hk, Sk, partial, queue, stream);
  return hipErrorInvalidValue;
}

}  // namespace va
