// Key-norm bound of the certified selections: device pieces shared by the
// standalone launch (key_norm.hip), the prefill's fused first launch
// (pool.hip) and the selection kernels that read the result.
#pragma once
#include "common.h"

namespace va {

constexpr int kNormParts = 256;  // key ranges per (b, kv head), one partial maximum each

// Partial maximum `part` of head bh: the largest squared key norm of its key
// range.  Rows of 16-byte vectors: lane l of a wave reads vector l % VPR of
// row l / VPR of each group of 64 / VPR rows (coalesced 1 KB per load
// instruction); the squared norm of a row is summed over its VPR lanes.
// Called by whole work-groups of kWaves waves.
template <typename T, int VPR, int kWaves>
__device__ inline void key_norm_part_vec(const T* __restrict__ k, int64_t skb, int64_t skh,
                                         int64_t sks, int64_t Hk, int64_t Sk, int64_t bh,
                                         int64_t part, float* __restrict__ partial) {
  constexpr int RPW = 64 / VPR;  // rows per wave load
  const int64_t b = bh / Hk, h = bh % Hk;
  const T* kh = k + b * skb + h * skh;
  const int64_t per = (Sk + kNormParts - 1) / kNormParts;
  const int64_t k0 = part * per;
  const int64_t k1 = (k0 + per < Sk) ? k0 + per : Sk;
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int r = lane / VPR, v = lane % VPR;
  double best = 0.0;
  // kLoads groups of rows at a time (their loads in flight together); rows
  // past the range read its last row again, which leaves the maximum as it is.
  // `base` is the same for every lane of the wave, so the shuffles below run
  // with the whole wave active.
  constexpr int kLoads = 4;
  for (int64_t base = k0 + wave * RPW; base < k1; base += kLoads * kWaves * RPW) {
    uint4 raw[kLoads];
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const int64_t key = base + u * kWaves * RPW + r;
      raw[u] = *reinterpret_cast<const uint4*>(kh + (key < k1 ? key : k1 - 1) * sks +
                                               v * (16 / sizeof(T)));
    }
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const T* e = reinterpret_cast<const T*>(&raw[u]);
      double ss = 0.0;
#pragma unroll
      for (int i = 0; i < int(16 / sizeof(T)); ++i) {
        const double x = double(to_f32(e[i]));
        ss = __builtin_fma(x, x, ss);
      }
#pragma unroll
      for (int o = 1; o < VPR; o <<= 1) ss += __shfl_xor(ss, o);  // sum over the row's lanes
      ss = ss == ss ? ss : __builtin_inf();  // a NaN bounds nothing
      best = ss > best ? ss : best;
    }
  }
#pragma unroll
  for (int o = VPR; o < 64; o <<= 1) {  // maximum over the wave's rows
    const double x = __shfl_xor(best, o);
    best = x > best ? x : best;
  }
  __shared__ double red[kWaves];
  if (lane == 0) red[wave] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < kWaves; ++w) best = red[w] > best ? red[w] : best;
    partial[bh * kNormParts + part] = float(best);
  }
}

// Upper bound of the key norms of head bh from its partial maxima, for whole
// waves: every lane gets the value.  Each selection work-group reads the 1 KB
// of partials itself; a launch of its own that reduced them took 7 us.
__device__ inline float key_norm_bound(const float* __restrict__ partial, int64_t bh) {
  const int lane = threadIdx.x % 64;
  const float* p = partial + bh * kNormParts + lane;
  float best = 0.f;
#pragma unroll
  for (int i = 0; i < kNormParts / 64; ++i) best = __builtin_fmaxf(best, p[64 * i]);
  // Non-negative floats order as their bit patterns; lanes a DPP move does not
  // reach read 0 (the shifts and broadcasts of wave_inclusive_sum).
  uint32_t u = float_to_bits(best);
  auto fold = [&](uint32_t x) { u = x > u ? x : u; };
  fold(__builtin_amdgcn_update_dpp(0, u, 0x111, 0xf, 0xf, false));  // row_shr:1
  fold(__builtin_amdgcn_update_dpp(0, u, 0x112, 0xf, 0xf, false));  // row_shr:2
  fold(__builtin_amdgcn_update_dpp(0, u, 0x114, 0xf, 0xf, false));  // row_shr:4
  fold(__builtin_amdgcn_update_dpp(0, u, 0x118, 0xf, 0xf, false));  // row_shr:8
  fold(__builtin_amdgcn_update_dpp(0, u, 0x142, 0xa, 0xf, false));  // row_bcast:15
  fold(__builtin_amdgcn_update_dpp(0, u, 0x143, 0xc, 0xf, false));  // row_bcast:31
  best = bits_to_float(__builtin_amdgcn_readlane(u, 63));
  // square root of an upper bound of the squared norm, rounded up generously
  return float(__builtin_sqrt(double(best)) * (1.0 + 0x1p-20));
}

}  // namespace va
