// What the bf16/fp16 selection kernels share: the exact score and the error
// bound that certifies decisions taken from MFMA scores.
#pragma once
#include "common.h"

namespace va {

// Canonical score from global memory: sequential fp64 FMAs over d (exact
// products), one rounding to fp32.
template <typename T, int D>
__device__ inline float exact_dot_global(const T* __restrict__ q, const T* __restrict__ k) {
  uint4 qr[D / 8], kr[D / 8];
#pragma unroll
  for (int c = 0; c < D / 8; ++c) {
    qr[c] = *reinterpret_cast<const uint4*>(q + 8 * c);
    kr[c] = *reinterpret_cast<const uint4*>(k + 8 * c);
  }
  double acc = 0.0;
#pragma unroll
  for (int c = 0; c < D / 8; ++c) {
    const T* qv = reinterpret_cast<const T*>(&qr[c]);
    const T* kv = reinterpret_cast<const T*>(&kr[c]);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc = __builtin_fma(double(to_f32(qv[e])), double(to_f32(kv[e])), acc);
  }
  return float(acc);
}

// Bounds of one pooled row, from the fp64 sum ss of its squares, the largest
// key norm kn (key_norm_bound) and the gap.  With delta the largest distance
// between an MFMA score and the exact sum and A = |q| max|k|: a key whose
// distance to the threshold exceeds `band` is decided by its MFMA score, and
// only keys within `win` of the largest MFMA score can hold the exact maximum.
// certified: every score is finite and far from overflow, and so are the
// bounds; infinities and NaNs among the row's values, the head's keys
// (key_norm_bound is then infinite) or the gaps make it false.  The kernels read
// signs and bit patterns of differences, which are never NaN only where it is
// true; of the other rows they send every key to their exact path.
struct Bounds {
  float band, win;
  bool certified;
};
template <int D>
__device__ inline Bounds score_bounds(double ss, float kn, float gap) {
  const double A = __builtin_sqrt(ss) * (1.0 + 0x1p-20) * double(kn) * (1.0 + 0x1p-20);
  const double delta = double(2 * (D / 16 + 2) + 1) * 0x1p-23 * A;
  const double ag = __builtin_fabs(double(gap));
  Bounds r;
  r.band = float(1.25 * (2.0 * delta + 6.0 * 0x1p-24 * (A + ag)) + 1e-28);
  r.win = float(1.25 * (2.0 * delta + 4.0 * 0x1p-24 * A) + 1e-28);
  if (!(A < 0x1p100)) r.win = __builtin_inff();  // any key can hold the maximum
  r.certified = A + ag < 0x1p100;
  return r;
}

}  // namespace va
