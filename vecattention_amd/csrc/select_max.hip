// Maxima pass of the two-pass selection (rows that are one group long) on
// bf16/fp16 MFMA: per (pooled row, key segment), what select_wave.hip's carry
// pass needs to start a later segment of the row: the segment's MFMA maximum
// and either the one tile that holds its exact maximum or that exact maximum.
//
// A key can only hold the exact maximum when its MFMA score is within `win` of
// the MFMA maximum (select_wave.hip).  A lane keeps the three largest 16-key
// maxima it has seen and where the first two were, ten VALU instructions a
// piece beside the maximum itself, where the selection kernel's own maxima mode
// carried its near-max lists and registers along.  When neither lane's third
// largest reaches the row's largest minus `win`, the candidates are those (up to
// four) tiles; otherwise (equal keys, or a threefold near tie) the wave walks
// the segment once more and takes the exact scores of every piece within `win`.
// Keeping one candidate sent one wave in sixty on that walk, which then lasted
// as long as the launch.  The walk takes its exact scores 16 rows by 16 keys at
// a time from the fp64 matrix cores: where a fifth of 32760 keys are one key
// (padding), this pass takes 2.2 ms, 6.8 ms with a key per lane on the vector
// units, 3.9 ms in the selection kernel's own maxima mode.
//
// 128 rows per work-group (4 waves of 32), K in chunks of 64 keys through LDS
// (three stages), at 80% of a library GEMM's rate: 512 rows of 24 heads over
// 119056 keys of 128 features 343 us (1.09 PFLOP/s; 600 us in the selection
// kernel), 512 rows of 12 heads over 32760 keys 60 us (115).
#include <type_traits>

#include "key_norm.h"
#include "lanes.h"
#include "mfma.h"
#include "select_carry.h"
#include "select_cert.h"

namespace va {

typedef double f64x4_t __attribute__((ext_vector_type(4)));

constexpr int kMxWaves = 4, kMxRows = 32, kMxChunk = 64;

template <typename T, int D>
__global__ __launch_bounds__(256, 3) void select_max_kernel(
    const T* __restrict__ qs, int64_t sqb, int64_t sqh, int64_t sqn, const T* __restrict__ k,
    int64_t skb, int64_t skh, int64_t sks, int64_t B, int64_t Hq, int64_t Hk, int64_t Sk,
    int64_t qps, int bk, int causal, int64_t bsq, const float* __restrict__ kmax, RowLayout lay,
    int64_t nrowsets, int segk, int nseg, SegCarry* __restrict__ carry) {
  using M = Mfma<T>;
  using vec = typename M::vec;
  constexpr int NS = D / 16, ROWB = 2 * D, NCH = D / 8;
  constexpr int STAGE = kMxChunk * ROWB;
  constexpr int RPC = 1024 / ROWB;
  constexpr int H = STAGE / 1024 / kMxWaves;
  __shared__ __attribute__((aligned(1024))) unsigned char kst[3 * STAGE];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;
  const int l32 = lane % 32, hh = lane / 32;
  const WorkOrder wo{nrowsets * nseg, B, Hq, Hk, causal == 0};
  int item, bh32;
  if (!wo.map_item32(blockIdx.x, item, bh32)) return;  // idle block (uniform)
  const int64_t bh = bh32;
  const int rs = item / nseg, seg = item % nseg;
  const uint32_t hq32 = uint32_t(Hq);
  const int64_t b = uint32_t(bh32) / hq32, h = uint32_t(bh32) % hq32;
  const int64_t hk = uint32_t(h) / (hq32 / uint32_t(Hk));
  const int64_t nc = lay.nc, J0 = lay.J0;
  const int64_t jr_wave = int64_t(rs) * (kMxWaves * kMxRows) + kMxRows * wave;
  const int64_t jr = jr_wave + l32;
  const bool valid = jr < nc;
  const int sk = int(Sk);  // < 2^24 (host check)
  const int smin = int(lay.smin());

  // Keys up to the end of a row set's last selectable tile (select_wave.hip).
  auto range_end = [&](int64_t row) -> int {
    if (!causal) return sk;
    const int64_t J = J0 + row, lim = row % bsq == 0 ? (J - 1) * qps + 1 : J * qps;
    const int64_t e = ((lim < 0 ? 0 : lim) + bk - 1) / bk * bk;
    return int(e < Sk ? e : Sk);
  };
  const int64_t rows_wave = nc - jr_wave < kMxRows ? nc - jr_wave : kMxRows;
  const int64_t left = nc - int64_t(rs) * (kMxWaves * kMxRows);
  const int64_t rows_wg = left < kMxWaves * kMxRows ? left : kMxWaves * kMxRows;
  const int seg_lo = seg * segk, seg_hi = seg_lo + segk;
  int wave_end = rows_wave > 0 ? range_end(jr_wave + rows_wave - 1) : 0;
  int wg_end = range_end(int64_t(rs) * (kMxWaves * kMxRows) + rows_wg - 1);
  if (wave_end > seg_hi) wave_end = seg_hi;
  if (wg_end > seg_hi) wg_end = seg_hi;

  const T* qrow = qs + b * sqb + h * sqh + jr * sqn;
  vec qreg[NS];
  double ss = 0.0;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    uint4 raw = make_uint4(0, 0, 0, 0);
    if (valid) raw = *reinterpret_cast<const uint4*>(qrow + 16 * s + 8 * hh);
    qreg[s] = __builtin_bit_cast(vec, raw);
    const T* e8 = reinterpret_cast<const T*>(&raw);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const double x = double(to_f32(e8[e]));
      ss = __builtin_fma(x, x, ss);
    }
  }
  {
    const uint64_t u = __builtin_bit_cast(uint64_t, ss);
    const uint32_t lo = other_half(uint32_t(u)), hi = other_half(uint32_t(u >> 32));
    ss += __builtin_bit_cast(double, (uint64_t(hi) << 32) | lo);
  }
  const float kn = key_norm_bound(kmax, b * Hk + hk);
  const Bounds bounds = score_bounds<D>(ss, kn, 0.f);
  const float win = bounds.win;
  // As select_wave.hip: in a wave with an uncertified row every piece is scored
  // exactly.
  const bool exact_wave = __builtin_amdgcn_ballot_w64(valid && !bounds.certified) != 0;

  // K copies and operand reads: the layout of select_wave.hip.
  const T* kh = k + b * skb + hk * skh;
  const uint32_t krb = uint32_t(sks * 2);
  const __amdgpu_buffer_rsrc_t krs = make_rsrc(kh, uint32_t(((Sk - 1) * sks + D) * 2));
  const uint32_t kst_lds = lds_addr(kst);
  auto kperm = [](int m) { return 16 * ((m >> 2) & 1) + 4 * (m >> 3) + (m & 3); };
  uint32_t coff[H];
#pragma unroll
  for (int x = 0; x < H; ++x) {
    const int R = (wave * H + x) * RPC + lane / NCH;
    coff[x] = uint32_t(32 * (R / 32) + kperm(R % 32)) * krb +
              uint32_t(16 * ((lane % NCH) ^ (R % NCH)));
  }
  auto issue_chunk = [&](int kb0, int st) {
    const uint32_t base = uint32_t(kb0) * krb;
#pragma unroll
    for (int x = 0; x < H; ++x)
      copy16_to_lds(krs, kst_lds + uint32_t(st * STAGE + (wave * H + x) * 1024), base + coff[x]);
  };
  uint32_t aoff[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s)
    aoff[s] = uint32_t(l32 * ROWB + 16 * ((2 * s + hh) ^ (l32 % NCH)));
  // Keys outside [smin, Sk) count as -inf.
  auto clip = [&](int kb, f32x16_t& a) {
    if (kb >= smin && kb + 32 <= sk) return;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int key = kb + 16 * hh + e;
      if (key < smin || key >= sk) a[e] = -__builtin_inff();
    }
  };
  auto max16 = [](const f32x16_t& a) {
    const float t0 = max3_plain(a[0], a[1], a[2]), t1 = max3_plain(a[3], a[4], a[5]);
    const float t2 = max3_plain(a[6], a[7], a[8]), t3 = max3_plain(a[9], a[10], a[11]);
    return max3_plain(max3_plain(t0, t1, t2), max3_plain(t3, a[12], a[13]),
                      max_plain(a[14], a[15]));
  };

  // The three largest 16-key maxima of this lane, and the first two's first keys.
  float m1 = -__builtin_inff(), m2 = m1, m3 = m1;
  int at1 = 0, at2 = 0;
  const int kfirst = (smin > seg_lo ? smin : seg_lo) / kMxChunk * kMxChunk;
  const int nchunks = wg_end > kfirst ? (wg_end - kfirst + kMxChunk - 1) / kMxChunk : 0;
  if (nchunks > 0) issue_chunk(kfirst, 0);
  if (nchunks > 1) issue_chunk(kfirst + kMxChunk, 1);
  for (int c = 0, st = 0; c < nchunks; ++c, st = st == 2 ? 0 : st + 1) {
    const int kb0 = kfirst + c * kMxChunk;
    // Chunk c landed (chunk c+1's copies stay in flight); every wave is done
    // with chunk c-1, whose stage takes chunk c+2.
    if (c + 1 < nchunks)
      vm_lds_barrier_keep<H>();
    else
      vm_lds_barrier();
    if (c + 2 < nchunks) issue_chunk(kb0 + 2 * kMxChunk, st == 0 ? 2 : st - 1);
    if (kb0 >= wave_end) continue;  // this wave's rows need no more keys (uniform)
    // Operands are read kAhead MFMAs ahead of use; block 0's maximum is taken
    // between block 1's MFMAs.
    constexpr int kAhead = 3;
    f32x16_t acc[2];
    vec a[2 * NS];
    const unsigned char* stage = kst + st * STAGE;
    auto aload = [&](int i) {
      return __builtin_bit_cast(vec, *reinterpret_cast<const uint4*>(
                                         stage + i / NS * 32 * ROWB + aoff[i % NS]));
    };
    auto take = [&](int bb) {
      const int kb = kb0 + 32 * bb;
      clip(kb, acc[bb]);
      const float t = max16(acc[bb]);
      const int key = kb + 16 * hh;
      const bool g1 = t > m1, g2 = t > m2;
      m3 = max_plain(m3, g2 ? m2 : t);
      at2 = g1 ? at1 : (g2 ? key : at2);
      m2 = g1 ? m1 : max_plain(m2, t);
      at1 = g1 ? key : at1;
      m1 = max_plain(m1, t);
    };
#pragma unroll
    for (int i = 0; i < kAhead; ++i) a[i] = aload(i);
#pragma unroll
    for (int i = 0; i < 2 * NS; ++i) {
      __builtin_amdgcn_sched_barrier(0);
      if (i + kAhead < 2 * NS) a[i + kAhead] = aload(i + kAhead);
      if (i % NS == 0)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i / NS][e] = 0.f;
      acc[i / NS] = M::run(a[i], qreg[i % NS], acc[i / NS]);
      if (i == NS + 2) take(0);
    }
    __builtin_amdgcn_sched_barrier(0);
    take(1);
  }

  const float m = max_halves(m1), third = max_halves(m3);
  const bool some = m > -__builtin_inff();
  const bool tie = valid && (exact_wave || (some && third >= m - win));
  // Up to two candidate tiles per lane, four per row.
  const bool c1 = some && m1 >= m - win, c2 = some && m2 >= m - win;
  const int t1 = c1 ? at1 / bk : -1, t2 = c2 ? at2 / bk : -1;
  const int o1 = int(other_half(uint32_t(t1))), o2 = int(other_half(uint32_t(t2)));
  float ex = -__builtin_inff();
  if (__builtin_amdgcn_ballot_w64(tie) != 0) {
    // Rare: every piece within `win` of a tied row's maximum, scored exactly for
    // the wave's 32 rows on the fp64 matrix cores, whose chain of four-product
    // steps is the canonical sequential sum (select_exact.hip): operand lane l
    // holds row or key l % 16, feature 4 * step + l / 16, result register r of
    // lane l row l / 16 + 4r, key l % 16.  K operands come from global memory (no
    // barriers here), the MFMA scores' a step ahead of their use.
    auto operands = [&](int kb, uint4 (&w)[NS]) {
      const int kr = kb + kperm(l32);
      const T* krow = kh + int64_t(kr < sk ? kr : sk - 1) * sks + 8 * hh;
#pragma unroll
      for (int s = 0; s < NS; ++s) w[s] = *reinterpret_cast<const uint4*>(krow + 16 * s);
    };
    const int c16 = lane % 16, g16 = lane / 16;
    const T* qr[2];  // rows 16x + c16 (past the wave's last row: that one)
    float exm[2][4];  // exact maxima, of this lane's keys
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const int64_t r = 16 * x + c16 < rows_wave ? 16 * x + c16 : rows_wave - 1;
      qr[x] = qs + b * sqb + h * sqh + (jr_wave + r) * sqn;
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) exm[x][r4] = -__builtin_inff();
    }
    auto feature = [&](uint64_t four) {  // of four features, this lane's
      const uint16_t u = uint16_t(four >> (16 * g16));
      return double(to_f32(__builtin_bit_cast(T, u)));
    };
    uint4 next[NS];
    if (kfirst < wave_end) operands(kfirst, next);
    for (int kb = kfirst; kb < wave_end; kb += 32) {
      f32x16_t a;
#pragma unroll
      for (int e = 0; e < 16; ++e) a[e] = 0.f;
#pragma unroll
      for (int s = 0; s < NS; ++s) a = M::run(__builtin_bit_cast(vec, next[s]), qreg[s], a);
      if (kb + 32 < wave_end) operands(kb + 32, next);
      clip(kb, a);
      const uint64_t hits =
          __builtin_amdgcn_ballot_w64(tie && (exact_wave || max16(a) >= m - win));
#pragma unroll 1
      for (int p = 0; p < 2; ++p) {
        if (uint32_t(hits >> (32 * p)) == 0u) continue;  // no row needs this piece (uniform)
        const int key = kb + 16 * p + c16;
        const bool visited = key >= smin && key < sk;
        const T* kx = kh + int64_t(visited ? key : sk - 1) * sks;
        f64x4_t acc[2] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
#pragma unroll 2
        for (int d = 0; d < D; d += 8) {
          uint64_t kv[2], qv[2][2];
          __builtin_memcpy(kv, kx + d, 16);
          __builtin_memcpy(qv[0], qr[0] + d, 16);
          __builtin_memcpy(qv[1], qr[1] + d, 16);
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const double kd = feature(kv[i]);
#pragma unroll
            for (int x = 0; x < 2; ++x)
              acc[x] = __builtin_amdgcn_mfma_f64_16x16x4f64(feature(qv[x][i]), kd, acc[x], 0, 0, 0);
          }
        }
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int r4 = 0; r4 < 4; ++r4)
            exm[x][r4] = __builtin_fmaxf(exm[x][r4],
                                         visited ? float(acc[x][r4]) : -__builtin_inff());
      }
    }
    float mine = -__builtin_inff();  // of row l32
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        float v = exm[x][r4];
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) v = __builtin_fmaxf(v, __shfl_xor(v, o));
        const float w = __shfl(v, 16 * (l32 % 4));  // row 16x + 4 * r4 + l32 % 4
        if (l32 / 4 == 4 * x + r4) mine = w;
      }
    if (tie) ex = mine;
  }
  if (valid && hh == 0) {
    SegCarry cr;
    cr.m = m;
    cr.ex = ex;
    cr.n = 0;
    cr.pad = 0;
    const int cand[kCarryTiles] = {t1, t2, o1, o2};
#pragma unroll
    for (int i = 0; i < kCarryTiles; ++i) cr.tile[i] = -1;
    if (!tie)
#pragma unroll
      for (int i = 0; i < kCarryTiles; ++i)
        if (cand[i] >= 0) {
#pragma unroll
          for (int j = 0; j < kCarryTiles; ++j)
            if (j == cr.n) cr.tile[j] = cand[i];
          ++cr.n;
        }
    carry[(bh * nc + jr) * nseg + seg] = cr;
  }
}

hipError_t launch_select_max(int dtype, const void* qs, int64_t sqb, int64_t sqh, int64_t sqn,
                             const void* k, int64_t skb, int64_t skh, int64_t sks, int64_t B,
                             int64_t Hq, int64_t Hk, int64_t Sk, int64_t D, int64_t qps,
                             int64_t bk, int causal, int64_t bsq, const float* kmax,
                             const RowLayout& lay, int64_t segk, void* carry, hipStream_t stream) {
  const int64_t nrowsets = (lay.nc + kMxWaves * kMxRows - 1) / (kMxWaves * kMxRows);
  const int64_t nseg = (Sk + segk - 1) / segk;
  const int64_t nblocks = WorkOrder{nrowsets * nseg, B, Hq, Hk, causal == 0}.grid_items();
  auto go = [&](auto kernel, auto* tag) {
    using T = std::remove_pointer_t<decltype(tag)>;
    hipLaunchKernelGGL(kernel, dim3(unsigned(nblocks)), dim3(256), 0, stream,
                       static_cast<const T*>(qs), sqb, sqh, sqn, static_cast<const T*>(k), skb, skh,
                       sks, B, Hq, Hk, Sk, qps, int(bk), causal, bsq, kmax, lay, nrowsets,
                       int(segk), int(nseg), static_cast<SegCarry*>(carry));
    return hipGetLastError();
  };
  if (dtype == kBF16)
    return D == 128 ? go(select_max_kernel<bf16_t, 128>, static_cast<bf16_t*>(nullptr))
                    : go(select_max_kernel<bf16_t, 64>, static_cast<bf16_t*>(nullptr));
  return D == 128 ? go(select_max_kernel<f16_t, 128>, static_cast<f16_t*>(nullptr))
                  : go(select_max_kernel<f16_t, 64>, static_cast<f16_t*>(nullptr));
}

}  // namespace va
