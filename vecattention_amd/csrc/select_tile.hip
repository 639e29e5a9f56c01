// TilingSelect for tiles of 128 keys that are groups of their own
// (k_local_size 128 with group_k_block 1, the reference signature's defaults),
// on bf16/fp16 MFMA with certified decisions.
//
// Same rule, certification and output as select_wave.hip, which takes tiles up
// to its 64-key chunk.  With one tile per group a row's running maximum at a
// key is its tile's maximum, so tiles do not depend on each other: a wave
// scores a whole tile of its 32 pooled rows (4 blocks of 32 keys, 64
// accumulator registers), takes the row maxima and decides, with no state but
// the row's count between tiles.  The exact work of a tile (keys within the
// certification band of the threshold) covers the tile's own keys: those whose
// MFMA score can be the exact maximum, and the ambiguous ones.
//
// A work-group is 4 waves, 128 rows, sharing each tile's K rows in LDS (two
// stages, the next tile's copies in flight).  Bound by VALU work and latency
// at two work-groups per CU.  The 64-row kernel (select_mfma.hip), which these
// tiles took before, holds one work-group per CU behind ten barriers per 256
// keys: a prefill of 16411 keys of 28 heads spent 182 us in its two selections,
// here 61; 436 -> 310 us as a whole (40000 keys of 32 heads 1381 -> 968).
#include <type_traits>

#include "key_norm.h"
#include "lanes.h"
#include "mfma.h"
#include "select_cert.h"

namespace va {

bool select_lists_32bit(int64_t dense_stride);

constexpr int kTRows = 32, kTWaves = 4, kTKeys = 128;

template <typename T, int D>
__global__ __launch_bounds__(256, 2) void select_tile_kernel(
    const T* __restrict__ qs, int64_t sqb, int64_t sqh, int64_t sqn, const T* __restrict__ k,
    int64_t skb, int64_t skh, int64_t sks, int64_t B, int64_t Hq, int64_t Hk, int64_t Sk,
    int64_t qps, int causal, int64_t bsq, float gap_scalar, const float* __restrict__ gaps,
    const float* __restrict__ kmax, RowLayout lay, int32_t* __restrict__ counts,
    int32_t* __restrict__ indices, int64_t nrowsets, int segk, int nseg) {
  using M = Mfma<T>;
  using vec = typename M::vec;
  constexpr int NS = D / 16, ROWB = 2 * D, NCH = D / 8;
  constexpr int NBK = kTKeys / 32;               // blocks of 32 keys
  constexpr int STAGE = kTKeys * ROWB;           // bytes of one tile of K
  constexpr int RPC = 1024 / ROWB;               // rows per 1 KB copy
  constexpr int H = STAGE / 1024 / kTWaves;      // copies per wave and tile

  __shared__ __attribute__((aligned(1024))) unsigned char kst[2 * STAGE];
  __shared__ uint32_t pieces[kTWaves][kTRows][2 * NBK];  // rare path: ambiguous | candidates << 16
  __shared__ int32_t jkey[kTWaves][kTKeys];              // rare path: key offsets of the jobs
  __shared__ uint32_t taken[kTWaves][NBK];               // rare path: resolved selections

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
  const int64_t jr_wave = int64_t(rs) * (kTWaves * kTRows) + kTRows * wave;
  const int64_t jr = jr_wave + l32;
  const bool valid = jr < nc;
  const float gap = gaps ? gaps[bh] : gap_scalar;
  const int sk = int(Sk);  // < 2^24 (host check)
  const int smin = int(lay.smin());

  // Causal tile limit of a row and the keys a row set needs (select_wave.hip).
  auto row_lim = [&](int64_t row) -> int {
    if (!causal) return 0x7fffffff;
    const int64_t J = J0 + row, r = row % bsq;
    const int64_t lim = (r == 0) ? (J - 1) * qps + 1 : J * qps;
    return int(lim < 0 ? 0 : (lim > 0x7fffffff ? 0x7fffffff : lim));
  };
  auto range_end = [&](int64_t last_row) -> int {
    if (!causal) return sk;
    const int64_t e = (int64_t(row_lim(last_row)) + kTKeys - 1) / kTKeys * kTKeys;
    return int(e < Sk ? e : Sk);
  };
  const int64_t rows_wave = nc - jr_wave < kTRows ? nc - jr_wave : kTRows;
  const int64_t left = nc - int64_t(rs) * (kTWaves * kTRows);
  const int64_t rows_wg = left < kTWaves * kTRows ? left : kTWaves * kTRows;
  const int seg_lo = seg * segk;
  const int seg_hi = nseg > 1 ? seg_lo + segk : 0x7fffffff;
  int wave_end = rows_wave > 0 ? range_end(jr_wave + rows_wave - 1) : 0;
  int wg_end = range_end(int64_t(rs) * (kTWaves * kTRows) + rows_wg - 1);
  if (wave_end > seg_hi) wave_end = seg_hi;
  if (wg_end > seg_hi) wg_end = seg_hi;
  const int lim = valid ? row_lim(jr) : 0;

  // ---- pooled rows (B operand), their norms and bounds ---------------------
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
  const Bounds bounds = score_bounds<D>(ss, kn, gap);
  const float band = bounds.band, win = bounds.win;
  const bool all_exact = valid && !bounds.certified;  // as select_wave.hip

  // ---- output of this lane's row, as select_wave.hip -----------------------
  int64_t ostart = 0, ocap = 0;
  if (valid) lay.segment_slots(bh, jr, seg, nseg, seg_lo, ostart, ocap);
  const int cap = int(ocap);
  const int64_t wrow0 = rows_wave > 0 ? lay.row_start(bh, jr_wave) : 0;
  const int64_t wrow_end = rows_wave > 0 ? lay.row_start(bh, jr_wave + rows_wave) : 0;
  const __amdgpu_buffer_rsrc_t ors = make_rsrc(
      indices ? indices + wrow0 : indices, uint32_t(indices ? (wrow_end - wrow0) * 4 : 0));
  const uint32_t ofirst = valid ? uint32_t(ostart - wrow0) * 4u : 0xfffffff0u;
  const uint32_t olast = valid && cap > 0 ? ofirst + uint32_t(cap - 1) * 4u : 0xfffffff0u;
  int rowcnt = 0;

  // ---- K copies and operand reads (layout of select_wave.hip: LDS row R of
  // block R/32 holds key 32*(R/32) + kperm(R % 32), chunks XOR-swizzled) ------
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
  auto issue_tile = [&](int kb0, int st) {
    const uint32_t base = uint32_t(kb0) * krb;
#pragma unroll
    for (int x = 0; x < H; ++x)
      copy16_to_lds(krs, kst_lds + uint32_t(st * STAGE + (wave * H + x) * 1024), base + coff[x]);
  };
  uint32_t aoff[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s)
    aoff[s] = uint32_t(l32 * ROWB + 16 * ((2 * s + hh) ^ (l32 % NCH)));

  // Exact decisions of the rows in `need`, one row at a time: the exact scores
  // of the tile's candidates (keys whose MFMA score can be the exact tile
  // maximum) and ambiguous keys, one per lane; the exact maximum; the
  // decisions.  Resolved selections are added to the row's `bits`.
  auto resolve = [&](uint64_t need, int kb0, uint32_t (&bits)[NBK]) {
    while (need) {
      const int r = __builtin_ctzll(need);
      need &= need - 1;
      const T* qr = qs + b * sqb + h * sqh + (jr_wave + r) * sqn;
      // job list: lane L looks at keys L and 64 + L of the tile
      int njobs = 0;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const uint32_t w = pieces[wave][r][4 * p + lane / 16] >> (lane % 16);
        const bool job = (w & 0x10001u) != 0u;
        const uint64_t m = __builtin_amdgcn_ballot_w64(job);
        const int at = njobs + int(__builtin_amdgcn_mbcnt_hi(
                                   uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0)));
        if (job)
          jkey[wave][at] = (64 * p + lane) | int((w & 1u) << 8) | int((w >> 16 & 1u) << 9);
        njobs += __builtin_popcountll(m);
      }
      if (lane < NBK) taken[wave][lane] = 0u;
      float ex[2], best = -__builtin_inff();
      int jk[2];
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int j = 64 * p + lane;
        jk[p] = j < njobs ? jkey[wave][j] : 0;
        ex[p] = -__builtin_inff();
        const int key = kb0 + (jk[p] & 127);
        if (j < njobs && key < sk) {
          const T* kr = kh + int64_t(key) * sks;
          double acc = 0.0;
#pragma unroll 4
          for (int c = 0; c < D / 8; ++c) {
            const uint4 qv = *reinterpret_cast<const uint4*>(qr + 8 * c);
            const uint4 kv = *reinterpret_cast<const uint4*>(kr + 8 * c);
            const T* q8 = reinterpret_cast<const T*>(&qv);
            const T* k8 = reinterpret_cast<const T*>(&kv);
#pragma unroll
            for (int e = 0; e < 8; ++e)
              acc = __builtin_fma(double(to_f32(q8[e])), double(to_f32(k8[e])), acc);
          }
          ex[p] = float(acc);
        }
        if (jk[p] & 512) best = __builtin_fmaxf(best, ex[p]);
      }
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) best = __builtin_fmaxf(best, __shfl_xor(best, o));
#pragma unroll
      for (int p = 0; p < 2; ++p)
        if ((jk[p] & 256) && (ex[p] + gap) >= best) {
          const int kk = jk[p] & 127;
          atomicOr(&taken[wave][kk / 32], 1u << (kk % 32));
        }
      if (l32 == r) {
#pragma unroll
        for (int bb = 0; bb < NBK; ++bb) bits[bb] |= (taken[wave][bb] >> (16 * hh)) & 0xffffu;
      }
    }
  };

  const int kfirst = smin > seg_lo ? smin : seg_lo;  // a tile start
  const int ntiles = wg_end > kfirst ? (wg_end - kfirst + kTKeys - 1) / kTKeys : 0;
  if (ntiles > 0) issue_tile(kfirst, 0);
  for (int t = 0; t < ntiles; ++t) {
    const int kb0 = kfirst + t * kTKeys, st = t & 1;
    vm_lds_barrier();  // tile t landed; every wave is done with tile t-1
    if (t + 1 < ntiles) issue_tile(kb0 + kTKeys, st ^ 1);
    if (kb0 >= wave_end) continue;  // this wave's rows need no more keys (uniform)
    f32x16_t acc[NBK];
    const unsigned char* stage = kst + st * STAGE;
#pragma unroll
    for (int bb = 0; bb < NBK; ++bb) {
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[bb][e] = 0.f;
#pragma unroll
      for (int s = 0; s < NS; ++s)
        acc[bb] = M::run(__builtin_bit_cast(vec, *reinterpret_cast<const uint4*>(
                                                     stage + bb * 32 * ROWB + aoff[s])),
                         qreg[s], acc[bb]);
    }
    if (kb0 + kTKeys > sk) {  // keys past the end are not visited
#pragma unroll
      for (int bb = 0; bb < NBK; ++bb)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (kb0 + 32 * bb + 16 * hh + e >= sk) acc[bb][e] = -__builtin_inff();
    }
    float m = -__builtin_inff();
#pragma unroll
    for (int bb = 0; bb < NBK; ++bb)
#pragma unroll
      for (int e = 0; e < 16; e += 2) m = max3_plain(m, acc[bb][e], acc[bb][e + 1]);
    m = max_halves(m);
    // Decisions from signs of x = hi - s^, as select_wave.hip: selected outright
    // when negative, ambiguous in [0, 2*band].
    const bool ok = valid && kb0 < lim && kb0 < sk;
    const float hi = ok ? (m - gap) + band : __builtin_inff();
    uint32_t bits[NBK], xmin = 0xffffffffu;
#pragma unroll
    for (int bb = 0; bb < NBK; ++bb) {
      uint32_t bt = 0;
#pragma unroll
      for (int e = 15; e >= 0; --e) {
        const uint32_t x = __builtin_bit_cast(uint32_t, hi - acc[bb][e]);
        bt = __builtin_amdgcn_alignbit(bt, x, 31u);  // (bt << 1) | sign(x)
        xmin = x < xmin ? x : xmin;
      }
      bits[bb] = bt;
    }
    const uint32_t band2 = all_exact ? 0xffffffffu : __builtin_bit_cast(uint32_t, 2.f * band);
    const bool amb = xmin <= band2;
    if (__builtin_amdgcn_ballot_w64(amb) != 0) {  // rare path
      const float cut = m - win;
#pragma unroll
      for (int bb = 0; bb < NBK; ++bb) {
        uint32_t w = 0;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          w |= uint32_t(__builtin_bit_cast(uint32_t, hi - acc[bb][e]) <= band2) << e;
          w |= uint32_t(acc[bb][e] >= cut) << (16 + e);
        }
        if (all_exact) {  // every key before the end of the keys
          const int left = sk - (kb0 + 32 * bb + 16 * hh);
          w = left <= 0 ? 0u : (left < 16 ? (1u << left) - 1u : 0xffffu) * 0x10001u;
        }
        if (!ok) w = 0;
        if (!valid || all_exact) bits[bb] = 0;
        pieces[wave][l32][2 * bb + hh] = w;
      }
      const bool row_amb = (uint32_t(amb) | other_half(uint32_t(amb))) != 0u;
      resolve(__builtin_amdgcn_ballot_w64(hh == 0 && ok && row_amb), kb0, bits);
    }
#pragma unroll
    for (int bb = 0; bb < NBK; ++bb) {
      uint32_t bt = bits[bb];
      const int cnt = __builtin_popcount(bt);
      const int ocnt = int(other_half(uint32_t(cnt)));
      if (indices) {
        uint32_t off = ofirst + uint32_t(rowcnt + (hh ? ocnt : 0)) * 4u;
        const int key0 = kb0 + 32 * bb + 16 * hh;
        while (bt) {
          const int e = __builtin_ctz(bt);
          bt &= bt - 1;
          __builtin_amdgcn_raw_buffer_store_b32(key0 + e, ors, off < olast ? off : olast, 0, 0);
          off += 4u;
        }
      }
      rowcnt += cnt + ocnt;
    }
  }
  if (valid && hh == 0 && counts) counts[(bh * nc + jr) * nseg + seg] = rowcnt < cap ? rowcnt : cap;
}

// Tiles of 128 keys, one per group, keys the copies' 32-bit offsets reach, and
// lists the stores' reach.
bool select_tile_ok(int dtype, int64_t D, int64_t bk, int64_t group, int64_t Sk, int64_t sks,
                    int64_t dense_stride) {
  return (dtype == kBF16 || dtype == kF16) && (D == 64 || D == 128) && bk == kTKeys &&
         group == 1 && sks >= D && Sk < (int64_t(1) << 24) &&
         (Sk + 2 * kTKeys) * sks * 2 < (int64_t(1) << 31) && select_lists_32bit(dense_stride);
}

hipError_t launch_select_tile(int dtype, const void* qs, int64_t sqb, int64_t sqh, int64_t sqn,
                              const void* k, int64_t skb, int64_t skh, int64_t sks, int64_t B,
                              int64_t Hq, int64_t Hk, int64_t Sk, int64_t D, int64_t qps,
                              int causal, int64_t bsq, float gap, const float* gaps,
                              const float* kmax, const RowLayout& lay, int32_t* counts,
                              int32_t* indices, int64_t segk, hipStream_t stream) {
  const int64_t nrowsets = (lay.nc + kTWaves * kTRows - 1) / (kTWaves * kTRows);
  const int64_t nseg = segk > 0 ? (Sk + segk - 1) / segk : 1;
  const int64_t nblocks = WorkOrder{nrowsets * nseg, B, Hq, Hk, causal == 0}.grid_items();
  auto go = [&](auto kernel, auto* tag) {
    using T = std::remove_pointer_t<decltype(tag)>;
    hipLaunchKernelGGL(kernel, dim3(unsigned(nblocks)), dim3(256), 0, stream,
                       static_cast<const T*>(qs), sqb, sqh, sqn, static_cast<const T*>(k), skb, skh,
                       sks, B, Hq, Hk, Sk, qps, causal, bsq, gap, gaps, kmax, lay, counts, indices,
                       nrowsets, int(segk > 0 ? segk : 0), int(nseg));
    return hipGetLastError();
  };
  if (dtype == kBF16)
    return D == 128 ? go(select_tile_kernel<bf16_t, 128>, static_cast<bf16_t*>(nullptr))
                    : go(select_tile_kernel<bf16_t, 64>, static_cast<bf16_t*>(nullptr));
  return D == 128 ? go(select_tile_kernel<f16_t, 128>, static_cast<f16_t*>(nullptr))
                  : go(select_tile_kernel<f16_t, 64>, static_cast<f16_t*>(nullptr));
}

}  // namespace va
