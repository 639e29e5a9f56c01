// Dense attention (every key, optionally causal) on CDNA4 bf16/fp16 MFMA, and
// its row-statistics form.
//
// The Full_prefill path (spattn/src/Fullprefill.py:4-16) and the dense softmax
// of the tuner's recall (spattn/threshold/model_tuner.py:193-220).  A
// work-group owns 128 query rows of one q head, each of its 4 waves 32 of
// them; GQA is native.
//
// The sparse kernel's dense form (attn_mfma.hip) gathers a K and a V row per
// 64 query rows, at which the copies into LDS take as long as the MFMAs
// (64 B per clock against 16 MFMAs of 32 clocks per wave and tile).  Here keys
// are consecutive, so a tile's copies need one add per address and no staged
// ids, and serve 128 rows: half of the copies per FLOP, half of the barriers,
// and no merge of key halves at the end.
//
// Precision.  A row has one running maximum over all 64 keys of a tile, where
// the 64-row form keeps one per key half, so one key of the first tile instead
// of two has a probability of exactly 1 and the rounding of the others to 16
// bits weighs 0.9% more (relative error against 64 bits of 16384 causal bf16
// rows 2.110e-3 there, 2.126e-3 with one maximum and nothing else).  The first
// tile's probabilities therefore enter P V and the row sum as two 16-bit parts,
// value and remainder, which is where rows of few keys have their error:
// 1.979e-3 (non-causal 3000 keys 2.324e-3 -> 2.304e-3), for one more pass of
// MFMAs over one tile: 0.0% of the time at 16384 causal keys, 1% at 3300.
//
// Bound by the power the matrix cores draw: 16384 causal keys of 28 heads
// take 1641 us (1173 TFLOP/s, 84% of a bf16 16384^3 library GEMM on the same
// card; 1893 us in the 64-row form), and 1130 us (1.70 PFLOP/s) on all-zero
// inputs.  Exponentials placed between the MFMAs of the same wave and other
// issue priorities measured within 1%.  The statistics form (no V) is bound
// by its VALU work, so five work-groups per CU on two K tiles each: the dense
// pass of 32760 keys of 12 heads takes 3.3 ms, 3.8 in the 64-row form.
#include "attn_common.h"
#include "lanes.h"
#include "mfma.h"

namespace va {

constexpr int kDenseRows = 128;  // query rows per work-group

template <int D>
struct DenseShape {
  static constexpr int kRowBytes = 2 * D;
  static constexpr int kTileBytes = kTileKeys * kRowBytes;    // one K (or V) tile
  static constexpr int kChunks = D / 8;                       // 16-byte chunks per row
  static constexpr int kRowsPerCopy = 1024 / kRowBytes;       // rows per 1 KB copy
  static constexpr int kCopies = kTileBytes / 1024 / 4;       // per wave and tile
};

// stats: row i of head bh gets stats[(bh * Sq + i) * 2 + {0, 1}] = (m, l), l =
// sum over its keys of 2^(s * scale_log2 - m) in fp32.  Row i sees keys up to
// qoff + i when causal.
template <typename T, int D, bool kStats>
__global__ __launch_bounds__(256, kStats ? (D == 128 ? 5 : 6) : (D == 128 ? 3 : 4)) void attn_dense_kernel(
    const T* __restrict__ q, int64_t sqb, int64_t sqh, int64_t sqs, const T* __restrict__ k,
    int64_t skb, int64_t skh, int64_t sks, const T* __restrict__ v, int64_t svb, int64_t svh,
    int64_t svs, T* __restrict__ out, int64_t sob, int64_t soh, int64_t sos, int64_t B,
    int64_t Hq, int64_t Hk, int64_t Sq, int64_t Sk, int causal, float scale_log2, int64_t nblk,
    int64_t qoff, float* __restrict__ stats) {
  using S = DenseShape<D>;
  using M = Mfma<T>;
  using vec = typename M::vec;
  constexpr int H = S::kCopies, NCH = S::kChunks, RPC = S::kRowsPerCopy;
  constexpr uint32_t TB = uint32_t(S::kTileBytes);
  constexpr int NQK = D / 16;   // QK MFMAs per 32 keys
  constexpr int NB = D / 32;    // output blocks of 32 features
  constexpr int NPV = 4 * NB;   // PV MFMAs per tile (16 keys each)
  __shared__ __attribute__((aligned(1024))) unsigned char smem[(kStats ? 2 : 3) * S::kTileBytes];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;
  const int l32 = lane % 32, hh = lane / 32;

  const WorkOrder wo{nblk, B, Hq, Hk, causal == 0};
  int jb, bh;
  if (!wo.map_item32(blockIdx.x, jb, bh)) return;  // idle block (uniform)
  const uint32_t hq32 = uint32_t(Hq);
  const int64_t b = uint32_t(bh) / hq32, h = uint32_t(bh) % hq32;
  const int64_t hk = uint32_t(h) / (hq32 / uint32_t(Hk));

  // ---- Q^T operand: lane holds row 32 wave + l32, features [16s + 8hh, +8).
  // Rows past Sq load row Sq - 1; their results are never written.
  const int row0 = jb * kDenseRows + 32 * wave;  // first row of this wave
  const int row = row0 + l32;
  vec qreg[NQK];
  {
    const T* qp = q + b * sqb + h * sqh + int64_t(row < Sq ? row : int(Sq) - 1) * sqs;
#pragma unroll
    for (int s = 0; s < NQK; ++s)
      qreg[s] = __builtin_bit_cast(vec, *reinterpret_cast<const uint4*>(qp + 16 * s + 8 * hh));
  }

  // Keys the work-group and this wave need: [0, kend), [0, wend) (every wave
  // copies its share of every tile; one past its rows' last key only that).
  const int sk = int(Sk);
  auto keys_of = [&](int last_row) {  // keys up to the last one that row sees
    if (!causal) return sk;
    const int e = int(qoff) + (last_row < int(Sq) ? last_row : int(Sq) - 1) + 1;
    return e < sk ? e : sk;
  };
  const int kend = keys_of(jb * kDenseRows + kDenseRows - 1);
  const int wtiles =
      __builtin_amdgcn_readfirstlane((keys_of(row0 + 31) + kTileKeys - 1) / kTileKeys);
  const int ntiles = __builtin_amdgcn_readfirstlane((kend + kTileKeys - 1) / kTileKeys);
  // Tiles from m_tile on hold keys that some row of this wave does not see:
  // the causal diagonal and the end of the keys.
  const int clear = causal ? (int(qoff) + row0 + 1 < sk ? int(qoff) + row0 + 1 : sk) : sk;
  const int m_tile = __builtin_amdgcn_readfirstlane(clear / kTileKeys);
  const int last_key = causal ? (int(qoff) + row < sk - 1 ? int(qoff) + row : sk - 1) : sk - 1;

  // ---- copies: copy x of this wave fills tile rows [(wave*H + x)*RPC, +RPC);
  // this lane fetches logical chunk p ^ chunk_swizzle(R) of its row R.
  const __amdgpu_buffer_rsrc_t krs =
      make_rsrc_rows(k + b * skb + hk * skh, uint32_t(sks * 2), uint32_t(Sk));
  const __amdgpu_buffer_rsrc_t vrs =
      kStats ? krs : make_rsrc_rows(v + b * svb + hk * svh, uint32_t(svs * 2), uint32_t(Sk));
  const uint32_t crow = uint32_t(wave * H * RPC + lane / NCH);  // row of copy 0
  // Chunk offset of copy 0; copy x's is c0 ^ x * kXorStep (the swizzle of row
  // crow + x * RPC: x is bits 2, 3 of the row's place in its bank period at D =
  // 128, bit 2 at D = 64).
  const uint32_t c0 = uint32_t(16 * ((lane % NCH) ^ chunk_swizzle<D>(int(crow))));
  constexpr uint32_t kXorStep = D == 128 ? 16 : 32;
  static_assert((D == 128 && H == 4) || (D == 64 && H == 2), "copy geometry");
  const uint32_t lds_copy_base =
      uint32_t(__builtin_amdgcn_readfirstlane(int(lds_addr(smem) + uint32_t(wave * H * 1024))));
  // Keys past Sk (the last tile's, and whole tiles past the end) read zeros.
  // The row and chunk pass through an empty asm: addresses are formed at each
  // copy (two VALU instructions) instead of being kept in registers that the
  // three work-groups per CU do not leave.
  auto copy = [&](const __amdgpu_buffer_rsrc_t& rs, auto base_tag, auto x_tag, int t) {
    constexpr int x = decltype(x_tag)::value;
    uint32_t r0 = crow, ch = c0;
    asm volatile("" : "+v"(r0), "+v"(ch));
    const uint32_t key = r0 + uint32_t(t * kTileKeys + x * RPC);
    copy16_row_to_lds_at<decltype(base_tag)::value + x * 1024u>(
        rs, lds_copy_base, uint64_t(key) | (uint64_t(ch ^ (x * kXorStep)) << 32));
  };

  // ---- LDS read offsets (see attn_mfma.hip): K row l32 (+ 32 for the second
  // half of the tile), chunk 2s + hh = k0 ^ 32s; V^T rows 8r + 4hh + j (+ 16
  // per MFMA step), features 32i + ...: v0r ^ 64i.
  const uint32_t k0 = uint32_t(l32 * S::kRowBytes + 16 * (hh ^ chunk_swizzle<D>(l32)));
  uint32_t v0[2];
  {
    const int j = (lane % 16) / 4, g2 = 2 * ((lane / 16) % 2) + (lane % 4) / 2;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int R = 8 * r + 4 * hh + j;
      v0[r] = uint32_t(R * S::kRowBytes + 16 * (g2 ^ chunk_swizzle<D>(R)) + 8 * (lane % 2));
    }
  }

  f32x16_t o[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[i][e] = 0.f;
  float mc = -__builtin_inff(), mneg = 0.f, thr = -__builtin_inff(), lsum = 0.f;
  const float inv_scale = 1.f / scale_log2;  // the host passes scale_log2 > 0
#pragma unroll
  for (int s = 0; s < NQK; ++s) asm volatile("" ::"v"(qreg[s]));  // Q landed before the copies

  // Move the running maximum when some row's tile maximum exceeds it by more
  // than the slack (rare, as attn_mfma.hip): rescale O and the row sums.
  auto rescale = [&](float tmax) {
    if (__builtin_amdgcn_ballot_w64(tmax > thr)) {
      tmax = max_halves(tmax);
      const float mnew = __builtin_fmaxf(mc, tmax * scale_log2);
      const float alpha = (mnew == mc) ? 1.f : __builtin_amdgcn_exp2f(mc - mnew);
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[i][e] *= alpha;  // dead code under kStats
      lsum *= alpha;
      mc = mnew;
      const bool none = mnew == -__builtin_inff();
      mneg = none ? 0.f : -mnew;
      thr = none ? -__builtin_inff() : (mnew + kRescaleSlack) * inv_scale;
    }
  };
  auto prob = [&](float s) { return __builtin_amdgcn_exp2f(__builtin_fmaf(s, scale_log2, mneg)); };
  auto kread = [&](const unsigned char* kb, uint32_t kx, int i) {  // operand of QK MFMA i
    return __builtin_bit_cast(vec, *reinterpret_cast<const uint4*>(
                                       kb + (kx ^ uint32_t(32 * (i % NQK))) +
                                       i / NQK * 32 * S::kRowBytes));
  };
  // S^T of a tile's two 32-key halves; the copies go out between the MFMAs.
  constexpr int kAhead = 2;
  auto qk = [&](const unsigned char* kb, f32x16_t (&sc)[2], auto&& copies) {
    uint32_t kx = k0;
    asm volatile("" : "+v"(kx));  // the offsets are rebuilt, not kept
    vec a[2 * NQK];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) a[i] = kread(kb, kx, i);
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int e = 0; e < 16; ++e) sc[hf][e] = 0.f;
    __builtin_amdgcn_s_setprio(2);
#pragma unroll
    for (int i = 0; i < 2 * NQK; ++i) {
      __builtin_amdgcn_sched_barrier(0);
      if (i + kAhead < 2 * NQK) a[i + kAhead] = kread(kb, kx, i + kAhead);
      sc[i / NQK] = M::run(a[i], qreg[i % NQK], sc[i / NQK]);
      static_for<H>([&](auto c) {
        if (c * 2 * NQK / H == i) copies(c);
      });
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
  };
  // Scores of keys this lane's row does not see become -inf (tiles from
  // m_tile on).  Slot of sc[hf][e]: 32hf + 8(e/4) + 4hh + e%4.
  auto mask = [&](int t, f32x16_t (&sc)[2]) {
    if (t < m_tile) return;
    const int lim = last_key - t * kTileKeys - 4 * hh;
#pragma unroll
    for (int e = 0; e < 32; ++e)
      sc[e / 16][e % 16] = 8 * (e / 4) + (e % 4) <= lim ? sc[e / 16][e % 16] : -__builtin_inff();
  };
  auto tile_max = [&](const f32x16_t (&sc)[2]) {
    float t0 = max3_plain(sc[0][0], sc[0][1], sc[0][2]), t1 = sc[0][3];
#pragma unroll
    for (int e = 4; e < 32; e += 4) {
      t0 = max3_plain(t0, sc[e / 16][e % 16], sc[e / 16][e % 16 + 1]);
      t1 = max3_plain(t1, sc[e / 16][e % 16 + 2], sc[e / 16][e % 16 + 3]);
    }
    return max_plain(t0, t1);
  };

  if constexpr (kStats) {
    // Two K tiles in turn: step t waits for K(t) and copies K(t+1) into the
    // slot of K(t-1); five work-groups per CU hide the wait.
    static_for<H>([&](auto x) { copy(krs, lds_off<0>{}, x, 0); });
    auto step = [&](int t, auto r_tag) {
      constexpr int r = decltype(r_tag)::value;
      vm_lds_barrier();
      auto copies = [&](auto c) { copy(krs, lds_off<(r ^ 1) * TB>{}, c, t + 1); };
      if (t >= wtiles) {  // this wave's rows see no more keys (uniform)
        static_for<H>(copies);
        return;
      }
      f32x16_t sc[2];
      qk(smem + r * TB, sc, copies);
      mask(t, sc);
      rescale(tile_max(sc));
      float ps[4];  // a tree of sums over the tile's keys
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        float pr[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) pr[e] = prob(sc[f / 2][8 * (f % 2) + e]);
        ps[f] = ((pr[0] + pr[1]) + (pr[2] + pr[3])) + ((pr[4] + pr[5]) + (pr[6] + pr[7]));
      }
      lsum += (ps[0] + ps[1]) + (ps[2] + ps[3]);
    };
    for (int t = 0; t < ntiles; t += 2) {
      step(t, std::integral_constant<int, 0>{});
      if (t + 1 < ntiles) step(t + 1, std::integral_constant<int, 1>{});
    }
    vm_lds_barrier();  // the last copies have landed
    const float l = sum_halves(lsum);
    if (hh == 0 && row < Sq)
      *reinterpret_cast<float2*>(stats + (int64_t(bh) * Sq + row) * 2) = make_float2(mc, l);
    return;
  } else {
    // Ring of three tile slots holding the operand stream K(0), V(0), K(1),
    // ...: as the sparse kernel's ring form.
    static_for<H>([&](auto x) { copy(krs, lds_off<0>{}, x, 0); });
    static_for<H>([&](auto x) { copy(vrs, lds_off<TB>{}, x, 0); });
    auto vread = [&](const unsigned char* vb, uint32_t va, uint32_t vb1, int f) {
      const int sub = f / NB, i = f % NB;  // 16 keys of step sub, features [32i, +32)
      const unsigned char* p0 = vb + (va ^ uint32_t(64 * i)) + sub * 16 * S::kRowBytes;
      const unsigned char* p1 = vb + (vb1 ^ uint32_t(64 * i)) + sub * 16 * S::kRowBytes;
      const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) s16x4_t*)(p0));
      const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) s16x4_t*)(p1));
      const s16x4_t both[2] = {lo, hi};
      return __builtin_bit_cast(vec, both);
    };
    // first: the step of tile 0, whose probabilities go in as two 16-bit parts.
    auto step = [&](int t, auto r_tag, auto first_tag) {
      constexpr int r = decltype(r_tag)::value;
      constexpr bool first = decltype(first_tag)::value;
      constexpr uint32_t k_this = uint32_t((2 * r) % 3) * TB;
      constexpr uint32_t v_this = uint32_t((2 * r + 1) % 3) * TB;
      constexpr uint32_t k_next = uint32_t((2 * r + 2) % 3) * TB;
      constexpr uint32_t v_next = k_this;
      auto kcopies = [&](auto c) { copy(krs, lds_off<k_next>{}, c, t + 1); };
      auto vcopies = [&](auto c) { copy(vrs, lds_off<v_next>{}, c, t + 1); };
      // ---- K(t) landed; every wave is done with V(t-1)
      vm_lds_barrier_keep<H>();
      if (t >= wtiles) {  // this wave's rows see no more keys (uniform)
        static_for<H>(kcopies);
        vm_lds_barrier_keep<H>();
        static_for<H>(vcopies);
        return;
      }
      f32x16_t sc[2];
      qk(smem + k_this, sc, kcopies);
      mask(t, sc);
      rescale(tile_max(sc));
      vec bfrag[4], brest[first ? 4 : 1];
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        __builtin_amdgcn_sched_barrier(0);  // bounds the live probabilities
        float pr[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) pr[e] = prob(sc[f / 2][8 * (f % 2) + e]);
        bfrag[f] = M::pack(pr);
        if constexpr (first) {
#pragma unroll
          for (int e = 0; e < 8; ++e) pr[e] -= float(bfrag[f][e]);
          brest[f] = M::pack(pr);
        }
      }
      // ---- V(t) landed; every wave is done with K(t)
      vm_lds_barrier_keep<H>();
      uint32_t va = v0[0], vb1 = v0[1];
      asm volatile("" : "+v"(va), "+v"(vb1));
      const unsigned char* vb = smem + v_this;
      constexpr int kVAhead = 2;
      vec vf[NPV];
#pragma unroll
      for (int f = 0; f < kVAhead; ++f) vf[f] = vread(vb, va, vb1, f);
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int f = 0; f < NPV; ++f) {
        __builtin_amdgcn_sched_barrier(0);
        if (f + kVAhead < NPV) vf[f + kVAhead] = vread(vb, va, vb1, f + kVAhead);
        o[f % NB] = M::run(vf[f], bfrag[f / NB], o[f % NB]);
        if constexpr (first) o[f % NB] = M::run(vf[f], brest[f / NB], o[f % NB]);
        static_for<H>([&](auto c) {
          if (c * NPV / H == f) vcopies(c);
        });
#pragma unroll
        for (int j = f * 16 / NPV; j < (f + 1) * 16 / NPV; ++j)
          lsum = M::add_pair(bfrag[j / 4], j % 4, lsum);
        if constexpr (first)
#pragma unroll
          for (int j = f * 16 / NPV; j < (f + 1) * 16 / NPV; ++j)
            lsum = M::add_pair(brest[j / 4], j % 4, lsum);
      }
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_setprio(0);
    };
    if (ntiles > 0) step(0, std::integral_constant<int, 0>{}, std::true_type{});
    for (int t = 1; t < ntiles; t += 3) {
      step(t, std::integral_constant<int, 1>{}, std::false_type{});
      if (t + 1 < ntiles) step(t + 1, std::integral_constant<int, 2>{}, std::false_type{});
      if (t + 2 < ntiles) step(t + 2, std::integral_constant<int, 0>{}, std::false_type{});
    }
    vm_lds_barrier();  // the last copies have landed
    const float l = sum_halves(lsum);
    const float inv = l > 0.f ? 1.f / l : 0.f;
    if (row >= Sq) return;
    T* orow = out + b * sob + h * soh + int64_t(row) * sos;
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const T e0 = Round<T>::store(o[i][4 * g + 0] * inv);
        const T e1 = Round<T>::store(o[i][4 * g + 1] * inv);
        const T e2 = Round<T>::store(o[i][4 * g + 2] * inv);
        const T e3 = Round<T>::store(o[i][4 * g + 3] * inv);
        uint2 w;
        w.x = uint32_t(e0.bits) | (uint32_t(e1.bits) << 16);
        w.y = uint32_t(e2.bits) | (uint32_t(e3.bits) << 16);
        *reinterpret_cast<uint2*>(orow + 32 * i + 8 * g + 4 * hh) = w;
      }
  }
}

template <typename T, int D>
static hipError_t launch_dense_td(const void* q, const int64_t* sq, const void* k,
                                  const int64_t* sk, const void* v, const int64_t* sv, void* out,
                                  const int64_t* so, int64_t B, int64_t Hq, int64_t Hk, int64_t Sq,
                                  int64_t Sk, int causal, float scale_log2, int64_t qoff,
                                  float* stats, hipStream_t stream) {
  static const int64_t zero[3] = {0, 0, 0};
  if (stats) sv = so = zero;  // no V, no output
  const int64_t nblk = (Sq + kDenseRows - 1) / kDenseRows;
  const int64_t grid = WorkOrder{nblk, B, Hq, Hk, causal == 0}.grid_items();
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(unsigned(grid)), dim3(256), 0, stream,
                       static_cast<const T*>(q), sq[0], sq[1], sq[2], static_cast<const T*>(k),
                       sk[0], sk[1], sk[2], static_cast<const T*>(v), sv[0], sv[1], sv[2],
                       static_cast<T*>(out), so[0], so[1], so[2], B, Hq, Hk, Sq, Sk, causal,
                       scale_log2, nblk, qoff, stats);
    return hipGetLastError();
  };
  return stats ? go(attn_dense_kernel<T, D, true>) : go(attn_dense_kernel<T, D, false>);
}

// Dense attention, or the row statistics when stats is given, of operands the
// MFMA attention takes (bf16/fp16, D 64 or 128, aligned rows).
hipError_t launch_attn_dense(int dtype, int64_t D, const void* q, const int64_t* sq,
                             const void* k, const int64_t* sk, const void* v, const int64_t* sv,
                             void* out, const int64_t* so, int64_t B, int64_t Hq, int64_t Hk,
                             int64_t Sq, int64_t Sk, int causal, float scale_log2, int64_t qoff,
                             float* stats, hipStream_t stream) {
#define VA_DENSE_CASE(TT, DD)                                                                    \
  return launch_dense_td<TT, DD>(q, sq, k, sk, v, sv, out, so, B, Hq, Hk, Sq, Sk, causal,       \
                                 scale_log2, qoff, stats, stream)
  if (dtype == kBF16 && D == 128) VA_DENSE_CASE(bf16_t, 128);
  if (dtype == kBF16 && D == 64) VA_DENSE_CASE(bf16_t, 64);
  if (dtype == kF16 && D == 128) VA_DENSE_CASE(f16_t, 128);
  if (dtype == kF16 && D == 64) VA_DENSE_CASE(f16_t, 64);
#undef VA_DENSE_CASE
  return hipErrorInvalidValue;
}

}  // namespace va
