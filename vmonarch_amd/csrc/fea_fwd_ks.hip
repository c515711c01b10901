// FlashEntropyAttention forward for launches with few query tiles (gfx950).
//
// The 128-query kernel (fea_fwd.hip) walks a problem's keys serially in 64-key stages of ~0.8 us (64-wide heads) to
// ~1.05 us (128-wide) with one workgroup to the CU, so a launch of few tiles takes one workgroup's whole key loop while most CUs idle: (1, 2,
// 1024, 64) was 16 workgroups of 16 stages, 16.8 us.  Here a workgroup takes fewer queries and its waves split the
// keys: wave (qg, kg) of QG x KG takes query block qg (32 queries) and the 32-key block kg of every stage of 32 KG
// keys, with its own sums and accumulators, all relative to the row's one reference point; a tree over the key
// groups through LDS adds them at the end.  1 x 8 (32 queries; 64-wide heads, whose 256-key stage fits the LDS
// twice) has a quarter, 2 x 4 (64 queries) half of the work per CU.  Measured (online entropy, us, 128-query kernel ->
// this): 64-wide, N = 1024, 2 heads 16.8 -> 9.7, N = 1000, 8 heads 17.2 -> 10.3, N = 4096, 4 heads 52.5 -> 31.8;
// 128-wide, N = 1024, 4 heads 22.0 -> 16.7, N = 4096, 4 heads 68.0 -> 46.9.
// (Eight waves on 128 queries, 4 x 2, leave each SIMD the same work: 37.9 -> 38.6 us at N = 2048, 8 heads, 128-wide.)
// Layouts, the fixed reference point m (the max of the problem's first 32 keys) with the exact two-pass fallback,
// the rounding of P and the entropy modes are those of the 128-query kernel: the same p bit for bit, summed in
// another order.
#include <atomic>
#include <type_traits>

#include "fea_fwd.h"

namespace vmo {

constexpr int kKsWaves = 8;
constexpr int kKsLdsMax = 160 * 1024;

template <int D, int DW0, int DW1, bool W0K, int KG>
constexpr int ks_stage_bytes() { return 32 * KG * (D + (W0K ? 0 : DW0) + DW1) * 2; }
template <int D, int DW0, int DW1, bool W0K, int KG>
constexpr int ks_slots() { return 3 * ks_stage_bytes<D, DW0, DW1, W0K, KG>() <= kKsLdsMax ? 3 : 2; }
// The merge's LDS: (l, h) of every wave's 32 rows, then one slot of NA accumulator blocks per receiving wave.
constexpr int kKsStatBytes = 4096;
template <int D, int DW0, int DW1, bool W0K, int KG>
constexpr int ks_lds_bytes() {
  constexpr int ring = ks_slots<D, DW0, DW1, W0K, KG>() * ks_stage_bytes<D, DW0, DW1, W0K, KG>();
  constexpr int merge = kKsStatBytes + kKsWaves / 2 * (DW0 + DW1) / 32 * 4096;
  return ring > merge ? ring : merge;
}

template <bool F16, int D, int DW0, int DW1, bool W0K, int ENT, int QG, int KG>
__global__ __launch_bounds__(64 * QG * KG, 2) void fea_fwd_ks_kernel(FwdParams p) {
  using E = Elem<F16>;
  using T = typename E::T;
  using V8 = typename E::V8;
  using V2 = typename E::V2;
  constexpr int WAVES = QG * KG, SK = 32 * KG;
  static_assert(WAVES == kKsWaves, "eight waves");
  constexpr int K_BYTES = SK * D * 2;
  constexpr int W0_BYTES = W0K ? 0 : SK * DW0 * 2;
  constexpr int STAGE = ks_stage_bytes<D, DW0, DW1, W0K, KG>();
  constexpr int NSLOT = ks_slots<D, DW0, DW1, W0K, KG>();
  static_assert(ks_lds_bytes<D, DW0, DW1, W0K, KG>() <= kKsLdsMax, "LDS");
  constexpr int NDS = D / 16, NA0 = DW0 / 32, NA1 = DW1 / 32, NA = NA0 + NA1;
  constexpr int DMA_PER_TILE = STAGE / 1024 / WAVES;
  static_assert(STAGE % (1024 * WAVES) == 0, "whole copy instructions per wave");
  static_assert(!W0K || DW0 == D, "w0 aliases k");
  static_assert(ENT != kEntFromPK || W0K, "entropy from P.K needs w0 == k");

  extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
  VMO_LDS char* smem = (VMO_LDS char*)smem_raw;
  const uint32_t smem_u32 = (uint32_t)(uintptr_t)smem;

  const int L = xcd_remap(gridDim.x);
  if (L >= p.total_wg) return;
  auto uni = [](int v) __attribute__((always_inline)) { return __builtin_amdgcn_readfirstlane(v); };
  const int qt = uni(L % p.q_tiles), prob = uni(L / p.q_tiles);
  const int f = uni(prob % p.frames), bh = uni(prob / p.frames), hh = uni(bh % p.heads), bb = uni(bh / p.heads);
  const T* qb = (const T*)p.q + bb * p.q_sb + hh * p.q_sh + (int64_t)f * p.nq * p.q_sn;
  const T* kb = (const T*)p.k + bb * p.k_sb + hh * p.k_sh + (int64_t)f * p.nk * p.k_sn;
  const T* w0b = (const T*)p.w0 + bb * p.w0_sb + hh * p.w0_sh + (int64_t)f * p.nk * p.w0_sn;
  const T* w1b = DW1 ? (const T*)p.w1 + bb * p.w1_sb + hh * p.w1_sh + (int64_t)f * p.nk * p.w1_sn : nullptr;

  const int n_tiles = uni((p.nk + SK - 1) / SK);
  const int tid = threadIdx.x, wave = uni(tid >> 6), lane = tid & 63, hl = lane >> 5, l32 = lane & 31;
  const int qg = wave % QG, kg = wave / QG;
  const int q0 = (qt * QG + qg) * 32;
  const bool wave_live = q0 < p.nq;
  const int qrow = q0 + l32;
  const bool qvalid = qrow < p.nq;

  // Q^T as the B operand: lane (query l32, half hl) holds q[query][16 ds + 8 hl + 0..7].
  V8 qf[NDS];
  {
    const T* qp = qb + (int64_t)(qvalid ? qrow : 0) * p.q_sn + hl * 8;
#pragma unroll
    for (int ds = 0; ds < NDS; ++ds) {
      const V8 v = *(const V8*)(qp + ds * 16);
      qf[ds] = qvalid ? v : V8{};
    }
  }

  const TileCopy<T, D, WAVES, D, SK> kcopy(kb, p.k_sn, wave, lane);
  const TileCopy<T, W0K ? 64 : DW0, WAVES, W0K ? 64 : DW0, SK> w0copy(w0b, p.w0_sn, wave, lane);
  const TileCopy<T, DW1 ? DW1 : 64, WAVES, DW1 ? DW1 : 64, SK> w1copy(w1b, p.w1_sn, wave, lane);
  auto issue = [&](int t) __attribute__((always_inline)) {
    const uint32_t st = smem_u32 + (uint32_t)((t % NSLOT) * STAGE);
    kcopy.issue(t * SK, p.nk, st);
    if constexpr (!W0K) w0copy.issue(t * SK, p.nk, st + K_BYTES);
    if constexpr (DW1 > 0) w1copy.issue(t * SK, p.nk, st + K_BYTES + W0_BYTES);
  };

  const float c = p.scale_log2;
  constexpr float kSumLimit = F16 ? 65504.f : 1.8446744e19f;   // as the 128-query kernel: fp16 max / 2^64
  float m_run = kMaskLogit, l_run = 0.f, h_run = 0.f;
  f32x16 acc[NA];
#pragma unroll
  for (int a = 0; a < NA; ++a) acc[a] = f32x16{};
  bool overflow = false;

  const int ksw = swz_rows<D * 2>(l32);
  const int trow = 4 * hl + ((lane & 15) >> 2);
  const int tchunk = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
  const int tbyte = (lane & 1) * 8;

  // S^T of key block blk of a stage, operand reads two ahead of their MFMAs
  constexpr int kPre = 2;
  auto qk_block = [&](const VMO_LDS char* Ks, int blk) __attribute__((always_inline)) {
    const VMO_LDS char* arow = Ks + (32 * blk + l32) * (D * 2);
    V8 a[NDS];
#pragma unroll
    for (int ds = 0; ds < NDS; ++ds) a[ds] = lds_read8<V8>(arow + ((2 * ds + hl) ^ ksw) * 16);
    f32x16 x = f32x16{};
#pragma unroll
    for (int ds = 0; ds < NDS; ++ds) x = E::mfma(a[ds], qf[ds], x);
    __builtin_amdgcn_sched_group_barrier(0x100, kPre, 0);
#pragma unroll
    for (int ds = 0; ds < NDS - kPre; ++ds) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, kPre, 0);
    return x;
  };
  auto mask_block = [&](f32x16& x, int nvalid) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 16; ++r)
      if (8 * (r >> 2) + 4 * hl + (r & 3) >= nvalid) x[r] = kMaskLogit;
  };
  auto block_max = [&](f32x16 x, int nvalid) __attribute__((always_inline)) {   // over the valid keys, in units of x c
    mask_block(x, nvalid);
    float v = x[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) v = fmaxf(v, x[r]);
    return wave_max32(v) * c;
  };
  auto pv_part = [&](const VMO_LDS char* W, auto rb_tag, auto na_tag, int a0, const V8 (&P)[2]) __attribute__((always_inline)) {
    constexpr int RB = decltype(rb_tag)::value, NAP = decltype(na_tag)::value;
    V8 wt[2 * NAP];
    const int tsw = swz_rows<RB>(trow);
#pragma unroll
    for (int a = 0; a < NAP; ++a) {
      const int c0 = trow * RB + (((4 * a + tchunk) ^ tsw) * 16 + tbyte);
#pragma unroll
      for (int h2 = 0; h2 < 2; ++h2) {   // rows 16 h2 + trow and 8 further down (chunk bit 1 of the swizzle flips)
        const VMO_LDS char* rp = W + (32 * kg + 16 * h2) * RB;
        wt[2 * a + h2] = lds_read_tr8<V8>(rp + c0, rp + 8 * RB + (c0 ^ 32));
      }
    }
#pragma unroll
    for (int a = 0; a < NAP; ++a)
#pragma unroll
      for (int h2 = 0; h2 < 2; ++h2) acc[a0 + a] = E::mfma(wt[2 * a + h2], P[h2], acc[a0 + a]);
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
    for (int o = 0; o < 2 * NAP - 2; ++o) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
  };
  // this wave's 32-key block of one stage
  auto block = [&](const VMO_LDS char* Ks, int nvalid, auto masked_tag) __attribute__((always_inline)) {
    f32x16 x = qk_block(Ks, kg);
#pragma unroll
    for (int r = 0; r < 16; ++r) x[r] = fmaf(x[r], c, -m_run);
    if constexpr (decltype(masked_tag)::value) mask_block(x, nvalid);
    float ls0, ls1, hs0, hs1;   // two partial sums per lane
    uint32_t w[8];
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
      const float p0 = fast_exp2(x[r]), p1 = fast_exp2(x[r + 1]);
      const V2 pk = E::pack2(p0, p1);
      w[r / 2] = __builtin_bit_cast(uint32_t, pk);
      float s2;
      if constexpr (ENT == kEntFromPK) {   // the sum of the rounded weights (the entropy's P.K mean uses them)
        if constexpr (F16) s2 = (float)pk[0] + (float)pk[1];
        else s2 = __uint_as_float(w[r / 2] << 16) + __uint_as_float(w[r / 2] & 0xffff0000u);
      } else {
        s2 = p0 + p1;
      }
      const float h2 = ENT == kEntOnline ? fmaf(p1, x[r + 1], p0 * x[r]) : 0.f;
      if (r == 0) { ls0 = s2; hs0 = h2; }
      else if (r == 2) { ls1 = s2; hs1 = h2; }
      else if (r & 2) { ls1 += s2; hs1 += h2; }
      else { ls0 += s2; hs0 += h2; }
    }
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const V8 P[2] = {__builtin_bit_cast(V8, u32x4{w[0], w[1], w[2], w[3]}),
                     __builtin_bit_cast(V8, u32x4{w[4], w[5], w[6], w[7]})};
    const float ls = ls0 + ls1;
    overflow |= !(ls <= kSumLimit);   // also catches inf / nan
    l_run += ls;
    if constexpr (ENT == kEntOnline) h_run += hs0 + hs1;
    pv_part(W0K ? Ks : Ks + K_BYTES, std::integral_constant<int, DW0 * 2>{}, std::integral_constant<int, NA0>{}, 0, P);
    if constexpr (DW1 > 0)
      pv_part(Ks + K_BYTES + W0_BYTES, std::integral_constant<int, DW1 * 2>{}, std::integral_constant<int, NA1>{}, NA0, P);
  };

  // Stages 0 .. n_tiles - 1 through the LDS ring, the copies NSLOT - 1 stages ahead; every wave takes part in every
  // copy and barrier.  Only the last stage has fewer than 32 keys for some wave (none, even), and it is peeled: the
  // steady body is one straight path and the accumulators stay in place.  Waves without queries compute on zero
  // rows and store nothing.
  auto slot = [&](int t) __attribute__((always_inline)) { return (const VMO_LDS char*)smem + (t % NSLOT) * STAGE; };
  auto prime = [&]() __attribute__((always_inline)) {
    issue(0);
    if (NSLOT == 3 && n_tiles > 1) issue(1);
  };
  const int n_last = p.nk - (n_tiles - 1) * SK - 32 * kg;   // this wave's valid keys in the last stage
  auto for_stages = [&](auto&& steady, auto&& last) __attribute__((always_inline)) {
    for (int t = 0; t < n_tiles - 1; ++t) {
      tile_sync<NSLOT == 3 ? DMA_PER_TILE : 0>();
      if (t + NSLOT - 1 < n_tiles) issue(t + NSLOT - 1);
      steady(slot(t));
    }
    tile_sync<0>();
    if (n_last > 0) last(slot(n_tiles - 1));
  };
  auto key_loop = [&]() __attribute__((always_inline)) {
    for_stages([&](const VMO_LDS char* Ks) __attribute__((always_inline)) { block(Ks, 32, std::false_type{}); },
               [&](const VMO_LDS char* Ks) __attribute__((always_inline)) { block(Ks, n_last, std::true_type{}); });
  };
  prime();
  if (NSLOT == 3 && n_tiles > 1) tile_sync<DMA_PER_TILE>(); else tile_sync<0>();
  m_run = block_max(qk_block(slot(0), 0), p.nk);   // (tile 0 stays in its slot for the loop)
  key_loop();

  __syncthreads();   // the ring is free
  VMO_LDS float* st = (VMO_LDS float*)smem;
  {
    const bool any = __builtin_amdgcn_ballot_w64(overflow) != 0;
    VMO_LDS int* words = (VMO_LDS int*)smem;
    if (lane == 0) words[wave] = any ? 1 : 0;
    __syncthreads();
    int some = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) some |= words[w];
    __syncthreads();
    if (some) {   // exact two-pass fallback: the true row max, over all key groups, then the loop again
      m_run = kMaskLogit;
      prime();
      for_stages([&](const VMO_LDS char* Ks) __attribute__((always_inline)) { m_run = fmaxf(m_run, block_max(qk_block(Ks, kg), 32)); },
                 [&](const VMO_LDS char* Ks) __attribute__((always_inline)) { m_run = fmaxf(m_run, block_max(qk_block(Ks, kg), n_last)); });
      l_run = h_run = 0.f;
#pragma unroll
      for (int a = 0; a < NA; ++a) acc[a] = f32x16{};
      tile_sync<0>();   // every wave is done with the ring
      if (hl == 0) st[wave * 32 + l32] = m_run;
      __syncthreads();
#pragma unroll
      for (int g = 0; g < KG; ++g) m_run = fmaxf(m_run, st[(g * QG + qg) * 32 + l32]);
      __syncthreads();
      prime();
      key_loop();
      __syncthreads();
    }
  }

  // Merge the key groups: sums relative to one reference point, so they add.
  {
    const float l_w = wave_sum32(l_run), h_w = ENT == kEntOnline ? wave_sum32(h_run) : 0.f;
    if (hl == 0) {
      st[wave * 32 + l32] = l_w;
      if constexpr (ENT == kEntOnline) st[256 + wave * 32 + l32] = h_w;
    }
  }
  __syncthreads();
  float l_tot = 0.f, h_tot = 0.f;
#pragma unroll
  for (int g = 0; g < KG; ++g) {
    l_tot += st[(g * QG + qg) * 32 + l32];
    if constexpr (ENT == kEntOnline) h_tot += st[256 + (g * QG + qg) * 32 + l32];
  }
  const float inv_l = 1.0f / l_tot;
  VMO_LDS char* slots = smem + kKsStatBytes;
#pragma unroll
  for (int h = KG / 2; h >= 1; h /= 2) {   // key groups h .. 2 h - 1 hand their blocks to 0 .. h - 1
    if (kg >= h && kg < 2 * h) {
      VMO_LDS char* d = slots + (wave - h * QG) * (NA * 4096) + lane * 16;
#pragma unroll
      for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 v{acc[a][4 * g], acc[a][4 * g + 1], acc[a][4 * g + 2], acc[a][4 * g + 3]};
          *(VMO_LDS f32x4*)(d + (4 * a + g) * 1024) = v;
        }
    }
    __syncthreads();
    if (kg < h) {
      const VMO_LDS char* d = slots + wave * (NA * 4096) + lane * 16;
#pragma unroll
      for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 v = *(const VMO_LDS f32x4*)(d + (4 * a + g) * 1024);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[a][4 * g + e] += v[e];
        }
    }
    if (h > 1) __syncthreads();   // the next round's slots are the first of this round's
  }
  if (kg > 0 || !wave_live) return;

  // sum_j p~_j q . k_j / l~ (the P.K entropy) from the q operand registers, as the
  // 128-query kernel takes it.
  float ent = 0.f;
  const float log2l = fast_log2(l_tot), lse = m_run + log2l;
  if constexpr (ENT == kEntOnline) {
    ent = (log2l - h_tot * inv_l) * kLn2;
  } else if constexpr (ENT == kEntFromPK) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    float d = 0.f;
#pragma unroll
    for (int ds = 0; ds < NDS; ++ds) {
      const u32x4 w = __builtin_bit_cast(u32x4, qf[ds]);
      const auto s0 = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
      const auto s1 = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
      const uint32_t xy[4] = {s0[0], s1[0], s0[1], s1[1]};
      const int r0 = 8 * (ds & 1);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const V2 x = __builtin_bit_cast(V2, xy[u]);
        d = fmaf((float)x[0], acc[ds >> 1][r0 + 2 * u], d);
        d = fmaf((float)x[1], acc[ds >> 1][r0 + 2 * u + 1], d);
      }
    }
    ent = lse * kLn2 - (c * kLn2) * wave_sum32(d) * inv_l;
  }
  // the wave's own slot was last read by itself: its row-store patch
  VMO_LDS float* patch = (VMO_LDS float*)(slots + wave * (NA * 4096));
  asm volatile("" ::: "memory");
  T* const ob = (T*)p.o + bb * p.o_sb + hh * p.o_sh + ((int64_t)f * p.nq + q0) * p.o_sn;
  store_acc_rows<F16>(patch, acc, NA, inv_l, kGradStore, (char*)ob, p.o_sn * 2, min(32, p.nq - q0), lane);
  if (qvalid && hl == 0) {
    const int64_t si = bb * p.st_sb + hh * p.st_sh + (int64_t)f * p.nq + qrow;
    if (ENT != kEntNone && p.ent) p.ent[si] = ent;
    if (p.lse) p.lse[si] = lse;
  }
}

template <bool F16, int D, int DW0, int DW1, bool W0K, int ENT, int QG>
static int launch_ks(FwdParams p, hipStream_t stream) {
  constexpr int KG = kKsWaves / QG;
  constexpr int LDS = ks_lds_bytes<D, DW0, DW1, W0K, KG>();
  p.q_tiles = (p.nq + 32 * QG - 1) / (32 * QG);
  p.total_wg = p.problems * p.q_tiles;
  auto kern = fea_fwd_ks_kernel<F16, D, DW0, DW1, W0K, ENT, QG, KG>;
  if (LDS > 65536) {
    static std::atomic<bool> done{false};   // the attribute is per function, and setting it again changes nothing
    if (!done.load(std::memory_order_relaxed)) {
      if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) != hipSuccess)
        return set_error(VMO_ERR_LAUNCH, "fea_fwd_ks: cannot raise the LDS limit to %d bytes", LDS);
      done.store(true, std::memory_order_relaxed);
    }
  }
  hipLaunchKernelGGL(kern, dim3(xcd_grid(p.total_wg)), dim3(64 * kKsWaves), LDS, stream, p);
  return launch_status("fea_fwd_ks");
}

// Query blocks per workgroup, or 0 for the 128-query kernel: the smallest tile that still leaves at most one
// workgroup per CU, since the launch then takes the time of one workgroup's key loop.  Past that line the smaller tile
// loses (64-wide, N = 2048: 8 heads, 256 tiles of 64 queries, 29.4 -> 18.6 us; 12 heads, 384 tiles, 29.9 -> 33.9).
// Below 512 keys the loop is too short to pay for the merge (values k, 256 keys: 7.6 -> 7.4 us, 128-wide 9.9 -> 10.3).
constexpr int kCus = 256, kKsMinKeys = 512;
static int ks_query_blocks(const FwdParams& p, bool eight) {
  auto wgs = [&](int queries) { return (int64_t)p.problems * ((p.nq + queries - 1) / queries); };
  if (p.nk < kKsMinKeys) return 0;
  return eight && wgs(32) <= kCus ? 1 : wgs(64) <= kCus ? 2 : 0;
}

template <bool F16, int D, int DW0, int DW1, bool W0K, int ENT>
static bool dispatch_ks(const FwdParams& p, hipStream_t s, int* rc, int* tile) {
  constexpr bool EIGHT = D == 64 && ks_lds_bytes<D, DW0, DW1, W0K, 8>() <= kKsLdsMax;
  const int qg = ks_query_blocks(p, EIGHT);
  if (qg == 0) return false;
  if (tile) { *tile = 32 * qg; return true; }
  if constexpr (EIGHT)
    if (qg == 1) { *rc = launch_ks<F16, D, DW0, DW1, W0K, ENT, 1>(p, s); return true; }
  *rc = launch_ks<F16, D, DW0, DW1, W0K, ENT, 2>(p, s);
  return true;
}

template <bool F16>
static bool dispatch_ks_dims(const FwdParams& p, int d, int dw0, int dw1, bool w0k, bool ent, hipStream_t s, int* rc, int* tile) {
#define VMO_KS(D_, DW0_, DW1_, W0K_, ENT_)                                                  \
  if (d == D_ && dw0 == DW0_ && dw1 == DW1_ && w0k == W0K_ && ent == (ENT_ != kEntNone))    \
    return dispatch_ks<F16, D_, DW0_, DW1_, W0K_, ENT_>(p, s, rc, tile);
  VMO_KS(64, 64, 0, false, kEntOnline)
  VMO_KS(64, 128, 0, false, kEntOnline)
  VMO_KS(128, 128, 0, false, kEntOnline)
  VMO_KS(64, 64, 0, true, kEntFromPK)
  VMO_KS(64, 64, 64, true, kEntFromPK)
  VMO_KS(128, 128, 0, true, kEntFromPK)
  VMO_KS(128, 128, 128, true, kEntFromPK)
#undef VMO_KS
  return false;
}

bool fwd_ks(const FwdParams& p, bool f16, int d, int dw0, int dw1, bool w0k, bool ent, hipStream_t stream, int* rc, int* tile) {
  return f16 ? dispatch_ks_dims<true>(p, d, dw0, dw1, w0k, ent, stream, rc, tile)
             : dispatch_ks_dims<false>(p, d, dw0, dw1, w0k, ent, stream, rc, tile);
}

}  // namespace vmo
