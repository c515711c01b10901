// Multi-block fused L-step for gfx950: grids of more than 32 frames (and head dims 16 / 32 / 64 / 128 at
// any frame count up to kMbMaxFrames), on MFMA.
//
// Reference: video_monarch_attention/vmonarch.py:51-63 -- per grid column j (the same spatial position in
// all m frames) an m x m attention over the frames:
//   attn[i, k] = softmax_k(scale q_i . kr_k + ent_k),  kr = out[..., :D]
//   last:      z_i = sum_k attn[i, k] y_k,  y = out[..., D:]
//   otherwise: u_k = scale / max(sum_i attn[i, k], min_col_mass) * sum_i attn[i, k] q_i
// (the one-tile kernels in lstep.hip take m <= 32 in a single 32 x 32 MFMA tile per column).
//
// Here one 4-wave workgroup owns a column: its q, kr (and y) rows -- tokens i b + j, i < m -- are staged
// whole into swizzled LDS tiles of M = 32 * MB rows (MB = ceil(m / 32) <= kMbMaxBlocks; rows past m are
// finite data whose weights are exact zeros), and the m x m products run on v_mfma_f32_32x32x16 in 32 x 32
// blocks (two-block grids run kernel instantiations, TWO, whose passes split over all four waves):
//   * last: wave w owns query block w.  S^T blocks (keys x queries: one query row per lane) for every key
//     block, softmax over all of them in registers (max, sum, normalise: the attention is rounded to the
//     16-bit type only once normalised, as the reference's attn.to(y.dtype)), then z^T += Y^T P^T with the
//     S^T accumulators as the B operand and Y^T read by ds_read_tr16_b64, whose 4-row groups match the
//     accumulator's (no key permutation);
//   * otherwise two passes: (1) wave w computes the log-sum-exp of its query block's rows (S^T blocks as
//     above) into LDS; (2) wave w owns key block w: L blocks (queries x keys: one key per lane) = Q Kr^T for
//     every query block, attn = exp2(L c + ent_k - lse_i) exactly normalised, the column mass as an in-lane
//     sum of the fp32 attn, and u^T += Q^T attn with Q^T by transposed reads.
// Rounding points as the one-tile kernels: logits in fp32 from the 16-bit q and kr, attn rounded to the
// 16-bit type where it multiplies q or y, the column mass from the fp32 attn, u / z rounded once when stored.
// Results leave through per-wave LDS patches as whole row segments (store_acc_rows).
#include <atomic>

#include "vmo_common.h"
#include "vmo_host.h"
#include "lstep_params.h"

namespace vmo {

constexpr int kMbWaves = 4;
constexpr int kMbMaxBlocks = 4;                  // one 32-row block per wave
constexpr int kMbMaxFrames = 32 * kMbMaxBlocks;  // m <= 128

// Byte offsets of a column's LDS arrays: 16-bit row tiles (q, kr, and y for the last step; the backward's
// upstream gradient), M-float vectors (entropy bias, row LSE; the backward's row sums rs_i, column factors f_k
// and dc_k).  The forward's row-store patches (kEpiPatchBytes per wave) reuse the start of the allocation
// once every wave has passed the barrier that ends the compute; the backward, which stores between its
// passes, has patches of its own -- half-size ones (16 rows at a time) for the last step up to 64 frames, whose
// four tiles at head dim 128 then leave room for two workgroups per CU (73.3 instead of 81.3 KB); beyond that one
// workgroup fits either way, and the whole patches store faster.
__host__ __device__ constexpr int mb_bwd_patch_rows(bool last, int M) { return last && M <= 64 ? 16 : 32; }
struct MbLayout {
  int q, k, y, g, e, lse, part, rs, f, dc, patch, patch_rows, mat0, mat1, total;
};
// A staged tile holds M = 32 ceil(m / 32) rows, those past m zeros (finite data whose weights are exact zeros).
// A compact tile (CT: the two-block last-step kernels up to kMbCompactMaxFrames, where it lets one more column
// share the CU) holds the m rows, the rows by which the last copy instruction overhangs them (copies of row
// m - 1; one instruction covers 1024 / rb rows of rb bytes) and one zero row, at which every operand read of a
// row past m is pointed.  The other kernels keep whole blocks: their reads take each block's rows at immediate
// offsets from one per-lane address, where the compact tile needs a clamped address per block (a build with
// compact tiles everywhere ran up to 14% slower on the grids it gave no extra column).
__host__ __device__ constexpr int mb_zero_row(int m, int rb) { return (m + 1024 / rb - 1) / (1024 / rb) * (1024 / rb); }
__host__ __device__ constexpr int mb_tile_bytes(int m, int rb, bool compact) {
  return compact ? (mb_zero_row(m, rb) + 1) * rb : (m + 31) / 32 * 32 * rb;
}
// Compact tiles are built for the two-block last step at head dims 128 / 128 and taken up to 40 frames: there its
// four tiles (three in the forward) shrink enough for one more column per CU (the backward 3 instead of 2, the
// forward 4 instead of 3); beyond that, or with narrower tiles, the per-row clamp costs without a column to gain.
constexpr int kMbCompactMaxFrames = 40;
constexpr bool mb_compact_built(int d, int dv, bool last) { return last && d == 128 && dv == 128; }
template <int RB, bool CT>
__device__ __forceinline__ int mb_phys_row(int r, int m) {
  if constexpr (CT) return r < m ? r : mb_zero_row(m, RB);
  else return r;
}

__host__ __device__ inline MbLayout mb_layout(int m, int d, int dv, bool last, bool bwd, bool compact) {
  MbLayout L{};
  const int M = 32 * ((m + 31) / 32);
  int off = 0;
  auto take = [&](int bytes) { const int o = off; off += (bytes + 255) / 256 * 256; return o; };
  L.q = take(mb_tile_bytes(m, d * 2, compact));
  L.k = take(mb_tile_bytes(m, d * 2, compact));
  L.y = last ? take(mb_tile_bytes(m, dv * 2, compact)) : 0;
  L.g = bwd ? take(mb_tile_bytes(m, (last ? dv : d) * 2, compact)) : 0;
  L.e = take(M * 4);
  L.lse = take(M * 4);
  L.part = take(4 * M * 4);   // two blocks' partial row / column vectors (the two-block passes)
  L.rs = bwd ? take(M * 4) : 0;
  L.f = bwd ? take(M * 4) : 0;
  L.dc = bwd ? take(M * 4) : 0;
  L.patch = bwd ? take(kMbWaves * mb_bwd_patch_rows(last, M) * 32 * 4) : 0;
  L.patch_rows = mb_bwd_patch_rows(last, M);
  L.total = off > kMbWaves * kEpiPatchBytes ? off : kMbWaves * kEpiPatchBytes;
  return L;
}

// The one-block-per-wave backward (every grid that is not two blocks on four waves) hands m x m matrices -- the
// attention, dl, a f, rounded to the 16-bit type as MFMA operands -- from the waves that form them (one row or column
// block each) to the waves that need them in the other orientation, through an LDS matrix of M rows of 256 bytes (M
// <= 128 columns).  It overlays what is dead by then: the last step's kr and y tiles, the other steps' q tile and the
// row-store patches after it.  The last step reads its waves' own q and g rows from HBM into registers (MFMA operands)
// and writes their tiles from there, where the other orientation needs them whole, beside the matrix; so kr and y are
// all it stages, and two columns share a CU up to 128 frames at 128-wide heads.  The patches hold 32, 16 or 8 rows
// per wave: the most that does not cost a column per CU.
constexpr int kMbMatRow = 256;
__host__ __device__ inline MbLayout mb_layout_bwd1(int m, int d, int dv, bool last) {
  const int M = 32 * ((m + 31) / 32), mat = M * kMbMatRow;
  MbLayout best{};
  for (int rows = 32; rows >= 8; rows /= 2) {
    MbLayout L{};
    int off = 0;
    auto take = [&](int bytes) { const int o = off; off += (bytes + 255) / 256 * 256; return o; };
    auto at_least = [](int a, int b) { return a > b ? a : b; };
    L.patch_rows = rows;
    const int patches = kMbWaves * rows * 32 * 4;
    if (last) {   // kr and y; once both are dead the matrix, and after it g's tile, then q's
      const int rows_gq = M * (d > dv ? d : dv) * 2;
      L.k = take(at_least(M * (d + dv) * 2, mat + rows_gq));
      L.y = L.k + M * d * 2;
      L.mat0 = L.mat1 = L.k;
      L.q = L.g = L.k + mat;
      L.patch = take(patches);
    } else {
      L.k = take(M * d * 2);
      L.g = take(M * d * 2);
      L.q = take(at_least(M * d * 2 + patches, mat));
      L.patch = L.q + M * d * 2;
      L.mat0 = L.mat1 = L.q;
      L.lse = take(M * 4);
      L.part = take(4 * M * 4);
    }
    L.e = take(M * 4);
    L.rs = take(M * 4);
    L.total = off;
    if (best.total == 0 || 160 * 1024 / L.total > 160 * 1024 / best.total) best = L;
  }
  return best;
}

// Stage the m rows of W 16-bit values (row r: src + r rs) into a tile whose chunk c of row r sits at chunk
// c ^ swz_rows(r): wave instruction inst covers rows inst RPI .. + RPI - 1, lane l lands at byte 16 l of its
// 1 KB and so loads global chunk (l % CH) ^ swz_rows(row).  Only instructions that hold a row below m copy
// (their rows past m repeat row m - 1); the rows after them are zeroed up to M (a compact tile: the one zero
// row, mb_zero_row).  SW < W: a 16-wide tensor in a 32-wide tile (tile_w), each row's two chunks stored twice.
template <class T, int W, int SW = W, bool CT = false>
__device__ __forceinline__ void mb_stage(const T* src, int64_t rs, int m, VMO_LDS char* dst, int wave, int lane) {
  constexpr int RB = W * 2, CH = RB / 16, RPI = 64 / CH;
  const int c = lane % CH;
  const int ninst = (m + RPI - 1) / RPI;
  for (int inst = wave; inst < ninst; inst += kMbWaves) {
    const int r = inst * RPI + lane / CH;
    const int rr = r < m ? r : m - 1;
    g2l_16(src + (int64_t)rr * rs + ((c ^ swz_rows<RB>(r)) & (SW / 8 - 1)) * 8, dst + inst * 1024);
  }
  const int end = CT ? ninst * 1024 + RB : (m + 31) / 32 * 32 * RB;
  for (int o = ninst * 1024 + (64 * wave + lane) * 16; o < end; o += 64 * kMbWaves * 16)
    *(VMO_LDS i32x4*)(dst + o) = i32x4{0, 0, 0, 0};
}

// Row-read MFMA operand: lane (row l32 of 32-row block blk of the tile, half hl) gets elements 16 ds + 8 hl .. + 7
// (zeros for a row past m).
template <class V8, int RB, bool CT = false>
__device__ __forceinline__ V8 mb_row8(const VMO_LDS char* tile, int blk, int m, int l32, int hl, int ds) {
  if constexpr (CT) {
    const int r = mb_phys_row<RB, CT>(32 * blk + l32, m);
    return lds_read8<V8>(tile + r * RB + ((2 * ds + hl) ^ swz_rows<RB>(r)) * 16);
  } else {   // (swz_rows depends on the row mod 16 alone)
    return lds_read8<V8>(tile + 32 * blk * RB + l32 * RB + ((2 * ds + hl) ^ swz_rows<RB>(l32)) * 16);
  }
}

// Transposed MFMA A operand for the 32 columns 32 a .. 32 a + 31 of a row-major tile, K step h2 (16 rows) of
// its 32-row block blk: the rows are taken in the S^T / L accumulator's order (rows 4 hl + 0..3 and
// 8 + 4 hl + 0..3 of the step), so that accumulator rows 8 h2 .. 8 h2 + 7, rounded, are the B operand.  Each
// lane reads 8 bytes of one row; a row past m is read from the zero row.
template <class V8, int RB, bool CT = false>
__device__ __forceinline__ V8 mb_tr8(const VMO_LDS char* tile, int blk, int m, int lane, int a, int h2) {
  const int hl = lane >> 5;
  const int trow = 4 * hl + ((lane & 15) >> 2);
  const int tchunk = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
  const int tbyte = (lane & 1) * 8;
  if constexpr (CT) {
    const int r0 = mb_phys_row<RB, CT>(32 * blk + 16 * h2 + trow, m);
    const int r1 = mb_phys_row<RB, CT>(32 * blk + 16 * h2 + trow + 8, m);
    return lds_read_tr8<V8>(tile + r0 * RB + ((4 * a + tchunk) ^ swz_rows<RB>(r0)) * 16 + tbyte,
                            tile + r1 * RB + ((4 * a + tchunk) ^ swz_rows<RB>(r1)) * 16 + tbyte);
  } else {   // row 8 further on: the swizzle's chunk bit 1 flips
    const int c0 = trow * RB + (((4 * a + tchunk) ^ swz_rows<RB>(trow)) * 16 + tbyte);
    const VMO_LDS char* rp = tile + (32 * blk + 16 * h2) * RB;
    return lds_read_tr8<V8>(rp + c0, rp + 8 * RB + (c0 ^ 32));
  }
}

// Accumulator rows 8 h2 .. 8 h2 + 7 of x, times f, rounded to the 16-bit type: a B operand.
template <class T, class V8>
__device__ __forceinline__ V8 mb_pack(const f32x16& x, int h2, float f) {
  V8 v;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = to_elem<T>(x[8 * h2 + e] * f);
  return v;
}

template <bool F16, int D, int DV, bool LAST, bool TWO, bool CT>
__global__ __launch_bounds__(64 * kMbWaves, TWO && !LAST ? 4 : 2) void lstep_mb_kernel(LParams p) {
  using E = Elem<F16>;
  using T = typename E::T;
  using V8 = typename E::V8;
  constexpr int DK = tile_w(D), DVK = tile_w(DV);   // widths in LDS
  static_assert(!CT || (LAST && TWO), "compact tiles: the two-block last-step kernels");
  constexpr int NDS = D / 16;
  constexpr int NACC = (LAST ? DVK : DK) / 32;
  constexpr int CW = (LAST ? DV : D) < 32 ? 16 : 32;   // stored columns per accumulator block
  constexpr int RBD = DK * 2, RBY = DVK * 2;
  extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
  VMO_LDS char* sm = (VMO_LDS char*)smem_raw;

  const int m = p.m, MB = (m + 31) / 32, M = 32 * MB;
  const MbLayout Lo = mb_layout(m, DK, DVK, LAST, false, CT);
  VMO_LDS char* q_t = sm + Lo.q;
  VMO_LDS char* k_t = sm + Lo.k;
  VMO_LDS char* y_t = sm + Lo.y;
  VMO_LDS float* e_t = (VMO_LDS float*)(sm + Lo.e);
  VMO_LDS float* lse_t = (VMO_LDS float*)(sm + Lo.lse);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int hl = lane >> 5, l32 = lane & 31;

  const int col = blockIdx.x, bh = col / p.bs, j = col % p.bs, hh = bh % p.heads, bb = bh / p.heads;
  const int64_t q_rs = (int64_t)p.bs * p.q_sn, o_rs = (int64_t)p.bs * p.out_sn, r_rs = (int64_t)p.bs * p.res_sn;
  const T* qcol = (const T*)p.q + bb * p.q_sb + hh * p.q_sh + (int64_t)j * p.q_sn;
  const T* ocol = (const T*)p.out + bb * p.out_sb + hh * p.out_sh + (int64_t)j * p.out_sn;
  T* rcol = (T*)p.res + bb * p.res_sb + hh * p.res_sh + (int64_t)j * p.res_sn;

  mb_stage<T, DK, D, CT>(qcol, q_rs, m, q_t, wave, lane);
  mb_stage<T, DK, D, CT>(ocol, o_rs, m, k_t, wave, lane);
  if constexpr (LAST) mb_stage<T, DVK, DV, CT>(ocol + D, o_rs, m, y_t, wave, lane);
  const float* ep = p.ent + bb * p.ent_sb + hh * p.ent_sh + j;
  for (int k = tid; k < M; k += 64 * kMbWaves) e_t[k] = k < m ? ep[(int64_t)k * p.bs] * kLog2e : -1.0e30f;
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();

  const float c = p.logit_scale_log2;
  // S^T blocks of query block ib against every key block, biased and in log2 units (keys past m at -1e30):
  // x[kb][r] for key 32 kb + 8 (r / 4) + 4 hl + r % 4 and query 32 ib + l32; returns the row max.
  auto s_blocks = [&](int ib, f32x16 (&x)[kMbMaxBlocks]) __attribute__((always_inline)) {
    V8 qb[NDS];
#pragma unroll
    for (int ds = 0; ds < NDS; ++ds) qb[ds] = mb_row8<V8, RBD, CT>(q_t, ib, m, l32, hl, ds);
    float mx = -3.0e38f;
#pragma unroll
    for (int kb = 0; kb < kMbMaxBlocks; ++kb) {
      if (kb >= MB) break;
      x[kb] = f32x16{};
#pragma unroll
      for (int ds = 0; ds < NDS; ++ds) x[kb] = E::mfma(mb_row8<V8, RBD, CT>(k_t, kb, m, l32, hl, ds), qb[ds], x[kb]);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 ev = *(const VMO_LDS f32x4*)(e_t + 32 * kb + 8 * g + 4 * hl);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[kb][4 * g + e] = fmaf(x[kb][4 * g + e], c, ev[e]);
          mx = fmaxf(mx, x[kb][4 * g + e]);
        }
      }
    }
    return wave_max32(mx);
  };

  // Two 32-frame blocks (33-64 frames) with an even number of output blocks: all four waves compute (with one
  // wave per block, waves 2 and 3 -- and so two of the CU's four SIMDs -- would idle through the passes, which
  // then took half of the launch at 33 frames).  The LSE pass splits the keys (wave w: query block w & 1 against
  // key block w >> 1; partial row max and sum through LDS), the product pass the output columns (wave w: row
  // block w & 1, column half w >> 1; both halves recompute the block's attention, the products' MFMAs are split).
  constexpr int NH = NACC / 2;
  if constexpr (TWO) {
    const int rb = wave & 1, half = wave >> 1;
    f32x16 acch[NH > 0 ? NH : 1];
#pragma unroll
    for (int a = 0; a < NH; ++a) acch[a] = f32x16{};
    float fsc = 1.f;
    if constexpr (LAST) {
      f32x16 x[kMbMaxBlocks];
      const float mx = s_blocks(rb, x);
      float sum = 0.f;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          x[kb][r] = fast_exp2(x[kb][r] - mx);
          sum += x[kb][r];
        }
      const float inv = 1.0f / wave_sum32(sum);
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const V8 P0 = mb_pack<T, V8>(x[kb], 0, inv), P1 = mb_pack<T, V8>(x[kb], 1, inv);
#pragma unroll
        for (int a = 0; a < NH; ++a) {
          acch[a] = E::mfma(mb_tr8<V8, RBY, CT>(y_t, kb, m, lane, half * NH + a, 0), P0, acch[a]);
          acch[a] = E::mfma(mb_tr8<V8, RBY, CT>(y_t, kb, m, lane, half * NH + a, 1), P1, acch[a]);
        }
      }
    } else {
      VMO_LDS float* pmax = (VMO_LDS float*)(sm + Lo.part);   // [key block][M]
      VMO_LDS float* psum = pmax + 2 * M;
      // The LSE pass takes key block rb against query block half: the kr rows it reads are the product pass's
      // B operand (same lanes and dims), and its q rows that pass's A operand for query block half, so both stay
      // in registers and the product pass reads one query block's rows from LDS instead of both and kr.
      V8 kr_op[NDS], q_op[NDS];
#pragma unroll
      for (int ds = 0; ds < NDS; ++ds) {
        kr_op[ds] = mb_row8<V8, RBD, CT>(k_t, rb, m, l32, hl, ds);
        q_op[ds] = mb_row8<V8, RBD, CT>(q_t, half, m, l32, hl, ds);
      }
      {   // S^T block (keys of block rb, queries of block half): partial max and sum per query row
        f32x16 x = f32x16{};
#pragma unroll
        for (int ds = 0; ds < NDS; ++ds) x = E::mfma(kr_op[ds], q_op[ds], x);
        float mx = -3.0e38f;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 ev = *(const VMO_LDS f32x4*)(e_t + 32 * rb + 8 * g + 4 * hl);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            x[4 * g + e] = fmaf(x[4 * g + e], c, ev[e]);
            mx = fmaxf(mx, x[4 * g + e]);
          }
        }
        mx = wave_max32(mx);
        float sum = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) sum += fast_exp2(x[r] - mx);
        sum = wave_sum32(sum);
        if (hl == 0) {
          pmax[rb * M + 32 * half + l32] = mx;
          psum[rb * M + 32 * half + l32] = sum;
        }
      }
      __syncthreads();
      if (tid < M) {   // LSE of query row tid from the two key blocks' partials; rows past m get +1e30
        const float m0 = pmax[tid], m1 = pmax[M + tid], mm = fmaxf(m0, m1);
        const float l = psum[tid] * fast_exp2(m0 - mm) + psum[M + tid] * fast_exp2(m1 - mm);
        lse_t[tid] = tid < m ? mm + fast_log2(l) : 1.0e30f;
      }
      __syncthreads();
      // u^T columns of half `half` for key block rb: one key per lane; query block half first (rows in registers)
      const float ek = e_t[32 * rb + l32];
      float cm = 0.f;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int ib = t == 0 ? half : 1 - half;
        f32x16 x = f32x16{};
#pragma unroll
        for (int ds = 0; ds < NDS; ++ds)
          x = E::mfma(t == 0 ? q_op[ds] : mb_row8<V8, RBD, CT>(q_t, ib, m, l32, hl, ds), kr_op[ds], x);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 lv = *(const VMO_LDS f32x4*)(lse_t + 32 * ib + 8 * g + 4 * hl);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float a = fast_exp2(fmaf(x[4 * g + e], c, ek - lv[e]));
            x[4 * g + e] = a;
            cm += a;
          }
        }
        const V8 P0 = mb_pack<T, V8>(x, 0, 1.f), P1 = mb_pack<T, V8>(x, 1, 1.f);
#pragma unroll
        for (int a = 0; a < NH; ++a) {
          acch[a] = E::mfma(mb_tr8<V8, RBD, CT>(q_t, ib, m, lane, half * NH + a, 0), P0, acch[a]);
          acch[a] = E::mfma(mb_tr8<V8, RBD, CT>(q_t, ib, m, lane, half * NH + a, 1), P1, acch[a]);
        }
      }
      fsc = p.scale / fmaxf(wave_sum32(cm), p.min_col_mass);
    }
    __syncthreads();   // every wave is done with the tiles: the patches reuse them
    VMO_LDS float* patch = (VMO_LDS float*)(sm + wave * kEpiPatchBytes);
    const int nrows = min(32, m - 32 * rb);
    T* const rows = rcol + 32 * rb * r_rs + half * NH * 32;
    if constexpr (LAST) {
      const int ibeg = p.skip > j ? (p.skip - j + p.bs - 1) / p.bs : 0;
      store_acc_rows<F16, CW>(patch, acch, NH, 1.f, kGradStore, (char*)rows, r_rs * 2, nrows, lane, max(0, ibeg - 32 * rb));
    } else {
      store_acc_rows<F16, CW>(patch, acch, NH, fsc, kGradStore, (char*)rows, r_rs * 2, nrows, lane);
    }
    return;
  } else {
    f32x16 acc[NACC];
#pragma unroll
    for (int a = 0; a < NACC; ++a) acc[a] = f32x16{};
    const int blk = wave;            // this wave's query block (last) or key block (otherwise)
    const bool busy = blk < MB;
    float fscale = 1.f;

    if constexpr (LAST) {
      if (busy) {
        f32x16 x[kMbMaxBlocks];
        const float mx = s_blocks(blk, x);
        float sum = 0.f;
#pragma unroll
        for (int kb = 0; kb < kMbMaxBlocks; ++kb) {
          if (kb >= MB) break;
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            x[kb][r] = fast_exp2(x[kb][r] - mx);
            sum += x[kb][r];
          }
        }
        const float inv = 1.0f / wave_sum32(sum);
        // z^T[dv][i] = sum_k y^T[dv][k] attn^T[k][i]
#pragma unroll
        for (int kb = 0; kb < kMbMaxBlocks; ++kb) {
          if (kb >= MB) break;
          const V8 P0 = mb_pack<T, V8>(x[kb], 0, inv), P1 = mb_pack<T, V8>(x[kb], 1, inv);
#pragma unroll
          for (int a = 0; a < NACC; ++a) {
            acc[a] = E::mfma(mb_tr8<V8, RBY, CT>(y_t, kb, m, lane, a, 0), P0, acc[a]);
            acc[a] = E::mfma(mb_tr8<V8, RBY, CT>(y_t, kb, m, lane, a, 1), P1, acc[a]);
          }
        }
      }
    } else {
      // pass 1: row log-sum-exp (log2 units) of every query row; rows past m get +1e30 (zero attention)
      if (busy) {
        f32x16 x[kMbMaxBlocks];
        const float mx = s_blocks(blk, x);
        float sum = 0.f;
#pragma unroll
        for (int kb = 0; kb < kMbMaxBlocks; ++kb) {
          if (kb >= MB) break;
#pragma unroll
          for (int r = 0; r < 16; ++r) sum += fast_exp2(x[kb][r] - mx);
        }
        const float lse = mx + fast_log2(wave_sum32(sum));
        if (hl == 0) lse_t[32 * blk + l32] = 32 * blk + l32 < m ? lse : 1.0e30f;
      }
      __syncthreads();
      // pass 2: key block blk; one key per lane
      if (busy) {
        V8 kb_op[NDS];
#pragma unroll
        for (int ds = 0; ds < NDS; ++ds) kb_op[ds] = mb_row8<V8, RBD, CT>(k_t, blk, m, l32, hl, ds);
        const float ek = e_t[32 * blk + l32];
        float cm = 0.f;
#pragma unroll
        for (int ib = 0; ib < kMbMaxBlocks; ++ib) {
          if (ib >= MB) break;
          // L[i][k] = q_i . kr_k: A = q rows (lane = query row), B = kr rows (lane = key)
          f32x16 x = f32x16{};
#pragma unroll
          for (int ds = 0; ds < NDS; ++ds) x = E::mfma(mb_row8<V8, RBD, CT>(q_t, ib, m, l32, hl, ds), kb_op[ds], x);
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const f32x4 lv = *(const VMO_LDS f32x4*)(lse_t + 32 * ib + 8 * g + 4 * hl);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float a = fast_exp2(fmaf(x[4 * g + e], c, ek - lv[e]));
              x[4 * g + e] = a;
              cm += a;
            }
          }
          // u^T[d][k] += sum_i q^T[d][i] attn[i][k]
          const V8 P0 = mb_pack<T, V8>(x, 0, 1.f), P1 = mb_pack<T, V8>(x, 1, 1.f);
#pragma unroll
          for (int a = 0; a < NACC; ++a) {
            acc[a] = E::mfma(mb_tr8<V8, RBD, CT>(q_t, ib, m, lane, a, 0), P0, acc[a]);
            acc[a] = E::mfma(mb_tr8<V8, RBD, CT>(q_t, ib, m, lane, a, 1), P1, acc[a]);
          }
        }
        fscale = p.scale / fmaxf(wave_sum32(cm), p.min_col_mass);
      }
    }

    __syncthreads();   // every wave is done with the tiles: the patches reuse them
    if (!busy) return;
    VMO_LDS float* patch = (VMO_LDS float*)(sm + wave * kEpiPatchBytes);
    const int nrows = min(32, m - 32 * blk);
    T* const rows = rcol + 32 * blk * r_rs;
    if constexpr (LAST) {
      // z rows i from the first one the recompute does not overwrite (token i b + j >= skip)
      const int ibeg = p.skip > j ? (p.skip - j + p.bs - 1) / p.bs : 0;
      store_acc_rows<F16, CW>(patch, acc, NACC, 1.f, kGradStore, (char*)rows, r_rs * 2, nrows, lane, max(0, ibeg - 32 * blk));
    } else {
      store_acc_rows<F16, CW>(patch, acc, NACC, fscale, kGradStore, (char*)rows, r_rs * 2, nrows, lane);
    }
  }
}


// Sums of an accumulator block's 16 rows over the 32 lanes of each half: lane l gets the total of one row (lanes l and
// l ^ 1 the same), 32-row index mb_lane_sums_row(l).  One permlane16 swap halves the registers, then every step
// keeps half of them, by a lane bit, and adds the mirrored lane's other half: 38 vector instructions.
__device__ __forceinline__ int mb_lane_sums_row(int lane) {
  const int r = ((lane & 8) >> 1) + ((lane & 4) >> 1) + ((lane & 2) >> 1) + ((lane & 16) >> 1);   // accumulator row
  return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
}
__device__ __forceinline__ float mb_lane_sums(const f32x16& t, int lane) {
  float s[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) {   // even 16-lane rows: accumulator row r, odd ones: r + 8
    const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(t[r]), __float_as_uint(t[r + 8]), false, false);
    s[r] = __uint_as_float(x[0]) + __uint_as_float(x[1]);
  }
  auto step = [&](int n, int bit, auto ctrl) __attribute__((always_inline)) {
    const bool up = (lane & bit) != 0;
#pragma unroll
    for (int r = 0; r < n; ++r) {
      const float keep = up ? s[r + n] : s[r], give = up ? s[r] : s[r + n];
      s[r] = keep + __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(give), decltype(ctrl)::value, 0xf, 0xf, true));
    }
  };
  step(4, 8, std::integral_constant<int, 0x140>{});   // row_mirror: lane 15 - j
  step(2, 4, std::integral_constant<int, 0x141>{});   // row_half_mirror: 7 - j
  step(1, 2, std::integral_constant<int, 0x1b>{});    // quad_perm: 3 - j
  return s[0] + __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(s[0]), 0xb1, 0xf, 0xf, true));   // j ^ 1
}

// Backward of the multi-block L-step (the gradient autograd takes through vmonarch.py:51-63 with the entropy
// bias detached, vmonarch.py:26), one 4-wave workgroup per grid column as the forward, with g the upstream
// gradient rows (dz rows i when last, du rows k otherwise) staged beside q, kr (and y):
//   last:  da[i,k] = g_i . y_k,  rs_i = sum_k a da,  dl = scale a (da - rs_i)
//          query blocks (one query row per lane): S^T and DA^T blocks -> lse_i, rs_i, dl, dq^T += Kr^T dl^T;
//          key blocks: dy^T += G^T a, dkr^T += Q^T dl
//   else:  c_k = sum_i a, gv_k = sum_i a (g_k . q_i), f_k = scale / max(c_k, mcm),
//          dc_k = -[c_k >= mcm] gv_k f_k / max(c_k, mcm),  da[i,k] = f_k (g_k . q_i) + dc_k
//          query blocks: lse_i;  key blocks (one key per lane): a, g_k . q_i -> c_k, gv_k, f_k, dc_k, da, each
//          wave's part of rs_i, then dl, dkr^T += Q^T dl;  query blocks: dq^T += Kr^T dl^T + G^T (a f)^T
// One block per wave: the a and da blocks are formed once, in one orientation, and reach the other as rounded MFMA
// operands through LDS matrices (mb_layout_bwd1).  Recomputing them in the second orientation, as this kernel did
// before, took 80 / 88 (last / otherwise) MFMAs and as many operand reads per block pair at 128-wide heads instead of
// 40 / 48.  What bounds a column is its chain (loads, passes, stores), so what counts most is a second column per CU
// to overlap it with (73-80 KB of LDS and 256 registers up to 96 frames; the last step up to 128) and no HBM round
// trips inside it (the rows dq is added to are read ahead).  12 heads x ~32760 tokens, 128-wide, non-last / last, us:
// 65 frames 526 / 347 -> 232 / 235, 96 frames 381 / 269 -> 185 / 188 (4.4 TB/s of the algorithmic bytes), 128 frames
// 344 / 251 -> 248 / 187.  The two-block kernels (TWO) recompute: their operands change hands through the row-store
// patches; reading dq's rows ahead took their non-last step from 318 to 289 us at 33 frames, 194 to 172 at 64.  The attention is exp2(logit - lse_i),
// exactly normalised.  MFMA operands a, dl and a f are
// rounded to the 16-bit type, the sums rs, c, gv kept in fp32 from the fp32 attention.  dq (fp32) is added
// to or overwritten, d out (the 16-bit type) written; rows past m carry zero attention and are not stored.
// MBX: the most row blocks it takes (2 with TWO).
template <int D, int DV, bool LAST, bool TWO, int MBX>
constexpr int mb_bwd_min_waves() {
  if (TWO) return 2;
  if (D <= 32 && (!LAST || DV <= 32)) return MBX == 2 ? 4 : MBX == 3 ? 3 : 2;   // narrow tiles: many columns per CU
  return LAST || MBX < 4 || D < 128 ? 2 : 1;
}
template <bool F16, int D, int DV, bool LAST, bool TWO, bool CT, int MBX>
__global__ __launch_bounds__(64 * kMbWaves, (mb_bwd_min_waves<D, DV, LAST, TWO, MBX>())) void lstep_mb_bwd_kernel(LBParams p) {
  using E = Elem<F16>;
  using T = typename E::T;
  using V8 = typename E::V8;
  constexpr int DK = tile_w(D), DVK = tile_w(DV);   // widths in LDS
  static_assert(!CT || (LAST && TWO), "compact tiles: the two-block last-step kernels");
  constexpr int NDS = D / 16, NDSV = DV / 16;
  constexpr int ND = DK / 32, NV = DVK / 32;
  constexpr int CWD = D < 32 ? 16 : 32, CWV = DV < 32 ? 16 : 32;   // stored columns per accumulator block
  constexpr int GW = LAST ? DV : D, GWK = tile_w(GW);
  constexpr int RBD = DK * 2, RBY = DVK * 2, RBG = GWK * 2;
  extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
  VMO_LDS char* sm = (VMO_LDS char*)smem_raw;

  const int m = p.m, MB = (m + 31) / 32, M = 32 * MB;
  const MbLayout Lo = TWO ? mb_layout(m, DK, DVK, LAST, true, CT) : mb_layout_bwd1(m, DK, DVK, LAST);
  VMO_LDS char* q_t = sm + Lo.q;
  VMO_LDS char* k_t = sm + Lo.k;
  VMO_LDS char* y_t = sm + Lo.y;
  VMO_LDS char* g_t = sm + Lo.g;
  VMO_LDS float* e_t = (VMO_LDS float*)(sm + Lo.e);
  VMO_LDS float* lse_t = (VMO_LDS float*)(sm + Lo.lse);
  VMO_LDS float* rs_t = (VMO_LDS float*)(sm + Lo.rs);
  VMO_LDS float* f_t = (VMO_LDS float*)(sm + Lo.f);
  VMO_LDS float* dc_t = (VMO_LDS float*)(sm + Lo.dc);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int hl = lane >> 5, l32 = lane & 31;
  VMO_LDS float* patch = (VMO_LDS float*)(sm + Lo.patch + wave * Lo.patch_rows * 32 * 4);

  const int col = blockIdx.x, bh = col / p.bs, j = col % p.bs, hh = bh % p.heads, bb = bh / p.heads;
  const int64_t q_rs = (int64_t)p.bs * p.q_sn, o_rs = (int64_t)p.bs * p.out_sn, g_rs = (int64_t)p.bs * p.g_sn;
  const int64_t dq_rs = (int64_t)p.bs * p.dq_sn, do_rs = (int64_t)p.bs * p.do_sn;
  const T* qcol = (const T*)p.q + bb * p.q_sb + hh * p.q_sh + (int64_t)j * p.q_sn;
  const T* ocol = (const T*)p.out + bb * p.out_sb + hh * p.out_sh + (int64_t)j * p.out_sn;
  const T* gcol = (const T*)p.g + bb * p.g_sb + hh * p.g_sh + (int64_t)j * p.g_sn;
  float* dqcol = p.dq + bb * p.dq_sb + hh * p.dq_sh + (int64_t)j * p.dq_sn;
  T* dcol = (T*)p.dout + bb * p.do_sb + hh * p.do_sh + (int64_t)j * p.do_sn;

  constexpr bool ROWS_IN_REGS = LAST && !TWO;   // the wave's q and g rows as MFMA operands, read from HBM
  V8 q_rows[ROWS_IN_REGS ? NDS : 1], g_rows[ROWS_IN_REGS ? NDSV : 1];
  if constexpr (ROWS_IN_REGS) {
    const int r = 32 * wave + l32, rr = r < m ? r : m - 1;
    const bool g_ok = r < m && (int64_t)r * p.bs + j >= p.skip;   // (z rows of tokens < skip are the recompute's)
#pragma unroll
    for (int ds = 0; ds < NDS; ++ds) {
      const V8 v = *(const V8*)(qcol + rr * q_rs + 16 * ds + 8 * hl);
      q_rows[ds] = r < m ? v : V8{};
    }
#pragma unroll
    for (int ds = 0; ds < NDSV; ++ds) {
      const V8 v = *(const V8*)(gcol + rr * g_rs + 16 * ds + 8 * hl);
      g_rows[ds] = g_ok ? v : V8{};
    }
  } else {
    mb_stage<T, DK, D, CT>(qcol, q_rs, m, q_t, wave, lane);
    mb_stage<T, GWK, GW, CT>(gcol, g_rs, m, g_t, wave, lane);
  }
  mb_stage<T, DK, D, CT>(ocol, o_rs, m, k_t, wave, lane);
  if constexpr (LAST) mb_stage<T, DVK, DV, CT>(ocol + D, o_rs, m, y_t, wave, lane);
  const float* ep = p.ent + bb * p.ent_sb + hh * p.ent_sh + j;
  for (int k = tid; k < M; k += 64 * kMbWaves) e_t[k] = k < m ? ep[(int64_t)k * p.bs] * kLog2e : -1.0e30f;
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if constexpr (LAST && TWO) {   // z rows of tokens < skip are the recompute's: no gradient reaches the L-path
    constexpr int CH = RBG / 16;
    for (int idx = tid; idx < m * CH; idx += 64 * kMbWaves) {
      const int r = idx / CH;
      if ((int64_t)r * p.bs + j < p.skip) *(VMO_LDS i32x4*)(g_t + r * RBG + (idx % CH) * 16) = i32x4{0, 0, 0, 0};
    }
    __syncthreads();
  }

  const float c = p.logit_scale_log2;
  const int blk = wave;
  const bool busy = blk < MB;
  const int dq_mode = p.dq_overwrite ? kGradStoreF32 : kGradAddF32;

  // S^T block (keys kb x queries of qb, one query row per lane), biased, log2 units
  auto s_block = [&](int kb, const V8 (&qb)[NDS]) __attribute__((always_inline)) {
    f32x16 x = f32x16{};
#pragma unroll
    for (int ds = 0; ds < NDS; ++ds) x = E::mfma(mb_row8<V8, RBD, CT>(k_t, kb, m, l32, hl, ds), qb[ds], x);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 ev = *(const VMO_LDS f32x4*)(e_t + 32 * kb + 8 * g + 4 * hl);
#pragma unroll
      for (int e = 0; e < 4; ++e) x[4 * g + e] = fmaf(x[4 * g + e], c, ev[e]);
    }
    return x;
  };
  // L block (queries ib x keys of key block kb, one key per lane): attn = exp2(c q.kr + e_k - lse_i); the kr
  // operand rows are read at each use (the passes that call this hold two accumulator sets)
  auto attn_block = [&](int ib, int kb, float ek) __attribute__((always_inline)) {
    f32x16 x = f32x16{};
#pragma unroll
    for (int ds = 0; ds < NDS; ++ds)
      x = E::mfma(mb_row8<V8, RBD, CT>(q_t, ib, m, l32, hl, ds), mb_row8<V8, RBD, CT>(k_t, kb, m, l32, hl, ds), x);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 lv = *(const VMO_LDS f32x4*)(lse_t + 32 * ib + 8 * g + 4 * hl);
#pragma unroll
      for (int e = 0; e < 4; ++e) x[4 * g + e] = fast_exp2(fmaf(x[4 * g + e], c, ek - lv[e]));
    }
    return x;
  };
  // query block's row LSE from its S^T blocks (kept in x for the caller)
  auto row_lse = [&](const V8 (&qb)[NDS], f32x16 (&x)[MBX]) __attribute__((always_inline)) {
    float mx = -3.0e38f;
#pragma unroll
    for (int kb = 0; kb < MBX; ++kb) {
      if (kb >= MB) break;
      x[kb] = s_block(kb, qb);
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, x[kb][r]);
    }
    mx = wave_max32(mx);
    float sum = 0.f;
#pragma unroll
    for (int kb = 0; kb < MBX; ++kb) {
      if (kb >= MB) break;
#pragma unroll
      for (int r = 0; r < 16; ++r) sum += fast_exp2(x[kb][r] - mx);
    }
    return mx + fast_log2(wave_sum32(sum));
  };
  auto load_rows = [&](V8 (&op)[NDS], const VMO_LDS char* tile, int b) __attribute__((always_inline)) {
#pragma unroll
    for (int ds = 0; ds < NDS; ++ds) op[ds] = mb_row8<V8, RBD, CT>(tile, b, m, l32, hl, ds);
  };
  const bool row_ok = 32 * blk + l32 < m;   // this lane's query row (query-block passes) or key (key-block passes)
  const int nrows = busy ? min(32, m - 32 * blk) : 0;
  // row stores through the patch: whole (32 rows), or 16 or 8 rows at a time
  auto store_rows = [&](auto cw_tag, const f32x16* acc, int nacc, int mode, char* row0, int64_t stride, int nr)
      __attribute__((always_inline)) {
    constexpr int CWS = decltype(cw_tag)::value;
    if (Lo.patch_rows == 32) store_acc_rows<F16, CWS, 32>(patch, acc, nacc, 1.f, mode, row0, stride, nr, lane);
    else if (TWO || Lo.patch_rows == 16) store_acc_rows<F16, CWS, 16>(patch, acc, nacc, 1.f, mode, row0, stride, nr, lane);
    else store_acc_rows<F16, CWS, 8>(patch, acc, nacc, 1.f, mode, row0, stride, nr, lane);
  };
  // The rows an fp32 result is added to, read ahead of the products that form it instead of one HBM round trip per
  // 32-column block at the end (base[a][i]: row lane / 8 + 8 i, columns CWD a + 4 (lane % 8) ..), and the store of
  // acc plus them.
  auto load_base = [&](auto& base, auto n_tag, const char* row0, int64_t stride, int nr) __attribute__((always_inline)) {
    constexpr int N = decltype(n_tag)::value;
#pragma unroll
    for (int a = 0; a < N; ++a)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int rr = (lane >> 3) + 8 * i, cc = lane & 7;
        base[a][i] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (rr < nr && 4 * cc < CWD) base[a][i] = *(const f32x4*)(row0 + rr * stride + (int64_t)(CWD * a + 4 * cc) * 4);
      }
  };
  auto store_rows_added = [&](const auto& acc, const auto& base, auto n_tag, char* row0, int64_t stride, int nr)
      __attribute__((always_inline)) {
    constexpr int N = decltype(n_tag)::value;
    const int pr_max = Lo.patch_rows, cc = lane & 7;
#pragma unroll
    for (int a = 0; a < N; ++a)
#pragma unroll
      for (int i = 0; i < 4; ++i) {   // 8 rows through the patch at a time: rows 8 i .. 8 i + 7
        if ((l32 >> 3) == i) {
#pragma unroll
          for (int g = 0; g < 4; ++g)
            *(VMO_LDS f32x4*)(patch + ((8 * i + (l32 & 7)) % pr_max) * 32 + ((2 * g + hl) ^ (l32 & 7)) * 4) =
                f32x4{acc[a][4 * g], acc[a][4 * g + 1], acc[a][4 * g + 2], acc[a][4 * g + 3]};
        }
        asm volatile("" ::: "memory");   // (lanes read what other lanes wrote, as in store_acc_rows)
        const int rr = (lane >> 3) + 8 * i;
        const f32x4 v = *(const VMO_LDS f32x4*)(patch + (rr % pr_max) * 32 + (cc ^ (rr & 7)) * 4);
        if (rr < nr && 4 * cc < CWD) *(f32x4*)(row0 + rr * stride + (int64_t)(CWD * a + 4 * cc) * 4) = base[a][i] + v;
        asm volatile("" ::: "memory");
      }
  };
  // p.delta: delta_k = sum_f out[k][f] d out[k][f] of this lane's key, from d out's accumulator blocks as stored and
  // out's row k as operands row(ds) (features 16 ds + 8 hl ..): this half's part.  Formed here it costs those operand
  // reads; the R-step backward's own pass read all of out and d out again.  96 x 341, 12 heads: that pass 100 -> 5 us, this
  // kernel 189 -> 227, the training step 2393 -> 2332; 48 x 211, 8 heads, 64-wide (three steps) 326 -> 317.  Last step
  // only: the other steps' kernel has no registers to spare (156 and more spilled).
  auto row_dot = [&](const auto& acc, auto n_tag, auto row, float d) __attribute__((always_inline)) {
    constexpr int N = decltype(n_tag)::value;
#pragma unroll
    for (int ds = 0; ds < N; ++ds) d = row_dot16<F16>(row(ds), mb_pack<T, V8>(acc[ds / 2], ds % 2, 1.f), d);
    return d;
  };
  float* delta = nullptr;   // in scalar registers: kept through every pass
  if (p.delta) {
    const uint64_t u = (uint64_t)(uintptr_t)(p.delta + bb * p.dl_sb + hh * p.dl_sh + j);
    delta = (float*)(uintptr_t)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(u >> 32)) << 32 |
                                (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)u));
  }
  // The two-block kernels (TWO) give each wave a (query block ib, key block kb) pair.  pair_lse: the row LSE of
  // the query rows from the S^T blocks of the pairs (each wave's x), as the partial max and sum of each key
  // block combined through `part` (rows past m get +1e30: their attention is exactly zero).  pair_row_sum: a
  // per-query-row sum over the two key blocks, each wave's partial v for its pair (every lane gets the total).
  VMO_LDS float* part = (VMO_LDS float*)(sm + Lo.part);   // [block][M] x two vectors
  auto pair_lse = [&](const f32x16& x, int ib, int kb) __attribute__((always_inline)) {
    float mx = -3.0e38f;
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, x[r]);
    mx = wave_max32(mx);
    float sum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) sum += fast_exp2(x[r] - mx);
    sum = wave_sum32(sum);
    if (hl == 0) {
      part[kb * M + 32 * ib + l32] = mx;
      part[2 * M + kb * M + 32 * ib + l32] = sum;
    }
    __syncthreads();
    if (tid < M) {
      const float m0 = part[tid], m1 = part[M + tid], mm = fmaxf(m0, m1);
      const float l = part[2 * M + tid] * fast_exp2(m0 - mm) + part[3 * M + tid] * fast_exp2(m1 - mm);
      lse_t[tid] = tid < m ? mm + fast_log2(l) : 1.0e30f;
    }
    __syncthreads();
  };
  auto pair_row_sum = [&](float v, int ib, int kb) __attribute__((always_inline)) {
    if (hl == 0) part[kb * M + 32 * ib + l32] = v;
    __syncthreads();
    return part[32 * ib + l32] + part[M + 32 * ib + l32];
  };

  // delta from the two column halves' partials (between two barriers: after the first the sums are read)
  auto put_pair_delta = [&](float d, int half, int kq) __attribute__((always_inline)) {
    d = wave_sum32(d);
    if (hl == 0) part[half * M + 32 * kq + l32] = d;
  };
  auto store_pair_delta = [&]() __attribute__((always_inline)) {
    if (tid < m) delta[(int64_t)tid * p.bs] = part[tid] + part[M + tid];
  };

  // One-block-per-wave passes.  put_mat: this wave's block row (lane: row l32 of block blk, accumulator order over
  // the columns) of a 16-bit matrix into LDS rows of kMbMatRow bytes, chunks swizzled like a tile's.  mat_product:
  // acc[f][c] (+)= sum_r tile[r][f] mat[r][c] for the columns c of block blk: both operands by transposed reads, in
  // the same row order.
  auto put_mat = [&](VMO_LDS char* mat, const V8 (&B)[MBX][2]) __attribute__((always_inline)) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    VMO_LDS char* row = mat + (32 * blk + l32) * kMbMatRow + hl * 8;
    const int sw = swz_rows<kMbMatRow>(l32);
#pragma unroll
    for (int cb = 0; cb < MBX; ++cb) {
      if (cb >= MB) break;
#pragma unroll
      for (int g = 0; g < 4; ++g) {   // columns 32 cb + 8 g + 4 hl .. + 3: chunk 4 cb + g, half hl
        const u32x4 w = __builtin_bit_cast(u32x4, B[cb][g >> 1]);
        *(VMO_LDS u32x2*)(row + ((4 * cb + g) ^ sw) * 16) = u32x2{w[2 * (g & 1)], w[2 * (g & 1) + 1]};
      }
    }
  };
  auto mat_product = [&](auto& acc, auto n_tag, auto rb_tag, const VMO_LDS char* tile, const VMO_LDS char* mat, bool zero)
      __attribute__((always_inline)) {
    constexpr int N = decltype(n_tag)::value, RB = decltype(rb_tag)::value;
    if (zero) {
#pragma unroll
      for (int a = 0; a < N; ++a) acc[a] = f32x16{};
    }
#pragma unroll
    for (int rb = 0; rb < MBX; ++rb) {
      if (rb >= MB) break;
#pragma unroll
      for (int h2 = 0; h2 < 2; ++h2) {
        const V8 b = mb_tr8<V8, kMbMatRow, false>(mat, rb, m, lane, blk, h2);
#pragma unroll
        for (int a = 0; a < N; ++a) acc[a] = E::mfma(mb_tr8<V8, RB, false>(tile, rb, m, lane, a, h2), b, acc[a]);
      }
    }
  };

  if constexpr (LAST) {
    if constexpr (TWO) {
      // Two blocks on four waves, as the non-last step's passes below: (query block, key block) pairs, the row
      // sums combined through `part`, the products split by output columns over operands exchanged in `xch`
      // (the row-store patches: 16-row ones up to 64 frames, room for two operands per wave and lane).
      constexpr int NH = ND / 2, NVH = NV / 2;
      VMO_LDS V8* xch = (VMO_LDS V8*)(sm + Lo.patch);
      const int ib = wave >> 1, kb = wave & 1;   // pass A: query block ib against key block kb
      const int kq = wave >> 1, iq = wave & 1;   // pass B: key block kq against query block iq
      // ---- pass A: row LSE from two partials, rs_i from two partials, then dq (query block ib, column half kb)
      {
        V8 qb[NDS];
        load_rows(qb, q_t, ib);
        f32x16 x = s_block(kb, qb);
        pair_lse(x, ib, kb);
        const float lse = lse_t[32 * ib + l32];
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = fast_exp2(x[r] - lse);   // attn^T[k][i]
        f32x16 d = f32x16{};   // DA^T[k][i] = y_k . g_i
#pragma unroll
        for (int ds = 0; ds < NDSV; ++ds)
          d = E::mfma(mb_row8<V8, RBY, CT>(y_t, kb, m, l32, hl, ds), mb_row8<V8, RBY, CT>(g_t, ib, m, l32, hl, ds), d);
        float rs = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) rs = fmaf(x[r], d[r], rs);
        rs = pair_row_sum(wave_sum32(rs), ib, kb);
        if (kb == 0 && hl == 0) rs_t[32 * ib + l32] = 32 * ib + l32 < m ? rs : 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) d[r] = p.scale * x[r] * (d[r] - rs);   // dl^T
        VMO_LDS V8* mine = xch + wave * 2 * 64 + lane;
        mine[0] = mb_pack<T, V8>(d, 0, 1.f);
        mine[64] = mb_pack<T, V8>(d, 1, 1.f);
        __syncthreads();
        f32x16 accq[NH];
#pragma unroll
        for (int a = 0; a < NH; ++a) accq[a] = f32x16{};
#pragma unroll
        for (int k2 = 0; k2 < 2; ++k2) {
          const VMO_LDS V8* src = xch + (2 * ib + k2) * 2 * 64 + lane;
          const V8 P0 = src[0], P1 = src[64];
#pragma unroll
          for (int a = 0; a < NH; ++a) {
            accq[a] = E::mfma(mb_tr8<V8, RBD, CT>(k_t, k2, m, lane, kb * NH + a, 0), P0, accq[a]);
            accq[a] = E::mfma(mb_tr8<V8, RBD, CT>(k_t, k2, m, lane, kb * NH + a, 1), P1, accq[a]);
          }
        }
        __syncthreads();   // every wave is done with xch: the patches may reuse it
        store_rows(std::integral_constant<int, CWD>{}, accq, NH, dq_mode, (char*)(dqcol + 32 * ib * dq_rs + 32 * kb * NH),
                   dq_rs * 4, min(32, m - 32 * ib));
      }
      __syncthreads();   // the patches are free again for xch, and rs_t is complete
      // ---- pass B: dy and dkr (key block kq, column half iq) over the two query blocks
      {
        const f32x16 at = attn_block(iq, kq, e_t[32 * kq + l32]);
        f32x16 dl = f32x16{};   // DA[i][k] = g_i . y_k
#pragma unroll
        for (int ds = 0; ds < NDSV; ++ds)
          dl = E::mfma(mb_row8<V8, RBY, CT>(g_t, iq, m, l32, hl, ds), mb_row8<V8, RBY, CT>(y_t, kq, m, l32, hl, ds), dl);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 rv = *(const VMO_LDS f32x4*)(rs_t + 32 * iq + 8 * g + 4 * hl);
#pragma unroll
          for (int e = 0; e < 4; ++e) dl[4 * g + e] = p.scale * at[4 * g + e] * (dl[4 * g + e] - rv[e]);
        }
        VMO_LDS V8* mine = xch + wave * 2 * 64 + lane;
        mine[0] = mb_pack<T, V8>(at, 0, 1.f);   // the attention block first: dy^T += G^T a
        mine[64] = mb_pack<T, V8>(at, 1, 1.f);
        __syncthreads();
        f32x16 accy[NVH];
#pragma unroll
        for (int a = 0; a < NVH; ++a) accy[a] = f32x16{};
#pragma unroll
        for (int i2 = 0; i2 < 2; ++i2) {
          const VMO_LDS V8* src = xch + (2 * kq + i2) * 2 * 64 + lane;
          const V8 A0 = src[0], A1 = src[64];
#pragma unroll
          for (int a = 0; a < NVH; ++a) {
            accy[a] = E::mfma(mb_tr8<V8, RBY, CT>(g_t, i2, m, lane, iq * NVH + a, 0), A0, accy[a]);
            accy[a] = E::mfma(mb_tr8<V8, RBY, CT>(g_t, i2, m, lane, iq * NVH + a, 1), A1, accy[a]);
          }
        }
        __syncthreads();
        mine[0] = mb_pack<T, V8>(dl, 0, 1.f);   // then dl: dkr^T += Q^T dl
        mine[64] = mb_pack<T, V8>(dl, 1, 1.f);
        __syncthreads();
        f32x16 acck[NH];
#pragma unroll
        for (int a = 0; a < NH; ++a) acck[a] = f32x16{};
#pragma unroll
        for (int i2 = 0; i2 < 2; ++i2) {
          const VMO_LDS V8* src = xch + (2 * kq + i2) * 2 * 64 + lane;
          const V8 P0 = src[0], P1 = src[64];
#pragma unroll
          for (int a = 0; a < NH; ++a) {
            acck[a] = E::mfma(mb_tr8<V8, RBD, CT>(q_t, i2, m, lane, iq * NH + a, 0), P0, acck[a]);
            acck[a] = E::mfma(mb_tr8<V8, RBD, CT>(q_t, i2, m, lane, iq * NH + a, 1), P1, acck[a]);
          }
        }
        if (delta) {
          auto y_row = [&](int ds) { return mb_row8<V8, RBY, CT>(y_t, kq, m, l32, hl, 2 * iq * NVH + ds); };
          auto k_row = [&](int ds) { return mb_row8<V8, RBD, CT>(k_t, kq, m, l32, hl, 2 * iq * NH + ds); };
          put_pair_delta(row_dot(acck, std::integral_constant<int, 2 * NH>{}, k_row,
                                 row_dot(accy, std::integral_constant<int, 2 * NVH>{}, y_row, 0.f)), iq, kq);
        }
        __syncthreads();
        if (delta) store_pair_delta();
        const int nr = min(32, m - 32 * kq);
        store_rows(std::integral_constant<int, CWV>{}, accy, NVH, kGradStore,
                   (char*)(dcol + 32 * kq * do_rs + D + 32 * iq * NVH), do_rs * 2, nr);
        store_rows(std::integral_constant<int, CWD>{}, acck, NH, kGradStore, (char*)(dcol + 32 * kq * do_rs + 32 * iq * NH),
                   do_rs * 2, nr);
      }
    } else {
      // ---- one query row per lane: a and da against every key block, rs_i, dl, dq; the other orientation's products
      // then take a and dl from an LDS matrix [i][k] each
      V8 P[MBX][2], A[MBX][2];
      if (busy) {
        f32x16 x[MBX], d[MBX];
        const float lse = row_lse(q_rows, x);
        float rs = 0.f;
#pragma unroll
        for (int kb = 0; kb < MBX; ++kb) {
          if (kb >= MB) break;
          d[kb] = f32x16{};   // DA^T[k][i] = y_k . g_i
#pragma unroll
          for (int ds = 0; ds < NDSV; ++ds) d[kb] = E::mfma(mb_row8<V8, RBY, CT>(y_t, kb, m, l32, hl, ds), g_rows[ds], d[kb]);
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            x[kb][r] = row_ok ? fast_exp2(x[kb][r] - lse) : 0.f;   // (rows past m: no attention)
            rs = fmaf(x[kb][r], d[kb][r], rs);
          }
        }
        rs = wave_sum32(rs);
        f32x16 accq[ND];
#pragma unroll
        for (int a = 0; a < ND; ++a) accq[a] = f32x16{};
#pragma unroll
        for (int kb = 0; kb < MBX; ++kb) {
          if (kb >= MB) break;
#pragma unroll
          for (int r = 0; r < 16; ++r) d[kb][r] = p.scale * x[kb][r] * (d[kb][r] - rs);
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            P[kb][h] = mb_pack<T, V8>(d[kb], h, 1.f);
            A[kb][h] = mb_pack<T, V8>(x[kb], h, 1.f);
          }
#pragma unroll
          for (int a = 0; a < ND; ++a) {
            accq[a] = E::mfma(mb_tr8<V8, RBD, CT>(k_t, kb, m, lane, a, 0), P[kb][0], accq[a]);
            accq[a] = E::mfma(mb_tr8<V8, RBD, CT>(k_t, kb, m, lane, a, 1), P[kb][1], accq[a]);
          }
        }
        store_rows(std::integral_constant<int, CWD>{}, accq, ND, dq_mode, (char*)(dqcol + 32 * blk * dq_rs), dq_rs * 4, nrows);
      }
      // this wave's rows (operands over W columns) into a tile of W-wide rows
      auto put_rows = [&](VMO_LDS char* tile, auto rb_tag, const auto& rows, int n) __attribute__((always_inline)) {
        constexpr int RB = decltype(rb_tag)::value;
        VMO_LDS char* row = tile + (32 * blk + l32) * RB;
#pragma unroll
        for (int ds = 0; ds < RB / 32; ++ds)   // (a 16-wide tensor in a 32-wide tile: its chunks twice)
          *(VMO_LDS V8*)(row + ((2 * ds + hl) ^ swz_rows<RB>(l32)) * 16) = rows[ds % n];
      };
      __syncthreads();   // every wave is done with kr and y
      if (busy) {
        put_mat(sm + Lo.mat0, A);
        put_rows(g_t, std::integral_constant<int, RBG>{}, g_rows, NDSV);
      }
      __syncthreads();
      // out's row of this lane's key, read again (kr and y are overlaid by now) beside the products
      auto load_out = [&](auto& row, int col0) __attribute__((always_inline)) {
        const T* const src = ocol + (int64_t)min(32 * blk + l32, m - 1) * o_rs + 8 * hl + col0;
        constexpr int N = sizeof(row) / sizeof(V8);
#pragma unroll
        for (int ds = 0; ds < N; ++ds) row[ds] = *(const V8*)(src + 16 * ds);
      };
      float dlt = 0.f;
      if (busy) {   // dy^T[dv][k] += sum_i g^T[dv][i] a[i][k]
        f32x16 accy[NV];
        V8 y_row[NDSV];
        if (delta) load_out(y_row, D);
        mat_product(accy, std::integral_constant<int, NV>{}, std::integral_constant<int, RBG>{}, g_t, sm + Lo.mat0, true);
        if (delta) dlt = row_dot(accy, std::integral_constant<int, NDSV>{}, [&](int ds) { return y_row[ds]; }, 0.f);
        store_rows(std::integral_constant<int, CWV>{}, accy, NV, kGradStore, (char*)(dcol + 32 * blk * do_rs + D),
                   do_rs * 2, nrows);
      }
      __syncthreads();
      if (busy) {
        put_mat(sm + Lo.mat1, P);
        put_rows(q_t, std::integral_constant<int, RBD>{}, q_rows, NDS);
      }
      __syncthreads();
      if (busy) {   // dkr^T[d][k] += sum_i q^T[d][i] dl[i][k]
        f32x16 acck[ND];
        V8 k_row[NDS];
        if (delta) load_out(k_row, 0);
        mat_product(acck, std::integral_constant<int, ND>{}, std::integral_constant<int, RBD>{}, q_t, sm + Lo.mat1, true);
        if (delta) {
          dlt = wave_sum32(row_dot(acck, std::integral_constant<int, NDS>{}, [&](int ds) { return k_row[ds]; }, dlt));
          if (row_ok && hl == 0) delta[(int64_t)(32 * blk + l32) * p.bs] = dlt;
        }
        store_rows(std::integral_constant<int, CWD>{}, acck, ND, kGradStore, (char*)(dcol + 32 * blk * do_rs), do_rs * 2,
                   nrows);
      }
    }
  } else {
    if constexpr (TWO) {
      // Two blocks on four waves: each pass takes one (query block, key block) pair per wave instead of one block
      // per wave (which left two waves idle).  The per-row / per-column sums over the pair's two blocks are
      // combined through `part`; the dq and dkr products are split by output columns (half NH of the ND
      // blocks per wave), each wave reading the 16-bit B operands that its block pair's waves wrote to `xch`
      // (the row-store patch region, free until the stores).  Each accumulator takes its products in the same
      // order as the one-block-per-wave passes.
      constexpr int NH = ND / 2;
      VMO_LDS V8* xch = (VMO_LDS V8*)(sm + Lo.patch);         // [wave][operand][lane]
      const int ib = wave >> 1, kb = wave & 1;   // passes 0 and 2: query block ib against key block kb
      const int kq = wave >> 1, iq = wave & 1;   // passes 1 and 3: key block kq against query block iq
      const bool ib_ok = 32 * ib + l32 < m;
      V8 qb[NDS];
      load_rows(qb, q_t, ib);
      // ---- pass 0: row LSE from the two key blocks' partial max / sum
      pair_lse(s_block(kb, qb), ib, kb);
      // ---- pass 1: column mass c_k and gv_k from the two query blocks' partials -> f_k, dc_k
      {
        V8 gop[NDS];
        load_rows(gop, g_t, kq);
        const f32x16 at = attn_block(iq, kq, e_t[32 * kq + l32]);
        f32x16 gq = f32x16{};   // GQ[i][k] = q_i . g_k
#pragma unroll
        for (int ds = 0; ds < NDS; ++ds) gq = E::mfma(mb_row8<V8, RBD, CT>(q_t, iq, m, l32, hl, ds), gop[ds], gq);
        float cs = 0.f, gv = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          cs += at[r];
          gv = fmaf(at[r], gq[r], gv);
        }
        cs = wave_sum32(cs);
        gv = wave_sum32(gv);
        if (hl == 0) {
          part[iq * M + 32 * kq + l32] = cs;
          part[2 * M + iq * M + 32 * kq + l32] = gv;
        }
      }
      __syncthreads();
      if (tid < M) {
        const float cs = part[tid] + part[M + tid], gv = part[2 * M + tid] + part[3 * M + tid];
        const float cm = fmaxf(cs, p.min_col_mass), f = p.scale / cm;
        f_t[tid] = f;
        dc_t[tid] = (tid < m && cs >= p.min_col_mass) ? -gv * f / cm : 0.f;
      }
      __syncthreads();
      // ---- pass 2: rs_i from the two key blocks' partials, then dq (query block ib, column half kb)
      {
        char* const dq0 = (char*)(dqcol + 32 * ib * dq_rs + 32 * kb * NH);
        const int dq_nr = min(32, m - 32 * ib);
        f32x4 base[NH][4];
        if (dq_mode == kGradAddF32) load_base(base, std::integral_constant<int, NH>{}, dq0, dq_rs * 4, dq_nr);
        f32x16 x = s_block(kb, qb);
        const float lse = lse_t[32 * ib + l32];
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = fast_exp2(x[r] - lse);   // attn^T[k][i]
        f32x16 d = f32x16{};   // da^T[k][i] = f_k (g_k . q_i) + dc_k
#pragma unroll
        for (int ds = 0; ds < NDS; ++ds) d = E::mfma(mb_row8<V8, RBD, CT>(g_t, kb, m, l32, hl, ds), qb[ds], d);
        f32x4 fv[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          fv[g] = *(const VMO_LDS f32x4*)(f_t + 32 * kb + 8 * g + 4 * hl);
          const f32x4 cv = *(const VMO_LDS f32x4*)(dc_t + 32 * kb + 8 * g + 4 * hl);
#pragma unroll
          for (int e = 0; e < 4; ++e) d[4 * g + e] = fmaf(fv[g][e], d[4 * g + e], cv[e]);
        }
        float rs = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) rs = fmaf(x[r], d[r], rs);
        rs = pair_row_sum(wave_sum32(rs), ib, kb);
        if (kb == 0 && hl == 0) rs_t[32 * ib + l32] = ib_ok ? rs : 0.f;
        f32x16 dl, af;
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int r = 4 * g + e;
            af[r] = x[r] * fv[g][e];
            dl[r] = p.scale * x[r] * (d[r] - rs);
          }
        VMO_LDS V8* mine = xch + wave * 4 * 64 + lane;
        mine[0] = mb_pack<T, V8>(dl, 0, 1.f);
        mine[64] = mb_pack<T, V8>(dl, 1, 1.f);
        mine[128] = mb_pack<T, V8>(af, 0, 1.f);
        mine[192] = mb_pack<T, V8>(af, 1, 1.f);
        __syncthreads();
        f32x16 accq[NH];
#pragma unroll
        for (int a = 0; a < NH; ++a) accq[a] = f32x16{};
#pragma unroll
        for (int k2 = 0; k2 < 2; ++k2) {
          const VMO_LDS V8* src = xch + (2 * ib + k2) * 4 * 64 + lane;
          const V8 P0 = src[0], P1 = src[64], F0 = src[128], F1 = src[192];
#pragma unroll
          for (int a = 0; a < NH; ++a) {
            const int ca = kb * NH + a;   // this wave's column half
            accq[a] = E::mfma(mb_tr8<V8, RBD, CT>(k_t, k2, m, lane, ca, 0), P0, accq[a]);
            accq[a] = E::mfma(mb_tr8<V8, RBD, CT>(k_t, k2, m, lane, ca, 1), P1, accq[a]);
            accq[a] = E::mfma(mb_tr8<V8, RBD, CT>(g_t, k2, m, lane, ca, 0), F0, accq[a]);
            accq[a] = E::mfma(mb_tr8<V8, RBD, CT>(g_t, k2, m, lane, ca, 1), F1, accq[a]);
          }
        }
        __syncthreads();   // every wave is done with xch: the patches may reuse it
        if (dq_mode == kGradAddF32) store_rows_added(accq, base, std::integral_constant<int, NH>{}, dq0, dq_rs * 4, dq_nr);
        else store_rows(std::integral_constant<int, CWD>{}, accq, NH, dq_mode, dq0, dq_rs * 4, dq_nr);
      }
      __syncthreads();   // the patches are free again for xch, and rs_t is complete
      // ---- pass 3: dkr (key block kq, column half iq) over the two query blocks
      {
        V8 gop[NDS];
        load_rows(gop, g_t, kq);
        const float fk = f_t[32 * kq + l32], dck = dc_t[32 * kq + l32];
        const f32x16 at = attn_block(iq, kq, e_t[32 * kq + l32]);
        f32x16 dl = f32x16{};
#pragma unroll
        for (int ds = 0; ds < NDS; ++ds) dl = E::mfma(mb_row8<V8, RBD, CT>(q_t, iq, m, l32, hl, ds), gop[ds], dl);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 rv = *(const VMO_LDS f32x4*)(rs_t + 32 * iq + 8 * g + 4 * hl);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int r = 4 * g + e;
            dl[r] = p.scale * at[r] * (fmaf(fk, dl[r], dck) - rv[e]);
          }
        }
        VMO_LDS V8* mine = xch + wave * 2 * 64 + lane;
        mine[0] = mb_pack<T, V8>(dl, 0, 1.f);
        mine[64] = mb_pack<T, V8>(dl, 1, 1.f);
        __syncthreads();
        f32x16 acck[NH];
#pragma unroll
        for (int a = 0; a < NH; ++a) acck[a] = f32x16{};
#pragma unroll
        for (int i2 = 0; i2 < 2; ++i2) {
          const VMO_LDS V8* src = xch + (2 * kq + i2) * 2 * 64 + lane;
          const V8 P0 = src[0], P1 = src[64];
#pragma unroll
          for (int a = 0; a < NH; ++a) {
            const int ca = iq * NH + a;
            acck[a] = E::mfma(mb_tr8<V8, RBD, CT>(q_t, i2, m, lane, ca, 0), P0, acck[a]);
            acck[a] = E::mfma(mb_tr8<V8, RBD, CT>(q_t, i2, m, lane, ca, 1), P1, acck[a]);
          }
        }
        __syncthreads();
        store_rows(std::integral_constant<int, CWD>{}, acck, NH, kGradStore, (char*)(dcol + 32 * kq * do_rs + 32 * iq * NH),
                   do_rs * 2, min(32, m - 32 * kq));
      }
      return;
    }
    // ---- row LSE (query blocks)
    if (busy) {
      V8 qb[NDS];
      load_rows(qb, q_t, blk);
      f32x16 x[MBX];
      const float lse = row_lse(qb, x);
      if (hl == 0) lse_t[32 * blk + l32] = row_ok ? lse : 1.0e30f;
    }
    __syncthreads();
    // ---- one key per lane: a and g_k . q_i against every query block, column mass c_k and gv_k = sum_i a (g_k . q_i)
    // -> f_k, dc_k (all in the key's lanes); then rs_i, a sum over the keys, from each wave's partial per query row
    V8 P[MBX][2], F[MBX][2];
    f32x16 at[MBX], da[MBX];
    VMO_LDS float* const wpart = part + blk * M;   // this wave's sums over its 32 keys, per query row
    if (busy) {
      V8 kop[NDS], gop[NDS];
      load_rows(kop, k_t, blk);
      load_rows(gop, g_t, blk);
      const float ek = e_t[32 * blk + l32];
      float cs = 0.f, gv = 0.f;
#pragma unroll
      for (int ib = 0; ib < MBX; ++ib) {
        if (ib >= MB) break;
        at[ib] = f32x16{};
        da[ib] = f32x16{};   // GQ[i][k] = q_i . g_k
#pragma unroll
        for (int ds = 0; ds < NDS; ++ds) {
          const V8 qr = mb_row8<V8, RBD, CT>(q_t, ib, m, l32, hl, ds);
          at[ib] = E::mfma(qr, kop[ds], at[ib]);
          da[ib] = E::mfma(qr, gop[ds], da[ib]);
        }
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 lv = *(const VMO_LDS f32x4*)(lse_t + 32 * ib + 8 * g + 4 * hl);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int r = 4 * g + e;
            at[ib][r] = fast_exp2(fmaf(at[ib][r], c, ek - lv[e]));
            cs += at[ib][r];
            gv = fmaf(at[ib][r], da[ib][r], gv);
          }
        }
      }
      cs = wave_sum32(cs);
      gv = wave_sum32(gv);
      const float cm = fmaxf(cs, p.min_col_mass), fk = row_ok ? p.scale / cm : 0.f;
      const float dck = row_ok && cs >= p.min_col_mass ? -gv * fk / cm : 0.f;
#pragma unroll
      for (int ib = 0; ib < MBX; ++ib) {
        if (ib >= MB) break;
        f32x16 t;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          da[ib][r] = fmaf(fk, da[ib][r], dck);
          t[r] = at[ib][r] * da[ib][r];
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) F[ib][h] = mb_pack<T, V8>(at[ib], h, fk);
        const float sum = mb_lane_sums(t, lane);   // over the wave's keys (lanes)
        if ((lane & 1) == 0) wpart[32 * ib + mb_lane_sums_row(lane)] = sum;
      }
    }
    __syncthreads();
    if (tid < M) {
      float rs = 0.f;
      for (int w = 0; w < MB; ++w) rs += part[w * M + tid];
      rs_t[tid] = tid < m ? rs : 0.f;
    }
    __syncthreads();
    f32x4 base[ND][4];
    const bool add_q = dq_mode == kGradAddF32;
    if (busy) {   // dl; dkr^T[d][k] += sum_i q^T[d][i] dl[i][k]
      f32x16 acck[ND];
#pragma unroll
      for (int a = 0; a < ND; ++a) acck[a] = f32x16{};
#pragma unroll
      for (int ib = 0; ib < MBX; ++ib) {
        if (ib >= MB) break;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 rv = *(const VMO_LDS f32x4*)(rs_t + 32 * ib + 8 * g + 4 * hl);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int r = 4 * g + e;
            da[ib][r] = p.scale * at[ib][r] * (da[ib][r] - rv[e]);
          }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) P[ib][h] = mb_pack<T, V8>(da[ib], h, 1.f);
#pragma unroll
        for (int a = 0; a < ND; ++a) {
          acck[a] = E::mfma(mb_tr8<V8, RBD, CT>(q_t, ib, m, lane, a, 0), P[ib][0], acck[a]);
          acck[a] = E::mfma(mb_tr8<V8, RBD, CT>(q_t, ib, m, lane, a, 1), P[ib][1], acck[a]);
        }
      }
      if (add_q) load_base(base, std::integral_constant<int, ND>{}, (const char*)(dqcol + 32 * blk * dq_rs), dq_rs * 4, nrows);
      store_rows(std::integral_constant<int, CWD>{}, acck, ND, kGradStore, (char*)(dcol + 32 * blk * do_rs), do_rs * 2, nrows);
    }
    __syncthreads();   // every wave is done with q and the patches
    // ---- dq^T[d][i] += sum_k kr^T[d][k] dl[i][k] + g^T[d][k] (a f)[i][k], from an LDS matrix [k][i] each
    if (busy) put_mat(sm + Lo.mat0, P);
    __syncthreads();
    f32x16 accq[ND];
    if (busy) mat_product(accq, std::integral_constant<int, ND>{}, std::integral_constant<int, RBD>{}, k_t, sm + Lo.mat0, true);
    __syncthreads();
    if (busy) put_mat(sm + Lo.mat1, F);
    __syncthreads();
    if (busy) mat_product(accq, std::integral_constant<int, ND>{}, std::integral_constant<int, RBD>{}, g_t, sm + Lo.mat1, false);
    __syncthreads();   // every wave is done with the matrix, which the patches overlay
    if (busy) {
      char* const row0 = (char*)(dqcol + 32 * blk * dq_rs);
      if (add_q) store_rows_added(accq, base, std::integral_constant<int, ND>{}, row0, dq_rs * 4, nrows);
      else store_rows(std::integral_constant<int, CWD>{}, accq, ND, dq_mode, row0, dq_rs * 4, nrows);
    }
  }
}

// Head-dim pairs the multi-block kernels are built for: 32 / 64 / 128 in any pair, and 16 with 16 (the
// reference's VMonarch runs d = dv).
static bool mb_dims(int d, int dv, bool last) {
  const auto ok = [](int x) { return x == 32 || x == 64 || x == 128; };
  if (d == 16) return !last || dv == 16;
  return ok(d) && (!last || ok(dv));
}

int mb_lstep_check(int m, int d, int dv, bool last, bool bwd) {
  if (!mb_dims(d, dv, last) || m < 1 || m > kMbMaxFrames) return 0;
  const int dk = tile_w(d), dvk = last ? tile_w(dv) : 0;
  if (mb_layout(m, dk, dvk, last, bwd, false).total > 160 * 1024) return 0;
  return !bwd || mb_layout_bwd1(m, dk, dvk, last).total <= 160 * 1024;
}

template <bool F16, int D, int DV, bool LAST, bool TWO, bool CT>
static int launch_mb_k(const LParams& p, hipStream_t s) {
  int lds = mb_layout(p.m, tile_w(D), tile_w(DV), LAST, false, CT).total;
  // The two-block non-last kernel is built for four columns per CU (33-48 frames: their chain of passes is
  // the bound, and a fourth column in flight hides more of it); past 48 frames the column's bytes dominate,
  // and its LDS request is raised to hold the CU at three (measured faster there).
  if constexpr (TWO && !LAST)
    if (p.m > 48) lds = lds > 160 * 1024 / 4 + 256 ? lds : 160 * 1024 / 4 + 256;
  auto kern = lstep_mb_kernel<F16, D, DV, LAST, TWO, CT>;
  static std::atomic<int> lds_limit{65536};   // this kernel's dynamic-LDS limit as raised so far
  if (lds > lds_limit.load(std::memory_order_relaxed)) {   // (idempotent: a race only repeats the call)
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
      return set_error(VMO_ERR_LAUNCH, "lstep_mb: cannot raise the LDS limit to %d bytes", lds);
    lds_limit.store(lds, std::memory_order_relaxed);
  }
  hipLaunchKernelGGL(kern, dim3(p.cols_total), dim3(64 * kMbWaves), lds, s, p);
  return launch_status("lstep_mb");
}
// Two 32-frame blocks with an even number of output blocks run the instantiation whose passes split over all
// four waves (TWO).
template <bool F16, int D, int DV, bool LAST>
static int launch_mb(const LParams& p, hipStream_t s) {
  constexpr bool TWO_OK = (tile_w(LAST ? DV : D) / 32) % 2 == 0;
  if constexpr (TWO_OK) {
    if ((p.m + 31) / 32 == 2) {
      if constexpr (mb_compact_built(D, DV, LAST))
        if (p.m <= kMbCompactMaxFrames) return launch_mb_k<F16, D, DV, LAST, true, true>(p, s);
      return launch_mb_k<F16, D, DV, LAST, true, false>(p, s);
    }
  }
  return launch_mb_k<F16, D, DV, LAST, false, false>(p, s);
}

template <bool F16>
static int dispatch_mb(const LParams& p, int d, int dv, bool last, hipStream_t s) {
#define VMO_MB(D_, DV_)                                                                   \
  if (d == D_ && dv == DV_ && last) return launch_mb<F16, D_, DV_, true>(p, s);
#define VMO_MB_U(D_) \
  if (d == D_ && !last) return launch_mb<F16, D_, D_, false>(p, s);
  VMO_MB_U(16) VMO_MB_U(32) VMO_MB_U(64) VMO_MB_U(128)
  VMO_MB(16, 16) VMO_MB(32, 32) VMO_MB(32, 64) VMO_MB(32, 128)
  VMO_MB(64, 32) VMO_MB(64, 64) VMO_MB(64, 128)
  VMO_MB(128, 32) VMO_MB(128, 64) VMO_MB(128, 128)
#undef VMO_MB
#undef VMO_MB_U
  return set_error(VMO_ERR_UNSUPPORTED, "lstep_mb: no kernel for d=%d dv=%d last=%d", d, dv, (int)last);
}

int mb_lstep_fwd(const LParams& p, bool f16, int d, int dv, bool last, hipStream_t s) {
  return f16 ? dispatch_mb<true>(p, d, dv, last, s) : dispatch_mb<false>(p, d, dv, last, s);
}

template <bool F16, int D, int DV, bool LAST, bool TWO, bool CT, int MBX>
static int launch_mb_bwd_k(const LBParams& p, hipStream_t s) {
  const int lds = TWO ? mb_layout(p.m, tile_w(D), tile_w(DV), LAST, true, CT).total
                      : mb_layout_bwd1(p.m, tile_w(D), tile_w(DV), LAST).total;
  auto kern = lstep_mb_bwd_kernel<F16, D, DV, LAST, TWO, CT, MBX>;
  static std::atomic<int> lds_limit{65536};   // as in launch_mb, per kernel
  if (lds > lds_limit.load(std::memory_order_relaxed)) {
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
      return set_error(VMO_ERR_LAUNCH, "lstep_mb_bwd: cannot raise the LDS limit to %d bytes", lds);
    lds_limit.store(lds, std::memory_order_relaxed);
  }
  hipLaunchKernelGGL(kern, dim3(p.cols_total), dim3(64 * kMbWaves), lds, s, p);
  return launch_status("lstep_mb_bwd");
}

// Grids of two row blocks (33-64 frames) take the kernel whose passes split the block pairs over all four waves,
// where the accumulator blocks split evenly (32-wide heads and 16-wide tiles have one block); the others keep one
// block per wave, up to three (96 frames: registers for two waves per SIMD at any head dim) or four.
template <bool F16, int D, int DV, bool LAST>
static int launch_mb_bwd(const LBParams& p, hipStream_t s) {
  constexpr bool TWO_OK = (tile_w(D) / 32) % 2 == 0 && (!LAST || (tile_w(DV) / 32) % 2 == 0);
  if constexpr (TWO_OK) {
    if ((p.m + 31) / 32 == 2) {
      if constexpr (mb_compact_built(D, DV, LAST))
        if (p.m <= kMbCompactMaxFrames) return launch_mb_bwd_k<F16, D, DV, LAST, true, true, 2>(p, s);
      return launch_mb_bwd_k<F16, D, DV, LAST, true, false, 2>(p, s);
    }
  }
  if constexpr (!TWO_OK)
    if (p.m <= 64) return launch_mb_bwd_k<F16, D, DV, LAST, false, false, 2>(p, s);
  if (p.m <= 96) return launch_mb_bwd_k<F16, D, DV, LAST, false, false, 3>(p, s);
  return launch_mb_bwd_k<F16, D, DV, LAST, false, false, 4>(p, s);
}

template <bool F16>
static int dispatch_mb_bwd(const LBParams& p, int d, int dv, bool last, hipStream_t s) {
#define VMO_MB(D_, DV_)                                                                   \
  if (d == D_ && dv == DV_ && last) return launch_mb_bwd<F16, D_, DV_, true>(p, s);
#define VMO_MB_U(D_) \
  if (d == D_ && !last) return launch_mb_bwd<F16, D_, D_, false>(p, s);
  VMO_MB_U(16) VMO_MB_U(32) VMO_MB_U(64) VMO_MB_U(128)
  VMO_MB(16, 16) VMO_MB(32, 32) VMO_MB(32, 64) VMO_MB(32, 128)
  VMO_MB(64, 32) VMO_MB(64, 64) VMO_MB(64, 128)
  VMO_MB(128, 32) VMO_MB(128, 64) VMO_MB(128, 128)
#undef VMO_MB
#undef VMO_MB_U
  return set_error(VMO_ERR_UNSUPPORTED, "lstep_mb_bwd: no kernel for d=%d dv=%d last=%d", d, dv, (int)last);
}

int mb_lstep_bwd(const LBParams& p, bool f16, int d, int dv, bool last, hipStream_t s) {
  return f16 ? dispatch_mb_bwd<true>(p, d, dv, last, s) : dispatch_mb_bwd<false>(p, d, dv, last, s);
}

}  // namespace vmo
