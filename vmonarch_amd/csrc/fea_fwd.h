// Flash-entropy forward: launch parameters, pipeline-stage sizes and tile copies shared by the 128-query kernel
// (fea_fwd.hip) and the key-group kernel of small grids (fea_fwd_ks.hip).
#pragma once

#include "vmo_common.h"
#include "vmo_host.h"

namespace vmo {

constexpr int kFwdQB = 1;             // 32-query MFMA blocks per wave
// Waves per workgroup (a template parameter of the kernel): 4 (128 queries, two workgroups per CU)
// or 8 (256 queries, one workgroup per CU).  Both keep two waves per SIMD; 8 halves the K / W tile
// traffic per flop, at the price of coarser query tiles.
constexpr int kFwdWavesSmall = 4;
constexpr int kFwdWavesLarge = 8;
constexpr int kFwdBN = 64;            // keys per pipeline stage
constexpr float kMaskLogit = -1.0e30f;

struct FwdParams {
  const void* q;
  const void* k;
  const void* w0;
  const void* w1;
  void* o;
  float* lse;
  float* ent;
  float* part_o;
  float* part_lse;
  int64_t q_sb, q_sh, q_sn;
  int64_t k_sb, k_sh, k_sn;
  int64_t w0_sb, w0_sh, w0_sn;
  int64_t w1_sb, w1_sh, w1_sn;
  int64_t o_sb, o_sh, o_sn;
  int64_t st_sb, st_sh;
  int heads, frames, nq, nk;
  int problems, q_tiles, splits, keys_per_split;
  int total_wg;
  float scale_log2;
  // fp8 S (QK8 variants): k quantized per problem, rows [nk][128] in the operand order of fea_fp8_keys_kernel,
  // one scale per 64-key tile (k8_tiles per problem)
  void* k8;
  float* k8_scale;
  int k8_tiles;
};

// Bytes of one pipeline stage: the K tile, the value tiles the K tile does not double as, and with fp8 S
// the fp8 K tile (one byte per element).
template <int D, int DW0, int DW1, bool W0K, bool QK8>
constexpr int fwd_stage_bytes() {
  return kFwdBN * (tile_w(D) + (W0K ? 0 : tile_w(DW0)) + (DW1 ? tile_w(DW1) : 0)) * 2 + (QK8 ? kFwdBN * D : 0);
}

// fp8 (e4m3) operand layout of the fp8 S product: a 128-wide row as two 64-dim products; lane half hl of
// product m takes dims 16 ds + 8 hl + e (ds = 4 m .. 4 m + 3, e = 0 .. 7), which are those the lane holds
// of the 16-bit q row, as 32 consecutive bytes.  Byte position of dim d in the stored row:
__host__ __device__ constexpr int fp8_dim_pos(int d) { return 64 * (d / 64) + 32 * ((d / 8) % 2) + 8 * ((d / 16) % 4) + d % 8; }
constexpr float kFp8Max = 448.f;   // e4m3's largest finite value (the conversion does not saturate: beyond it is NaN)

// LDS ring slots per workgroup: prefetch two tiles ahead when three slots stay within 64 KB (and with it within the
// workgroup's share of the CU's 160 KB), else one ahead.  The key loop reads every slot at compile-time offsets from
// shared per-lane addresses, and a read's offset field is 16 bits: three 24 KB slots (64-wide q / k with 128-wide
// values, 128 with 64) took a second set of addresses, which cost the online-entropy variants their second workgroup
// per CU (64 / 128: spills, so one; now 229 registers) or spills (128 / 64: 13, now none).  64 / 128, fp16, us at three
// slots and one workgroup per CU -> two and two: 48 heads x 777 tokens 34.3 -> 24.8, 24 x 8192 793 -> 647; 32 / 64, bf16,
// 12 x 4096 110 -> 77; 128 / 64, 48 x 777 26.1 -> 24.3.
constexpr int fwd_slots(int stage_bytes) {
  return 3 * stage_bytes <= 64 * 1024 ? 3 : 2;
}

// Copies of ROWS-row tiles (kFwdBN, one pipeline stage of the 128-query kernel) of a row-major (token, W) tensor into swizzled LDS tiles.  Wave
// instruction inst (= i * WAVES + wave) covers rows inst * RPI .. inst * RPI + RPI - 1 (1 KB);
// lane l copies chunk l % CH of row inst * RPI + l / CH to chunk (l % CH) ^ swz_rows(row).  The
// swizzle depends on the row modulo 16 only, which does not change with i when WAVES * RPI is a
// multiple of 16 (and alternates with i otherwise), so the lane's byte offset from its instruction's
// first row takes one or two values: a full tile costs scalar address arithmetic only.  A tile that runs
// past the end of the tensor (row >= nrows) re-reads the last row instead: finite data, masked out
// later.  Each wave issues NI copies per tile (vmcnt units).  SW < W (a 16-wide tensor in a 32-wide tile):
// logical chunk c of a row holds the source row's chunk c % (SW / 8).
template <class T, int W, int WAVES, int SW = W, int ROWS = kFwdBN>
struct TileCopy {
  static constexpr int CH = W / 8;       // 16-byte chunks per row
  static constexpr int RPI = 64 / CH;    // rows per wave instruction
  static constexpr int NI = ROWS / RPI / WAVES;
  static constexpr int NV = (WAVES * RPI) % 16 == 0 ? 1 : 2;   // distinct lane offsets
  static_assert(CH >= 4 && NI >= 1 && RPI >= 2, "tile shape");
  uint64_t ubase;     // base as a scalar byte address
  uint64_t rbytes;    // bytes per row
  uint32_t voff[NV];
  int wave, lane;

  __device__ __forceinline__ TileCopy(const T* b, int64_t s, int w, int l) : wave(w), lane(l) {
    ubase = uniform64((uint64_t)(uintptr_t)b);
    rbytes = uniform64((uint64_t)s * 2);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int r = (v * WAVES + w) * RPI + l / CH;   // the lane's row in instruction i = v
      voff[v] = (uint32_t)((int64_t)(l / CH) * s * 2) + (uint32_t)((((l % CH) ^ swz_rows<W * 2>(r)) & (SW / 8 - 1)) * 16);
    }
  }
  __device__ __forceinline__ void issue(int row0, int nrows, uint32_t dst) const {
    // row0 and nrows are uniform, but may arrive in vector registers (the variants that keep the
    // tile indices in vector registers): without readfirstlane the full-tile test becomes an exec
    // mask branch and the tile address a vector 64-bit multiply per copy.
    row0 = __builtin_amdgcn_readfirstlane(row0);
    nrows = __builtin_amdgcn_readfirstlane(nrows);
    // The per-instruction addresses are loop invariant up to row0; hoisted out of the key loop
    // they would pin dozens of scalar registers.  The empty asm hides where ub comes from, so they
    // are recomputed here (a few scalar adds per copy).
    uint64_t ub = ubase;
    asm volatile("" : "+s"(ub));
    if (row0 + ROWS <= nrows) {
      const uint64_t tb = ub + (uint64_t)(row0 + wave * RPI) * rbytes;
#pragma unroll
      for (int i = 0; i < NI; ++i)
        dma16_async_s(tb + (uint64_t)(i * WAVES * RPI) * rbytes, voff[i % NV], dst + (i * WAVES + wave) * 1024);
    } else {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int inst = i * WAVES + wave;
        const int r = inst * RPI + lane / CH;
        const int gr = min(row0 + r, nrows - 1);
        dma16_async((const void*)(uintptr_t)(ub + (uint64_t)gr * rbytes +
                                             (((lane % CH) ^ swz_rows<W * 2>(r)) & (SW / 8 - 1)) * 16),
                    dst + inst * 1024);
      }
    }
  }
};

// Entropy modes: none; online h = sum p (s c - m) in fp32 (kernel.py:49-50), e = log2 l - h / l; or,
// when the first value block is k itself (the VMonarch R-step), from the P.K accumulator at the end:
//   e = LSE ln2 - sm_scale q . (sum_j p~_j k_j) / l~   (nats), with l~ = sum_j p~_j
// -- no per-element product in the loop.  p~ is p rounded to the 16-bit type (the MFMA operand), and
// this mode sums exactly those rounded weights into l (also used for o and the LSE), so the mean logit
// is a proper average under one distribution.  Normalising the rounded moment by the fp32 sum instead
// leaves an error of (mean logit) x (relative rounding of the dominant p), several times the 2e-2
// tolerance on rows with logits of std 4 to 8.
enum { kEntNone = 0, kEntOnline = 1, kEntFromPK = 2 };

// The key-group forward kernel (fea_fwd_ks.hip) for launches whose 128-query tiles would leave the chip idle:
// true when it takes this one, with the launch's status in *rc.  With `tile` nothing is launched: its queries per workgroup.
bool fwd_ks(const FwdParams& p, bool f16, int d, int dw0, int dw1, bool w0k, bool ent, hipStream_t stream, int* rc,
            int* tile = nullptr);

}  // namespace vmo
